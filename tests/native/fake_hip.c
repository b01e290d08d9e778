/*
 * fake_hip.c - the HIP runtime calls that libhip_moe.so makes, on host
 * memory and without a GPU: loaded with RTLD_GLOBAL before the library, it
 * takes the place of libamdhip64 (tests/test_host_paths.py).  Kernels do not
 * run; their names are logged.  Allocations are counted, and can be made to
 * fail with the error left behind until hipGetLastError, as the runtime
 * leaves it.
 */
#define _GNU_SOURCE
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <sys/mman.h>

#define OOM 2 /* hipErrorOutOfMemory */
#define PAGE 4096

static int last_error;
static size_t fail_size;    /* allocations of exactly this size fail */
static size_t fail_host;    /* and the next ones of host memory, if not 0 */
static size_t host_allocs;
static char log_buf[1 << 20], sizes_buf[1 << 20];
static struct {
	const void *host;
	const char *name;
} fns[4096];
static int nfns;

/* the names launched, then the device allocations' sizes, since the last call */
const char *fake_log(void)
{
	static char out[sizeof(log_buf)];
	strcpy(out, log_buf);
	log_buf[0] = 0;
	return out;
}

const char *fake_sizes(void)
{
	static char out[sizeof(sizes_buf)];
	strcpy(out, sizes_buf);
	sizes_buf[0] = 0;
	return out;
}

size_t fake_host_allocs(void)
{
	return host_allocs;
}

void fake_fail_size(size_t n)
{
	fail_size = n;
}

void fake_fail_host(size_t on)
{
	fail_host = on;
}

static void note(char *buf, size_t cap, const char *s)
{
	const size_t n = strlen(buf);
	if (n + strlen(s) + 2 < cap)
		sprintf(buf + n, "%s\n", s);
}

/* lazily backed, the length in a page before it */
static void *take(size_t n)
{
	void *p = mmap(NULL, n + PAGE, PROT_READ | PROT_WRITE,
		       MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
	if (p == MAP_FAILED)
		return NULL;
	*(size_t *)p = n;
	return (char *)p + PAGE;
}

static void give(void *p)
{
	if (p)
		munmap((char *)p - PAGE, *(size_t *)((char *)p - PAGE) + PAGE);
}

int hipMalloc(void **p, size_t n)
{
	char s[32];
	if (n == fail_size)
		return last_error = OOM;
	snprintf(s, sizeof(s), "%zu", n);
	note(sizes_buf, sizeof(sizes_buf), s);
	*p = take(n);
	return *p ? 0 : (last_error = OOM);
}

int hipFree(void *p)
{
	give(p);
	return 0;
}

int hipHostMalloc(void **p, size_t n, unsigned flags)
{
	if (fail_host)
		return last_error = OOM;
	host_allocs++;
	*p = take(n);
	return *p ? 0 : (last_error = OOM);
}

int hipHostFree(void *p)
{
	give(p);
	return 0;
}

int hipGetLastError(void)
{
	const int e = last_error;
	last_error = 0;
	return e;
}

int hipMemcpy(void *d, const void *s, size_t n, int kind)
{
	memcpy(d, s, n);
	return 0;
}

int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *stream)
{
	memcpy(d, s, n);
	return 0;
}

int hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, int kind,
		     void *stream)
{
	for (size_t i = 0; i < h; i++)
		memcpy((char *)d + i * dp, (const char *)s + i * sp, w);
	return 0;
}

int hipMemset(void *p, int v, size_t n)
{
	if (v)
		memset(p, v, n); /* fresh memory is zero */
	return 0;
}

/* dim3 arguments follow the function's address, which is all that is read */
int hipLaunchKernel(const void *f)
{
	for (int i = 0; i < nfns; i++)
		if (fns[i].host == f) {
			note(log_buf, sizeof(log_buf), fns[i].name);
			return 0;
		}
	note(log_buf, sizeof(log_buf), "?");
	return 0;
}

void **__hipRegisterFatBinary(const void *data)
{
	static void *module;
	return &module;
}

void __hipRegisterFunction(void **modules, const void *host, char *dev, const char *name)
{
	if (nfns < (int)(sizeof(fns) / sizeof(fns[0]))) {
		fns[nfns].host = host;
		fns[nfns++].name = strdup(name);
	}
}

void __hipRegisterVar(void **modules)
{
}

void __hipUnregisterFatBinary(void **modules)
{
}

int __hipPushCallConfiguration(void)
{
	return 0;
}

int __hipPopCallConfiguration(void)
{
	return 0;
}

int hipGetSymbolAddress(void **p, const void *symbol)
{
	static void *area;
	if (!area)
		area = take((size_t)16 << 20);
	*p = area;
	return area ? 0 : OOM;
}

int hipDeviceGetAttribute(int *v, int attr, int dev)
{
	*v = 256;
	return 0;
}

int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int block, size_t lds)
{
	*n = 2;
	return 0;
}

int hipGetDeviceCount(int *n)
{
	*n = 1;
	return 0;
}

int hipGetDevice(int *d)
{
	*d = 0;
	return 0;
}

int hipSetDevice(int d)
{
	return 0;
}

int hipDeviceSynchronize(void)
{
	return 0;
}

const char *hipGetErrorString(int e)
{
	return e == OOM ? "out of memory" : "error";
}

static int handle(void **p)
{
	static char any;
	*p = &any;
	return 0;
}

int hipStreamCreateWithFlags(void **s, unsigned flags)
{
	return handle(s);
}

int hipStreamDestroy(void *s)
{
	return 0;
}

int hipStreamSynchronize(void *s)
{
	return 0;
}

int hipStreamIsCapturing(void *s, int *status)
{
	*status = 0;
	return 0;
}

int hipStreamBeginCapture(void *s, int mode)
{
	return 0;
}

int hipStreamEndCapture(void *s, void **g)
{
	return handle(g);
}

int hipGraphInstantiate(void **e, void *g, void *a, void *b, size_t n)
{
	return handle(e);
}

int hipGraphLaunch(void *e, void *s)
{
	return 0;
}

int hipGraphDestroy(void *g)
{
	return 0;
}

int hipGraphExecDestroy(void *e)
{
	return 0;
}

int hipEventCreate(void **e)
{
	return handle(e);
}

int hipEventDestroy(void *e)
{
	return 0;
}

int hipEventRecord(void *e, void *s)
{
	return 0;
}

int hipEventElapsedTime(float *ms, void *a, void *b)
{
	*ms = 0.0f;
	return 0;
}
