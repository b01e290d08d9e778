/*
 * moe_qgemv.h - the row-group loop of the dense quantized product
 * (moe_qgemv.hip), shared with the model kernels (lm_kernels.hip), which
 * stage their token themselves (a normalised residual stream) and watch
 * the outputs (the greedy pick of the lm_head).
 */
#ifndef MOE_QGEMV_H
#define MOE_QGEMV_H

#include "moe_device.h"
#include "moe_internal.h"

#define QG_WAVES 4
#define QG_GRID 768 /* workgroups when the caller passes no grid */

#define QG_ARGS                                                                         \
	const uint8_t *__restrict__ W, size_t rb, int N, int K, const float *__restrict__ x, \
		const float *__restrict__ add, float *__restrict__ out

/* no watcher of the outputs */
struct QgNoHook {
	__device__ void operator()(int, float) const {}
};

/*
 * out[j] = (add ? add[j] : 0) + dot(x, row j of W).  STAGED: the caller has
 * put the token in LDS (segment layout, SEG_STRIDE floats per 64 columns) and
 * synchronised.  hook(row, value) sees every stored output (lanes with seg ==
 * 0).
 */
template <int WT, int C, bool STAGED = false, class Hook = QgNoHook>
__device__ __forceinline__ static void qgemv_body(float *sx, QG_ARGS, Hook hook = Hook())
{
	constexpr int RPS = WAVE / C; /* rows per wave and group */
	constexpr int DW = qseg<WT>::DW;
	const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
	const int seg = lane % C, sub = lane / C; /* C == K / MOE_SEG_COLS */
	const int ngroups = (N + QG_WAVES * RPS - 1) / (QG_WAVES * RPS);

	/* rows past N repeat the last row (their results are not stored) */
	auto load = [&](int g, u32(&d)[DW]) {
		const int row = min(g * (QG_WAVES * RPS) + wave * RPS + sub, N - 1);
		load_dwords<DW>(W + (size_t)row * rb + (size_t)seg * qseg<WT>::BYTES, d);
	};

	int g = blockIdx.x;
	if (g >= ngroups)
		return; /* the whole workgroup: no barrier below is left waiting */
	u32 dn[DW];
	load(g, dn);
	if (!STAGED) {
		for (int i = threadIdx.x; i < K / 4; i += QG_WAVES * WAVE)
			*(float4 *)(sx + (i / 16) * SEG_STRIDE + 4 * (i % 16)) = ((const float4 *)x)[i];
		__syncthreads();
	}
	/* the token's block sums; its columns stay in LDS */
	const float(&xr)[64] = *(const float(*)[64])(sx + seg * SEG_STRIDE);
	float xs0, xs1;
	{
		float v[64];
		lds_x64(sx, seg, v);
		xs0 = sum32(v);
		xs1 = sum32(v + 32);
	}
	/* groups blockIdx.x, + gridDim.x, ...: the next group's weights load
	 * while this one's dots run */
	for (; g < ngroups; g += gridDim.x) {
		u32 d[DW];
#pragma unroll
		for (int i = 0; i < DW; i++)
			d[i] = dn[i];
		if (g + (int)gridDim.x < ngroups)
			load(g + gridDim.x, dn);
		float v;
		if constexpr (WT == 1)
			v = seg_dot_q8_0(d, xr, xs0, xs1);
		else
			v = seg_dot_q4_0(d, xr, xs0, xs1);
		v = group_sum<C>(v);
		const int row = g * (QG_WAVES * RPS) + wave * RPS + sub;
		if (seg == 0 && row < N) {
			const float r = (add ? add[row] : 0.0f) + v;
			out[row] = r;
			hook(row, r);
		}
	}
}

#endif
