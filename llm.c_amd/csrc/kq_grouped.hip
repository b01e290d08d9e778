/*
 * kq_grouped.hip - products of many tokens with K-quant matrices (Q4_K,
 * Q6_K) on the matrix cores, bit for bit the reference's default -DQ8_DOT
 * build: the experts of a prompt-sized MoE layer (fused_ffn_silu,
 * nn.c:449-539, per expert instead of per token) and the dense product
 * (tensor_mma_transposed_2x2, matmul.c:270-324).
 *
 *   k_kq_rec      every token's Q8_K blocks (quantize_row_q8, quant.c:
 *                 627-654) as matrix-core operands: f16 quants, f16 sums
 *                 of 16 (one record per 256 values), and the scales
 *   k_kq_mm       per (32-row tile of one expert's pairs, 128 h columns)
 *                 gate, up and h = silu(g) * u in sorted row order
 *   k_kq_down_mm  y[pair][i] = dot_f32_quant(h[pair], down row i) per
 *                 (32-row tile, 64 output columns)
 *   k_kq_dense    out = add + x . W^T per (32 tokens, 128 columns)
 *
 * Why these stay exact.  dot_q4_K_q8_K / dot_q6_K_q8_K (quant_avx2.h:8-209)
 * are exact integer sums per super-block of 256, then a sequential chain of
 * fp32 FMAs over the super-blocks.  The integer sums run on
 * v_mfma_f32_32x32x16_f16 with integer operands and fp32 accumulators that
 * never pass 2^24, so every partial sum is exact in whatever order the
 * matrix core adds:
 *   Q4_K: operand sc_j * q4 (<= 63 * 15 = 945, exact in f16) times q8; the
 *         halves of a super-block apart (128 * 945 * 127 < 2^24), their sum
 *         rounded once: the reference's (float)sumi.  The minima's
 *         sum_j m_j * bsum_j from the sums of 16 (|bsum| <= 2032, exact in
 *         f16; 16 * 63 * 2032 < 2^24).
 *   Q6_K: sc = 16 sh + sl; operands sl * (q6 - 32) and sh * (q6 - 32)
 *         (<= 480 and 256 in magnitude), both sums below 2^24 over the whole
 *         super-block, fma(16, SH, SL) = (float)sumi rounded once.
 * The down dot is eight fp32 FMA chains over the elements l, l + 8, ...
 * (quant.c:198-418).  v_mfma_f32_16x16x4_f32 adds its four products to the
 * accumulator as four FMAs in k order, denormals, infinities and signed
 * zeros included (checked against fmaf chains on the device), so each chain
 * is one accumulator tile that takes its elements four at a time; the tree
 * of vector_avx2.h:126-132 joins the eight tiles at the end.
 *
 * Measured (Q4_K gate/up, Q6_K down): 2048 x 1024, 64 experts top-8, 301
 * tokens: 3456 -> 282 us a layer against a workgroup per pair and 32 rows
 * (under a profiler gate/up 930 -> 91, down 2608 -> 191 us); 4096 x 14336, 8
 * top-2, 200 tokens: 15490 -> 988 us (under a profiler, a tenth slower: 6361 ->
 * 315, 9176 -> 767).
 */
#include "kq_device.h"
#include "moe_internal.h"

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
/* native vector types: arrays of the uint4 struct stay in scratch memory */
typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef u32 u32x2 __attribute__((ext_vector_type(2)));
/* super-blocks of Q6_K start on any even address */
typedef u32 u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef u32 u32x2_a2 __attribute__((ext_vector_type(2), aligned(2)));

#define KR_BYTES 544 /* a record: 32 chunks of 16 bytes of quants, 2 of sums */
#define KR_PAIRS 17  /* pairs of chunks */
#define KM_ROWS 32   /* rows (tokens or pairs) of a tile */

/* ------------------------------------------------------------------ */
/* the tokens' records                                                  */
/* ------------------------------------------------------------------ */

/*
 * One wave per 256 values; lane l holds values 4l .. 4l + 3.  Chunk 2 s + h
 * is what lane half h of the MFMA reads for K-slice s: slice s = 2 i + u
 * covers values 32 i + 16 h + 8 u .. + 7, and inside a chunk the values go
 * 0, 2, 1, 3, 4, 6, 5, 7, the order in which masking a dword of weight
 * bytes yields them (bytes 0 and 2, then 1 and 3).
 */
__global__ __launch_bounds__(256) void k_kq_rec(const float *__restrict__ x, int blocks,
						uint8_t *__restrict__ rec,
						float *__restrict__ scale)
{
	const int b = blockIdx.x * 4 + threadIdx.x / WAVE, l = threadIdx.x % WAVE;
	if (b >= blocks)
		return;
	const float4 v = ((const float4 *)(x + (size_t)b * 256))[l];
	float d;
	int bs;
	const u32 q = kg_q8k(v, l, &d, &bs);
	uint8_t *r = rec + (size_t)b * KR_BYTES;
	half4_t o;
	o[0] = (_Float16)(float)(int8_t)(q & 0xff);
	o[1] = (_Float16)(float)(int8_t)((q >> 16) & 0xff);
	o[2] = (_Float16)(float)(int8_t)((q >> 8) & 0xff);
	o[3] = (_Float16)(float)(int8_t)(q >> 24);
	const int i = l / 8, h = (l / 4) & 1, u = (l / 2) & 1;
	*(half4_t *)(r + ((2 * i + u) * 2 + h) * 16 + (l & 1) * 8) = o;
	/* a block whose scale overflowed (largest magnitude below 127 / FLT_MAX)
	 * has meaningless sums and d = 0: clamped, they stay finite in f16 */
	if (l % 4 == 0)
		*(_Float16 *)(r + 512 + 2 * (l / 4)) = (_Float16)(float)max(-2048, min(2048, bs));
	if (l == 0)
		scale[b] = d;
}

/* ------------------------------------------------------------------ */
/* weight operands                                                      */
/* ------------------------------------------------------------------ */

__device__ static inline half2_t km_h2(u32 v)
{
	return __builtin_bit_cast(half2_t, v);
}

/* 8 weights from two dwords of bytes (mask m selects the value's bits in
 * each byte; `off` = -(1024 + bias) * s): (1024 + v) * s + off, exact */
__device__ static inline half8_t km_op(u32 a, u32 b, u32 m, half2_t s, half2_t off)
{
	const half2_t e = __builtin_elementwise_fma(km_h2((a & m) | 0x64006400u), s, off);
	const half2_t f = __builtin_elementwise_fma(km_h2(((a >> 8) & m) | 0x64006400u), s, off);
	const half2_t g = __builtin_elementwise_fma(km_h2((b & m) | 0x64006400u), s, off);
	const half2_t k = __builtin_elementwise_fma(km_h2(((b >> 8) & m) | 0x64006400u), s, off);
	return __builtin_shufflevector(__builtin_shufflevector(e, f, 0, 1, 2, 3),
				       __builtin_shufflevector(g, k, 0, 1, 2, 3), 0, 1, 2, 3, 4, 5,
				       6, 7);
}

/* A lane's share of one super-block of its column: lane half h of the four
 * chunks (Q4_K), of ql and qh (Q6_K), and the block's scales */
template <int WT> struct kmw;

template <> struct kmw<3> {
	u32x4 hd, q[4];
	__device__ inline void load(const uint8_t *blk, int h)
	{
		hd = *(const u32x4 *)blk;
#pragma unroll
		for (int j = 0; j < 4; j++)
			q[j] = *(const u32x4 *)(blk + 16 + 32 * j + 16 * h);
	}
	/* orders what follows after the point of the program this stands at */
	__device__ inline void pin()
	{
		asm volatile("" : "+v"(hd), "+v"(q[0]), "+v"(q[1]), "+v"(q[2]), "+v"(q[3]));
	}
	__device__ inline u32 dw(int j, int k) const
	{
		return k == 0 ? q[j].x : k == 1 ? q[j].y : k == 2 ? q[j].z : q[j].w;
	}
};

template <> struct kmw<5> {
	u32x4_a2 ql[4], qh[2], sc;
	unsigned short d;
	__device__ inline void load(const uint8_t *blk, int h)
	{
#pragma unroll
		for (int i = 0; i < 4; i++)
			ql[i] = *(const u32x4_a2 *)(blk + 32 * i + 16 * h);
#pragma unroll
		for (int c = 0; c < 2; c++)
			qh[c] = *(const u32x4_a2 *)(blk + 128 + 32 * c + 16 * h);
		sc = *(const u32x4_a2 *)(blk + 192);
		d = *(const unsigned short *)(blk + 208);
	}
	__device__ inline void pin()
	{
		u32 e = d;
		asm volatile(""
			     : "+v"(ql[0]), "+v"(ql[1]), "+v"(ql[2]), "+v"(ql[3]), "+v"(qh[0]),
			       "+v"(qh[1]), "+v"(sc), "+v"(e));
		d = (unsigned short)e;
	}
};

/*
 * The integer sums of one super-block: a 32 x 32 tile (rows of records in
 * LDS, columns of weights).  S1, S2: the halves' sums (Q4_K) or the sl and
 * sh sums (Q6_K).
 */
#define KM_LROW (KM_ROWS * 16) /* LDS bytes of one chunk index: the 32 rows */
/* the same where the kernel quantizes the rows itself: four chunks' stores of
 * 8 rows then start 16 banks apart (two lanes a bank, the least 512 bytes take) */
#define KM_LROW_Q (KM_LROW + 64)

template <int LR> __device__ static inline half8_t km_a(const uint8_t *sa, int chunk, int m)
{
	return *(const half8_t *)(sa + chunk * LR + m * 16);
}

/* the minima's part: acc_m = fma(-yd * dmin, msum, acc_m) for a lane's 16
 * rows (row 8 q + 4 h + i: yd points at the scales of rows 4 h ..) */
template <int LR>
__device__ static inline void km_mins(const kmw<3> &w, const uint8_t *sa, int m, int h,
				      const floatx4 *yd, floatx16 &accm)
{
	const u32 s1 = w.hd.z, s2 = w.hd.w;
	/* get_scale_min_k4 (quant.h:63-73): a byte per sub-block; the sums of
	 * 16 of sub-blocks 4h .. 4h + 3 */
	const u32 mw = h ? ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u)
			 : s1 & 0x3f3f3f3fu;
	const floatx16 z = {};
	half8_t mo;
#pragma unroll
	for (int k = 0; k < 4; k++)
		mo[2 * k] = mo[2 * k + 1] = (_Float16)(float)((mw >> (8 * k)) & 0xff);
	const floatx16 M =
		__builtin_amdgcn_mfma_f32_32x32x16_f16(km_a<LR>(sa, 32 + h, m), mo, z, 0, 0, 0);
	const float dm = f16_bits_to_f32(w.hd.x >> 16);
#pragma unroll
	for (int j = 0; j < 16; j++)
		accm[j] = __builtin_fmaf(-yd[2 * (j / 4)][j % 4] * dm, M[j], accm[j]);
}

template <int LR>
__device__ static inline void km_mins(const kmw<5> &, const uint8_t *, int, int, const floatx4 *,
				      floatx16 &)
{
}

/* Both run in steps of two MFMAs, the next step's operands (LDS reads and
 * unpacking) beside them: left to itself the scheduler reads every operand
 * first and spills, or each right before its MFMA and waits for it. */
template <int LR>
__device__ static inline void km_sums(const kmw<3> &w, const uint8_t *sa, int m, int h,
				      floatx16 &S1, floatx16 &S2)
{
	const u32 s0 = w.hd.y, s2 = w.hd.w;
	const u32 sc_lo = s0 & 0x3f3f3f3fu;
	const u32 sc_hi = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
	const floatx16 z = {};
	half8_t a[2][2], o[2][2]; /* [step & 1][low, high nibbles] */
	auto operands = [&](int t) {
		const int j = t / 2, u = t % 2;
		const u32 sw = j < 2 ? sc_lo : sc_hi;
		const _Float16 c = (_Float16)(float)((sw >> (16 * (j & 1))) & 0xff);
		const _Float16 d = (_Float16)(float)((sw >> (16 * (j & 1) + 8)) & 0xff);
		const _Float16 co = (_Float16)-1024.0f * c, ds = (_Float16)0.0625f * d,
			       dof = (_Float16)-64.0f * d;
		const half2_t c2 = {c, c}, co2 = {co, co}, d2 = {ds, ds}, do2 = {dof, dof};
		a[t & 1][0] = km_a<LR>(sa, ((4 * j + u) * 2) + h, m);
		a[t & 1][1] = km_a<LR>(sa, ((4 * j + 2 + u) * 2) + h, m);
		const u32 x = w.dw(j, 2 * u), y = w.dw(j, 2 * u + 1);
		o[t & 1][0] = km_op(x, y, 0x000f000fu, c2, co2);
		o[t & 1][1] = km_op(x, y, 0x00f000f0u, d2, do2);
	};
	operands(0);
	__builtin_amdgcn_sched_barrier(0);
#pragma unroll
	for (int t = 0; t < 8; t++) {
		if (t + 1 < 8)
			operands(t + 1);
		floatx16 &S = t < 4 ? S1 : S2;
		S = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t & 1][0], o[t & 1][0], t & 3 ? S : z, 0, 0,
							   0);
		S = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t & 1][1], o[t & 1][1], S, 0, 0, 0);
		__builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
#pragma unroll
		for (int i = 0; i < 2; i++) {
			__builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
			__builtin_amdgcn_sched_group_barrier(0x2, 14, 0);
		}
		__builtin_amdgcn_sched_barrier(0);
	}
}

template <int LR>
__device__ static inline void km_sums(const kmw<5> &w, const uint8_t *sa, int m, int h,
				      floatx16 &S1, floatx16 &S2)
{
	const floatx16 z = {};
	half8_t a[2], o[2][2]; /* [step & 1][sl, sh] */
	auto operands = [&](int t) {
		const int i = t / 2, u = t % 2, c = i / 4, g = i % 4;
		/* values 32 i ..; sub-block 2 i + h */
		const int sc = (int)(int8_t)((w.sc[i / 2] >> (16 * (i & 1) + 8 * h)) & 0xff);
		const _Float16 sl = (_Float16)(float)(sc & 15), sh = (_Float16)(float)(sc >> 4);
		const _Float16 slo = (_Float16)-1056.0f * sl, sho = (_Float16)-1056.0f * sh;
		const half2_t sl2 = {sl, sl}, slo2 = {slo, slo}, sh2 = {sh, sh}, sho2 = {sho, sho};
		u32 v[2];
#pragma unroll
		for (int k = 0; k < 2; k++) {
			const u32 q = w.ql[2 * c + (g & 1)][2 * u + k];
			const u32 lo = g < 2 ? q & 0x0f0f0f0fu : (q >> 4) & 0x0f0f0f0fu;
			v[k] = lo | (((w.qh[c][2 * u + k] >> (2 * g)) & 0x03030303u) << 4);
		}
		a[t & 1] = km_a<LR>(sa, ((2 * i + u) * 2) + h, m);
		o[t & 1][0] = km_op(v[0], v[1], 0x00ff00ffu, sl2, slo2);
		o[t & 1][1] = km_op(v[0], v[1], 0x00ff00ffu, sh2, sho2);
	};
	operands(0);
	__builtin_amdgcn_sched_barrier(0);
#pragma unroll
	for (int t = 0; t < 16; t++) {
		if (t + 1 < 16)
			operands(t + 1);
		S1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t & 1], o[t & 1][0], t ? S1 : z, 0, 0, 0);
		S2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[t & 1], o[t & 1][1], t ? S2 : z, 0, 0, 0);
		__builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
		for (int i = 0; i < 2; i++) {
			__builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
			__builtin_amdgcn_sched_group_barrier(0x2, 16, 0);
		}
		__builtin_amdgcn_sched_barrier(0);
	}
}

/* the fp32 step of one super-block: acc = fma(yd * d, sumi, acc) */
__device__ static inline void km_step(const kmw<3> &w, const floatx16 &S1, const floatx16 &S2,
				      const floatx4 *yd, floatx16 &acc)
{
	const float d = f16_bits_to_f32(w.hd.x);
#pragma unroll
	for (int j = 0; j < 16; j++)
		acc[j] = __builtin_fmaf(yd[2 * (j / 4)][j % 4] * d, S1[j] + S2[j], acc[j]);
}

__device__ static inline void km_step(const kmw<5> &w, const floatx16 &S1, const floatx16 &S2,
				      const floatx4 *yd, floatx16 &acc)
{
	const float d = f16_bits_to_f32(w.d);
#pragma unroll
	for (int j = 0; j < 16; j++)
		acc[j] = __builtin_fmaf(yd[2 * (j / 4)][j % 4] * d,
					__builtin_fmaf(16.0f, S2[j], S1[j]), acc[j]);
}

/* ------------------------------------------------------------------ */
/* gate/up of grouped pairs                                              */
/* ------------------------------------------------------------------ */

/* workgroup id -> item: the XCDs are dealt workgroups round-robin, so class
 * id % 8 takes a contiguous run of the items, whose tiles of one expert are
 * neighbours and share its weights in that XCD's L2; -1 past the items */
__device__ static inline int km_item(int id, int items)
{
	const int per = (items + 7) / 8, k = id / 8;
	const int it = (id % 8) * per + k;
	return k < per && it < items ? it : -1;
}

/*
 * A workgroup of NW waves takes a tile of 32 rows and NW * 32 columns: wave
 * w columns 32 w .. 32 w + 31 of gate and of up.  Per super-block the rows' records come by LDS-DMA (two buffers;
 * one load moves a pair of chunks of all 32 rows, which an operand read then
 * takes as 1 KB in a run) and are shared by the waves; a lane's columns' raw
 * blocks load straight into registers, each matrix's next super-block once
 * its last one is used.
 *
 * Bound: the VALU, of which the operands take about 2/3 (9 instructions per
 * 8 weights) and the fp32 steps 1/3, beside 17 (Q4_K: 16 and the minima's) or
 * 32 (Q6_K) MFMAs a matrix and super-block (two waves a SIMD overlap them); for many-expert layers of few rows a tile
 * the weights' bytes come next.  32 rows a tile: 64 need 256 registers of
 * accumulators, and the experts of a prompt average 10 to 60 rows.
 */
template <int WT, int NW>
__global__ __launch_bounds__(NW * WAVE, 2) void k_kq_mm(
	const uint8_t *__restrict__ W, const uint8_t *__restrict__ W2, size_t stride,
	const int *__restrict__ rows, const int *__restrict__ tile_e, int Tmax,
	const uint8_t *__restrict__ rec, const float *__restrict__ scale, int topk, int K, int N,
	float *__restrict__ out)
{
	constexpr int BY = kqb<WT>::BYTES, NC = 2, LR = KM_LROW;
	extern __shared__ __attribute__((aligned(16))) uint8_t km_lds[];
	uint8_t *s_a = km_lds;                                   /* [2][34][32] chunks */
	float *s_yd = (float *)(km_lds + 2 * 34 * KM_LROW);      /* [nb][32] */
	const int nb = K / 256, tid = threadIdx.x, lane = tid % WAVE;
	const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
	const int m = lane & 31, h = lane >> 5;
	const int cbs = (N + NW * 32 - 1) / (NW * 32);
	const int ntiles = tile_e[Tmax];
	const int item = km_item(blockIdx.x, ntiles * cbs);
	if (item < 0)
		return; /* the whole workgroup */
	const int tile = item % ntiles, cb = item / ntiles;
	const int col = cb * (NW * 32) + wave * 32 + m;
	const size_t eo = (size_t)tile_e[tile] * stride;
	/* columns past N repeat the last one (never stored) */
	const size_t co = eo + (size_t)min(col, N - 1) * nb * BY;
	const uint8_t *wp[2] = {W + co, W2 + co};

	/* row r of the tile's token */
	auto token = [&](int r) {
		const int p = rows[tile * KM_ROWS + r];
		return p < 0 ? 0 : p / topk; /* padding rows compute token 0's */
	};
	for (int i = tid; i < nb * KM_ROWS; i += NW * WAVE)
		s_yd[i] = scale[(size_t)token(i % KM_ROWS) * nb + i / KM_ROWS];
	const u32 src = (u32)token(m) * (u32)(nb * KR_BYTES) + (u32)h * 16u;
	const u32 l0 = __builtin_amdgcn_readfirstlane(lds_addr(s_a));
	/* pairs wave, wave + NW, ... of super-block sb into buffer sb & 1 */
	auto issue = [&](int sb) {
		const u32 lb = l0 + (u32)((sb & 1) * 34 * KM_LROW);
#pragma unroll
		for (int k = 0; k < (KR_PAIRS + NW - 1) / NW; k++) {
			const int i = wave + k * NW;
			if (i < KR_PAIRS)
				dma_dwordx4(rec, src + (u32)(sb * KR_BYTES + i * 32),
					    lb + (u32)(i * 2 * KM_LROW));
		}
	};
	kmw<WT> w[NC];
	floatx16 acc[NC] = {}, accm[NC] = {};
	issue(0);
#pragma unroll
	for (int c = 0; c < NC; c++)
		w[c].load(wp[c], h);
	/* waited for here: left in flight, the loop's own waits would assume the
	 * order of these loads and drain the next records' too */
#pragma unroll
	for (int c = 0; c < NC; c++)
		w[c].pin();
	for (int sb = 0; sb < nb; sb++) {
		/* super-block sb's records have landed once the first matrix's
		 * weights have: those loads were issued after them, and loads
		 * retire in order (the compiler waits for them here: a wait that
		 * counted the loads behind the records would rest on how many
		 * it makes of them) */
		w[0].pin();
		asm volatile("" ::: "memory");
		__syncthreads(); /* every wave's share; the other buffer is free */
		const int nx = min(sb + 1, nb - 1);
		if (sb + 1 < nb)
			issue(sb + 1);
		__builtin_amdgcn_sched_barrier(0);
		const uint8_t *sa = s_a + (sb & 1) * (34 * KM_LROW);
		const floatx4 *yd = (const floatx4 *)(s_yd + sb * KM_ROWS + 4 * h);
#pragma unroll
		for (int c = 0; c < NC; c++) {
			floatx16 S1, S2;
			if (c)
				w[c].pin(); /* not ahead of the other matrix's loads */
			km_mins<LR>(w[c], sa, m, h, yd, accm[c]);
			__builtin_amdgcn_sched_barrier(0);
			km_sums<LR>(w[c], sa, m, h, S1, S2);
			km_step(w[c], S1, S2, yd, acc[c]);
			__builtin_amdgcn_sched_barrier(0);
			/* the next super-block's, into the registers just read */
			w[c].load(wp[c] + (size_t)nx * BY, h);
			__builtin_amdgcn_sched_barrier(0);
		}
	}
	if (col >= N)
		return;
#pragma unroll
	for (int j = 0; j < 16; j++) {
		const int r = tile * KM_ROWS + 8 * (j / 4) + 4 * h + j % 4;
		const float g = WT == 3 ? acc[0][j] + accm[0][j] : acc[0][j];
		const float u = WT == 3 ? acc[1][j] + accm[1][j] : acc[1][j];
		out[(size_t)r * N + col] = (g / (1.0f + moe_expf(-g))) * u;
	}
}

/* ------------------------------------------------------------------ */
/* the dense product                                                    */
/* ------------------------------------------------------------------ */

/* the value of lane ^ 1, of lane ^ 2, of the mirrored lane among eight: VALU
 * moves, where a shuffle goes through LDS (whose round trips, one after the
 * other, took most of kq_stage's time) */
template <int CTRL> __device__ static inline int km_dpp(int v)
{
	return __builtin_amdgcn_mov_dpp(v, CTRL, 0xf, 0xf, true);
}

template <int CTRL> __device__ static inline float km_dpp(float v)
{
	return __builtin_bit_cast(float, km_dpp<CTRL>(__builtin_bit_cast(int, v)));
}

#define KM_X1 0xb1  /* quad_perm 1 0 3 2 */
#define KM_X2 0x4e  /* quad_perm 2 3 0 1 */
#define KM_M8 0x141 /* row_half_mirror */

/*
 * quantize_row_q8 (quant.c:627-654) of one super-block of a tile's 32 rows
 * into operand chunks at sa and scales at yd, by 256 threads: eight a row,
 * thread i of a row holding its float4s i, i + 8, ... (v[j]: values 4 (i + 8 j)
 * on), so that a load reads 128-byte runs.  The value of largest magnitude
 * comes from the signed extremes; only where both magnitudes are equal does
 * the index decide (the first wins).
 */
__device__ static inline void kq_stage(const float4 (&v)[8], uint8_t *sa, float *yd, int row, int i)
{
	constexpr int LR = KM_LROW_Q;
	float hi = 0.0f, lo = 0.0f;
#pragma unroll
	for (int j = 0; j < 8; j++) {
		hi = fmaxf(fmaxf(fmaxf(hi, v[j].x), fmaxf(v[j].y, v[j].z)), v[j].w);
		lo = fminf(fminf(fminf(lo, v[j].x), fminf(v[j].y, v[j].z)), v[j].w);
	}
	hi = fmaxf(hi, km_dpp<KM_X1>(hi));
	lo = fminf(lo, km_dpp<KM_X1>(lo));
	hi = fmaxf(hi, km_dpp<KM_X2>(hi));
	lo = fminf(lo, km_dpp<KM_X2>(lo));
	hi = fmaxf(hi, km_dpp<KM_M8>(hi));
	lo = fminf(lo, km_dpp<KM_M8>(lo));
	float bv = hi > -lo ? hi : lo;
	if (hi == -lo && hi > 0.0f) { /* the eight threads of a row agree */
		int key = 0x7fffffff;
#pragma unroll
		for (int j = 7; j >= 0; j--) {
			const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
			for (int k = 3; k >= 0; k--)
				if (fabsf(e[k]) == hi)
					key = (4 * (i + 8 * j) + k) * 2 + (e[k] < 0.0f);
		}
#pragma unroll
		for (int off = 1; off < 8; off <<= 1)
			key = min(key, __shfl_xor(key, off, WAVE));
		bv = key & 1 ? lo : hi;
	}
	const bool zero = bv == 0.0f;
	const float iscale = zero ? 0.0f : -127.0f / bv;
	const int h = i >> 2, u = (i >> 1) & 1;
#pragma unroll
	for (int j = 0; j < 8; j++) {
		const float e[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
		half4_t o;
		int s = 0;
#pragma unroll
		for (int k = 0; k < 4; k++) {
			int q = zero ? 0 : (int)roundf(iscale * e[k]);
			q = q < 127 ? q : 127;
			s += q;
			/* values 0, 2, 1, 3: the order of a weight operand (k_kq_rec) */
			o[k == 1 ? 2 : k == 2 ? 1 : k] = (_Float16)(float)(int8_t)(q & 0xff);
		}
		*(half4_t *)(sa + ((2 * j + u) * 2 + h) * LR + row * 16 + (i & 1) * 8) = o;
		s += km_dpp<KM_X1>(s);
		s += km_dpp<KM_X2>(s);
		/* sum i / 4 + 2 j of 16 values, finite in f16 as in k_kq_rec */
		if ((i & 3) == 0)
			*(_Float16 *)(sa + (32 + (j >> 2)) * LR + row * 16 + 2 * ((h + 2 * j) & 7)) =
				(_Float16)(float)max(-2048, min(2048, s));
	}
	if (i == 0)
		yd[row] = zero ? 0.0f : 1.0f / iscale;
}

#define KD_WAVES 4 /* of a workgroup's eight: the ones that multiply */

/*
 * out = add + x . W^T for T tokens: a workgroup takes a tile of 32 tokens and
 * 128 columns, as k_kq_mm takes one matrix, but quantizes its tokens itself
 * into the LDS buffer the next super-block is read from: a call then holds no
 * scratch memory, so calls on one matrix may overlap and be captured.  Four
 * waves multiply, four quantize the next super-block meanwhile (one of each
 * on every SIMD): the quantization is done again for every 128 columns and
 * costs about as much as the operands of one wave's 32 columns.
 *
 * Bound: the VALU, which the MFMAs' cycles add to where they share a SIMD.
 * Kernel times under a profiler, 4096 x 4096 Q4_K: 77 tokens 384 -> 42 us (the
 * whole call 413 -> 44), 333 tokens 1771 -> 70 us against the per-token
 * product (whose groups of tokens re-read and re-unpack every weight); Q6_K
 * 390 -> 55 and 1772 -> 96 us; 4096 x 14336 Q4_K, 77 tokens: 2132 -> 140 us.
 * With every wave quantizing and then multiplying: 47, 71, 78, 115 and 154 us.
 */
template <int WT>
__global__ __launch_bounds__(2 * KD_WAVES * WAVE, 4) void k_kq_dense(
	const uint8_t *__restrict__ W, const float *__restrict__ x, int T, int K, int N,
	const float *__restrict__ add, int add_rows, float *__restrict__ out)
{
	constexpr int BY = kqb<WT>::BYTES, LR = KM_LROW_Q;
	__shared__ __attribute__((aligned(16))) uint8_t s_a[2][34 * LR];
	__shared__ __attribute__((aligned(16))) float s_yd[2][KM_ROWS];
	const int nb = K / 256, tid = threadIdx.x, lane = tid % WAVE;
	const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
	const int m = lane & 31, h = lane >> 5;
	const int ntiles = (T + KM_ROWS - 1) / KM_ROWS, cbs = (N + KD_WAVES * 32 - 1) / (KD_WAVES * 32);
	const int item = km_item(blockIdx.x, ntiles * cbs);
	if (item < 0)
		return; /* the whole workgroup */
	const int tile = item % ntiles, col = item / ntiles * (KD_WAVES * 32) + wave * 32 + m;
	/* columns past N repeat the last one, rows past T the last token (never stored) */
	const uint8_t *wp = W + (size_t)min(col, N - 1) * nb * BY;
	if (wave >= KD_WAVES) { /* quantize: eight threads a token */
		const int pt = tid - KD_WAVES * WAVE, row = pt >> 3, i = pt & 7;
		const float4 *xp =
			(const float4 *)(x + (size_t)min(tile * KM_ROWS + row, T - 1) * K) + i;
		float4 v[8];
		auto fetch = [&](int sb) {
#pragma unroll
			for (int j = 0; j < 8; j++)
				v[j] = xp[(size_t)min(sb, nb - 1) * 64 + 8 * j];
		};
		fetch(0);
		kq_stage(v, s_a[0], s_yd[0], row, i);
		fetch(1);
		for (int sb = 0; sb < nb; sb++) {
			__syncthreads(); /* buffer sb & 1 is whole, the other one is free */
			if (sb + 1 < nb)
				kq_stage(v, s_a[(sb & 1) ^ 1], s_yd[(sb & 1) ^ 1], row, i);
			fetch(sb + 2);
		}
		return;
	}
	kmw<WT> w;
	floatx16 acc = {}, accm = {};
	w.load(wp, h);
	for (int sb = 0; sb < nb; sb++) {
		const int b = sb & 1;
		__syncthreads(); /* the other waves' one */
		/* the next super-block's; Q6_K's only once the sums' operands are
		 * done with (128 registers hold two workgroups a CU) */
		kmw<WT> wn;
		const uint8_t *next = wp + (size_t)min(sb + 1, nb - 1) * BY;
		if (WT == 3)
			wn.load(next, h);
		__builtin_amdgcn_sched_barrier(0);
		const floatx4 *yd = (const floatx4 *)(s_yd[b] + 4 * h);
		floatx16 S1, S2;
		km_mins<LR>(w, s_a[b], m, h, yd, accm);
		__builtin_amdgcn_sched_barrier(0);
		km_sums<LR>(w, s_a[b], m, h, S1, S2);
		if (WT != 3)
			wn.load(next, h);
		__builtin_amdgcn_sched_barrier(0);
		km_step(w, S1, S2, yd, acc);
		w = wn;
	}
	if (col >= N)
		return;
#pragma unroll
	for (int j = 0; j < 16; j++) {
		const int r = tile * KM_ROWS + 8 * (j / 4) + 4 * h + j % 4;
		if (r >= T)
			continue;
		const size_t o = (size_t)r * N + col;
		out[o] = (add ? add[add_rows ? o : (size_t)col] : 0.0f) +
			 (WT == 3 ? acc[j] + accm[j] : acc[j]);
	}
}

/* ------------------------------------------------------------------ */
/* down of grouped pairs                                                */
/* ------------------------------------------------------------------ */

/* a lane's share of one down super-block: its row's bytes 8 g .. 8 g + 7 of
 * every 32 values, g = lane / 16, and the scales */
template <int WT> struct kdw;

template <> struct kdw<3> {
	u32x4 hd;
	u32x2 q[4];
	__device__ inline void load(const uint8_t *blk, int g)
	{
		hd = *(const u32x4 *)blk;
#pragma unroll
		for (int j = 0; j < 4; j++)
			q[j] = *(const u32x2 *)(blk + 16 + 32 * j + 8 * g);
	}
	/* values 32 s + 8 g .. + 7: fl(fl(d * sc) * q) - fl(dmin * m) */
	__device__ inline void values(int s, int, float (&v)[8]) const
	{
		const u32 s0 = hd.y, s1 = hd.z, s2 = hd.w;
		const u32 scw = s < 4 ? s0 & 0x3f3f3f3fu
				      : (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
		const u32 mw = s < 4 ? s1 & 0x3f3f3f3fu
				     : ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
		const float d = f16_bits_to_f32(hd.x), dmin = f16_bits_to_f32(hd.x >> 16);
		const float ds = d * (float)((scw >> (8 * (s & 3))) & 0xff);
		const float ms = dmin * (float)((mw >> (8 * (s & 3))) & 0xff);
#pragma unroll
		for (int k = 0; k < 2; k++) {
			const u32 raw = k ? q[s / 2].y : q[s / 2].x;
			const u32 b = s & 1 ? (raw >> 4) & 0x0f0f0f0fu : raw & 0x0f0f0f0fu;
#pragma unroll
			for (int i = 0; i < 4; i++) {
				const float t = ds * (float)((b >> (8 * i)) & 0xff);
				v[4 * k + i] = t - ms;
			}
		}
	}
};

template <> struct kdw<5> {
	u32x2_a2 ql[4], qh[2];
	u32x4_a2 sc;
	unsigned short d;
	__device__ inline void load(const uint8_t *blk, int g)
	{
#pragma unroll
		for (int i = 0; i < 4; i++)
			ql[i] = *(const u32x2_a2 *)(blk + 32 * i + 8 * g);
#pragma unroll
		for (int c = 0; c < 2; c++)
			qh[c] = *(const u32x2_a2 *)(blk + 128 + 32 * c + 8 * g);
		sc = *(const u32x4_a2 *)(blk + 192);
		d = *(const unsigned short *)(blk + 208);
	}
	/* values 32 s + 8 g .. + 7: fl((q - 32) * fl(d * sc)), as fma(q, vs,
	 * -32 vs): the exact product rounded once (-32 vs is exact) */
	__device__ inline void values(int s, int g, float (&v)[8]) const
	{
		const int c = s / 4, x = s % 4;
		const int si = (int)(int8_t)((sc[s / 2] >> (16 * (s & 1) + 8 * (g >> 1))) & 0xff);
		const float vs = f16_bits_to_f32(d) * (float)si, nvs = -32.0f * vs;
#pragma unroll
		for (int k = 0; k < 2; k++) {
			const u32 raw = ql[2 * c + (x & 1)][k];
			const u32 lo = x < 2 ? raw & 0x0f0f0f0fu : (raw >> 4) & 0x0f0f0f0fu;
			const u32 b = lo | (((qh[c][k] >> (2 * x)) & 0x03030303u) << 4);
#pragma unroll
			for (int i = 0; i < 4; i++)
				v[4 * k + i] = __builtin_fmaf((float)((b >> (8 * i)) & 0xff), vs, nvs);
		}
	}
};

#define KW_HS 260 /* LDS floats of a row's 256 h values: rows 4 banks apart */
#define KW_COLS 64

/*
 * Bound: the fp32 matrix rate (157 TFLOP/s; the reference's order leaves no
 * faster unit): 4096 x 14336, 400 pairs, 47 GFLOP = 300 us without padding;
 * about 38 cycles a 16x16x4 instruction measured where 32 are nominal, and the
 * unpacking's VALU cycles add to them.
 * Eight chains of 16 x 16 accumulators per half tile and wave keep the
 * matrix core's latency covered; a wave unpacks its own 16 rows' weights
 * (26 VALU instructions per 8 MFMAs of a half tile), and the rows' h comes
 * through LDS, shared by the four waves (two buffers of a super-block).  The
 * loads of the next super-block go out at its top and a step's operands are
 * made one step ahead, both held there by hand (the compiler put each right
 * before its use): 831 -> 786 us at 400 pairs of 4096 x 14336, 202 -> 187 at
 * 2408 of 2048 x 1024 under a profiler.  Weights two super-blocks ahead
 * measured 7% slower (the copies between register sets wait for the loads).
 */
/* NS 16-row halves of the tile in use.  Wave w: down rows cb * 64 + 16 w ..
 * + 15; MFMA step (s, c): element 32 s + 8 k + c of chain c, k = lane / 16 */
template <int WT, int NS>
__device__ static inline void kd_tile(const uint8_t *__restrict__ base, int nb,
				      const float *__restrict__ hrow, int EI, float *s_h,
				      const int *__restrict__ rows, int r0, int E,
				      float *__restrict__ y)
{
	constexpr int BY = kqb<WT>::BYTES;
	constexpr int NL = NS * 16 * 64 / 256; /* float4 of h a thread moves */
	const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
	const int m = lane & 15, g = lane >> 4;
	const uint8_t *row = base + (size_t)(r0 + wave * 16 + m) * nb * BY;
	floatx4 st[NL];
	auto fetch = [&](int sb) {
#pragma unroll
		for (int k = 0; k < NL; k++) {
			const int i = tid + k * 256;
			st[k] = ((const floatx4 *)(hrow + (size_t)(i / 64) * EI + (size_t)sb * 256))[i % 64];
		}
	};
	auto stage = [&](int b) {
#pragma unroll
		for (int k = 0; k < NL; k++) {
			const int i = tid + k * 256;
			*(floatx4 *)(s_h + (size_t)b * (KM_ROWS * KW_HS) + (i / 64) * KW_HS +
				     4 * (i % 64)) = st[k];
		}
	};
	floatx4 acc[8][NS];
#pragma unroll
	for (int c = 0; c < 8; c++)
#pragma unroll
		for (int n = 0; n < NS; n++)
			acc[c][n] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
	kdw<WT> w;
	fetch(0);
	w.load(row, g);
	stage(0);
	for (int sb = 0; sb < nb; sb++) {
		__syncthreads(); /* buffer sb & 1 is whole, the other one is free */
		kdw<WT> wn;
		const int nx = min(sb + 1, nb - 1);
		fetch(nx);
		wn.load(row + (size_t)nx * BY, g);
		/* here, not next to their use a super-block later, where the
		 * compiler would put them */
		__builtin_amdgcn_sched_barrier(0);
		const float *sh = s_h + (size_t)(sb & 1) * (KM_ROWS * KW_HS) + m * KW_HS + 8 * g;
		float v[2][8];
		floatx4 a[2][NS][2];
		auto operands = [&](int s) {
#pragma unroll
			for (int n = 0; n < NS; n++) {
				a[s & 1][n][0] = *(const floatx4 *)(sh + n * 16 * KW_HS + 32 * s);
				a[s & 1][n][1] = *(const floatx4 *)(sh + n * 16 * KW_HS + 32 * s + 4);
			}
			w.values(s, g, v[s & 1]);
		};
		operands(0);
#pragma unroll
		for (int s = 0; s < 8; s++) { /* the next operands beside this step's MFMAs */
			if (s + 1 < 8)
				operands(s + 1);
#pragma unroll
			for (int c = 0; c < 8; c++)
#pragma unroll
				for (int n = 0; n < NS; n++)
					acc[c][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(
						a[s & 1][n][c / 4][c % 4], v[s & 1][c], acc[c][n], 0, 0, 0);
			__builtin_amdgcn_sched_group_barrier(0x100, 2 * NS, 0);
#pragma unroll
			for (int i = 0; i < 8 * NS; i++) {
				__builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
				__builtin_amdgcn_sched_group_barrier(0x2, 4, 0);
			}
			__builtin_amdgcn_sched_barrier(0);
		}
		stage((sb + 1) & 1);
		w = wn;
	}
	/* vector_reduce_sum's tree (vector_avx2.h:126-132) */
#pragma unroll
	for (int n = 0; n < NS; n++)
#pragma unroll
		for (int j = 0; j < 4; j++) {
			const int p = rows[n * 16 + 4 * g + j];
			const float v = ((acc[0][n][j] + acc[4][n][j]) + (acc[2][n][j] + acc[6][n][j])) +
					((acc[1][n][j] + acc[5][n][j]) + (acc[3][n][j] + acc[7][n][j]));
			if (p >= 0)
				y[(size_t)p * E + r0 + wave * 16 + m] = v;
		}
}

template <int WT>
__global__ __launch_bounds__(256, 2) void k_kq_down_mm(const uint8_t *__restrict__ down,
						     size_t dn_stride, const int *__restrict__ rows,
						     const int *__restrict__ tile_e, int Tmax,
						     const float *__restrict__ h, int E, int EI,
						     float *__restrict__ y)
{
	__shared__ __attribute__((aligned(16))) float s_h[2 * KM_ROWS * KW_HS];
	const int ntiles = tile_e[Tmax];
	const int item = km_item(blockIdx.x, ntiles * (E / KW_COLS));
	if (item < 0)
		return; /* the whole workgroup */
	const int tile = item % ntiles, r0 = item / ntiles * KW_COLS;
	const uint8_t *base = down + (size_t)tile_e[tile] * dn_stride;
	const float *hrow = h + (size_t)tile * KM_ROWS * EI;
	const int *tr = rows + tile * KM_ROWS;
	/* a tile's pairs come first: its second half may be padding */
	if (tr[16] < 0)
		kd_tile<WT, 1>(base, EI / 256, hrow, EI, s_h, tr, r0, E, y);
	else
		kd_tile<WT, 2>(base, EI / 256, hrow, EI, s_h, tr, r0, E, y);
}

/* ------------------------------------------------------------------ */
/* host side                                                            */
/* ------------------------------------------------------------------ */

/* the tokens' records, then their scales */
extern "C" size_t moe_kq_rec_bytes(size_t T, size_t K)
{
	return T * (K / 256) * (KR_BYTES + sizeof(float));
}

static const float *rec_scales(const void *rec, size_t T, size_t K)
{
	return (const float *)((const uint8_t *)rec + T * (K / 256) * KR_BYTES);
}

static size_t km_lds_bytes(int K)
{
	return 2 * 34 * KM_LROW + (size_t)(K / 256) * KM_ROWS * sizeof(float);
}

extern "C" int moe_kq_tile_rows(void)
{
	return KM_ROWS;
}

extern "C" int moe_launch_kq_rec(const float *x, int T, int K, void *rec, void *stream)
{
	const int blocks = T * (K / 256);
	hipLaunchKernelGGL(k_kq_rec, dim3((blocks + 3) / 4), dim3(256), 0, (hipStream_t)stream, x,
			   blocks, (uint8_t *)rec, (float *)rec_scales(rec, (size_t)T, (size_t)K));
	return (int)hipGetLastError();
}

extern "C" int moe_launch_kq_grouped(int gt, int dt, const uint8_t *gate, const uint8_t *up,
				     const uint8_t *down, size_t gu_stride, size_t dn_stride,
				     const int *rows, const int *tile_e, int Tmax, const void *rec,
				     float *h, float *y, int T, int topk, int E, int EI, void *stream)
{
	/* the records' byte offsets are 32-bit */
	if (moe_kq_rec_bytes((size_t)T, (size_t)E) > 0xffffffffull ||
	    (long long)Tmax * (EI / 128 > E / KW_COLS ? EI / 128 : E / KW_COLS) > 0x7fffff00ll)
		return (int)hipErrorInvalidValue;
	hipStream_t s = (hipStream_t)stream;
	const unsigned gg = (unsigned)(((long long)Tmax * (EI / 128) + 7) / 8 * 8);
	const unsigned gd = (unsigned)(((long long)Tmax * (E / KW_COLS) + 7) / 8 * 8);
	const float *scale = rec_scales(rec, (size_t)T, (size_t)E);
	if (gt == 3)
		hipLaunchKernelGGL((k_kq_mm<3, 4>), dim3(gg), dim3(256), km_lds_bytes(E), s, gate, up,
				   gu_stride, rows, tile_e, Tmax, (const uint8_t *)rec, scale, topk, E,
				   EI, h);
	else
		hipLaunchKernelGGL((k_kq_mm<5, 4>), dim3(gg), dim3(256), km_lds_bytes(E), s, gate, up,
				   gu_stride, rows, tile_e, Tmax, (const uint8_t *)rec, scale, topk, E,
				   EI, h);
	if (dt == 3)
		hipLaunchKernelGGL(k_kq_down_mm<3>, dim3(gd), dim3(256), 0, s, down, dn_stride, rows,
				   tile_e, Tmax, h, E, EI, y);
	else
		hipLaunchKernelGGL(k_kq_down_mm<5>, dim3(gd), dim3(256), 0, s, down, dn_stride, rows,
				   tile_e, Tmax, h, E, EI, y);
	return (int)hipGetLastError();
}

/* A tile costs the same for 1 and for 32 tokens, the per-token product grows
 * with T.  Where they cross, per-token / tile in us: Q4_K 4096 x 4096 T = 7
 * 40.6 / 40.3, T = 8 45.7 / 40.3; 2048 x 2048 T = 7 21.3 / 22.1, T = 8 23.6 /
 * 22.1; Q6_K 4096 x 4096 T = 9 51.3 / 53.0, T = 10 55.7 / 53.0; 2048 x 2048 T =
 * 9 30.9 / 28.0.  Matrices whose 128-row blocks fill half the chip or more
 * cross earlier: Q4_K 50304 x 2048 T = 6 41.9 / 36.3; Q6_K T = 7 55.0 / 49.9 */
extern "C" int moe_kq_dense_better(int wtype, size_t N, size_t T)
{
	if (N >= 16384)
		return T >= (wtype == 3 ? 6 : 7);
	return T >= (wtype == 3 ? 8 : 10);
}

extern "C" int moe_launch_kq_dense(int wtype, const uint8_t *W, int N, int K, const float *x, int T,
				   const float *add, int add_rows, float *out, void *stream)
{
	const long long items = (long long)((T + KM_ROWS - 1) / KM_ROWS) *
				((N + KD_WAVES * 32 - 1) / (KD_WAVES * 32));
	if ((wtype != 3 && wtype != 5) || N < 1 || T < 1 || K < 256 || K % 256 || items > 0x7fffff00ll)
		return (int)hipErrorInvalidValue;
	const dim3 grid((unsigned)((items + 7) / 8 * 8)), blk(2 * KD_WAVES * WAVE);
	hipStream_t s = (hipStream_t)stream;
	if (wtype == 3)
		hipLaunchKernelGGL(k_kq_dense<3>, grid, blk, 0, s, W, x, T, K, N, add, add_rows, out);
	else
		hipLaunchKernelGGL(k_kq_dense<5>, grid, blk, 0, s, W, x, T, K, N, add, add_rows, out);
	return (int)hipGetLastError();
}
