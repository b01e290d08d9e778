/*
 * moe_qmm.hip - the dense quantized product for several tokens on the
 * gfx950 matrix cores, at fp32 accuracy:
 *   out[t][n] = add[t][n] (or add[n]) + sum_k x[t][k] * W[n][k]
 * with W N rows of K columns in Q8_0 or Q4_0 blocks (the reference's
 * tensor_mma_transposed_2x2 with a quantized right operand, matmul.c:451-462
 * -> 270-324, whose batched form tiles tokens and rows, matmul.c:145-165;
 * per element it is dot_f32_quant, quant.c:577-614).
 *
 * Exactness: a weight block is d * q with q small integers, exact in f16;
 * the block scale d stays out of the operand and is applied per block in
 * fp32.  A token block x (32 values) is scaled by a power of two 2^e (its
 * largest magnitude into [2^13, 2^14)) and split into two f16 parts,
 * hi = f16(x 2^e) and lo = f16(x 2^e - hi), which together hold x to ~22
 * bits.  One block of 16 tokens x 16 rows is then two
 * v_mfma_f32_16x16x32_f16 (hi, then lo, into a fresh accumulator: the
 * products q * hi and q * lo are exact in fp32), and
 *   acc += (d * 2^-e) * block
 * in fp32.  The result differs from an fp32 dot by the fp32 roundings of
 * other summation orders (~1e-7 relative), not by f16 rounding.
 *
 * Layouts.  The MFMA's K = 32 is split over the four 16-lane groups g of a
 * wave, eight values each; lane l holds token l % 16 (A) and row l % 16 (B)
 * of group l / 16, and the result D[token 4g + j][row l % 16] (j < 4).  The
 * values of group g are the block's elements 8g .. 8g+7 for Q8_0 (quant
 * bytes 8g.. of the block) and 4g .. 4g+3, 16+4g .. 16+4g+3 for Q4_0 (the
 * low and high nibbles of quant bytes 4g ..).
 *
 * Work: a workgroup of four waves takes 64 rows (16 a wave), one tile of 16
 * tokens and one stretch of QMM_PZ pairs of blocks (512 columns) of K.  It
 * first puts every load of its weights in flight (each wave its 16 rows:
 * Q4_0 five, Q8_0 seven dwords per lane and pair of blocks, windows aligned
 * to 4 bytes), then stages the 16 tokens' columns of its stretch in LDS,
 * split as above (hi and lo in [block][group][token] order, so a wave's
 * operand reads are 1 KB contiguous), so each token value is read once
 * per 64 rows.  With K longer than one stretch the stretches are
 * workgroups of their own (grid z), whose partial sums a second launch
 * adds in stretch order (k_qmm_reduce): deterministic, and enough
 * workgroups for the few-thousand-row projections.  (Adding them in the
 * product launch instead, by the last stretch of a tile to arrive, polling
 * epoch-tagged partials, measured 26.7 us against 22.8 us for the two
 * launches at 16 tokens x 6144 x 4096 Q4_0: the last arrivals' polls sit
 * in series behind the slowest stretch.)
 *
 * Many tokens, or very many rows, take k_qmm_tile below: tiles of 32 or 64
 * tokens over the whole of K, the same split with a scale per block.
 *
 * Bound of k_qmm: HBM for a few tokens (the weights are read once per token tile;
 * the tokens, T * K * 4 bytes, come from L2).  Algorithmic bytes per call:
 * N * K/32 * block bytes + T*K*4 + T*N*4.
 */
#include "moe_device.h"
#include "moe_internal.h"

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

#define QMM_ROWS 16
#define QMM_TOK 16
#define QMM_WAVES 4
#define QMM_PZ 8 /* pairs of blocks per workgroup: 512 columns of K; at 16
		  * the weights in flight take 256 VGPRs and one wave per SIMD
		  * fits (1.4x slower at 16 tokens x 6144 x 4096 Q4_0) */

/* ---------------------------------------------------------------------- */
/* the product                                                            */
/* ---------------------------------------------------------------------- */

__device__ static inline u32 qmm_ld(const uint8_t *p)
{
	return *(const u32 *)p;
}

/* two f16 (1024 + byte) from the bytes v_perm selects */
__device__ static inline u32 qmm_magic(u32 u, u32 sel)
{
	return __builtin_amdgcn_perm(0x64646464u, u, sel);
}

/* 8 bytes (w0 = bytes 0-3, w1 = 4-7), each biased by `off` - 1024, to 8 f16
 * byte - (off - 1024): exact small integers */
__device__ static inline half8_t qmm_half8(u32 w0, u32 w1, _Float16 off)
{
	typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
	const half2_t o2 = {off, off};
	const half2_t a = __builtin_bit_cast(half2_t, qmm_magic(w0, 0x04010400u)) - o2;
	const half2_t b = __builtin_bit_cast(half2_t, qmm_magic(w0, 0x04030402u)) - o2;
	const half2_t c = __builtin_bit_cast(half2_t, qmm_magic(w1, 0x04010400u)) - o2;
	const half2_t e = __builtin_bit_cast(half2_t, qmm_magic(w1, 0x04030402u)) - o2;
	half8_t r;
	r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
	r[4] = c[0]; r[5] = c[1]; r[6] = e[0]; r[7] = e[1];
	return r;
}

/* a lane's raw weights of one pair of blocks (2P, 2P+1) of its row */
template <int WT> struct qmm_pair;

template <> struct qmm_pair<2> { /* Q4_0: 36 bytes, 4-byte aligned */
	static constexpr int DW = 5;
	__device__ static inline void load(const uint8_t *base, int g, u32 (&w)[DW])
	{
		w[0] = qmm_ld(base + 4 * g);      /* even block: quant bytes 4g.. at +2+4g */
		w[1] = qmm_ld(base + 4 * g + 4);
		w[2] = qmm_ld(base + 20 + 4 * g); /* odd block: quant bytes 4g.. at +20+4g */
		w[3] = qmm_ld(base);              /* even scale: bytes 0-1 */
		w[4] = qmm_ld(base + 16);         /* odd scale: bytes 18-19 */
	}
	/* block h (0 even, 1 odd): the unscaled operand and d */
	__device__ static inline half8_t operand(const u32 (&w)[DW], int h, float &d)
	{
		const u32 q = h ? w[2] : __builtin_amdgcn_alignbit(w[1], w[0], 16);
		d = f16_bits_to_f32(h ? w[4] >> 16 : w[3] & 0xffffu);
		return qmm_half8(q & 0x0f0f0f0fu, (q >> 4) & 0x0f0f0f0fu, (_Float16)1032.0f);
	}
};

template <> struct qmm_pair<1> { /* Q8_0: 68 bytes, 4-byte aligned */
	static constexpr int DW = 7;
	__device__ static inline void load(const uint8_t *base, int g, u32 (&w)[DW])
	{
		w[0] = qmm_ld(base + 8 * g);      /* even block: quants 8g.. at +2+8g */
		w[1] = qmm_ld(base + 8 * g + 4);
		w[2] = qmm_ld(base + 8 * g + 8);
		w[3] = qmm_ld(base + 36 + 8 * g); /* odd block: quants 8g.. at +36+8g */
		w[4] = qmm_ld(base + 40 + 8 * g);
		w[5] = qmm_ld(base);              /* even scale: bytes 0-1 */
		w[6] = qmm_ld(base + 32);         /* odd scale: bytes 34-35 */
	}
	__device__ static inline half8_t operand(const u32 (&w)[DW], int h, float &d)
	{
		u32 q0, q1;
		if (h) {
			q0 = w[3];
			q1 = w[4];
		} else {
			q0 = __builtin_amdgcn_alignbit(w[1], w[0], 16);
			q1 = __builtin_amdgcn_alignbit(w[2], w[1], 16);
		}
		d = f16_bits_to_f32(h ? w[6] >> 16 : w[5] & 0xffffu);
		/* signed bytes: q ^ 0x80 = q + 128 */
		return qmm_half8(q0 ^ 0x80808080u, q1 ^ 0x80808080u, (_Float16)1152.0f);
	}
};

/* the split of one token block: the 8 values of a lane group scaled by the
 * block's 2^e (the 4 groups of a block are lanes l, l ^ 16, l ^ 32, l ^ 48) */
__device__ static inline void qmm_split8(const float (&v)[8], half8_t &hi, half8_t &lo,
					 float &unscale)
{
	float m = 0.0f;
#pragma unroll
	for (int k = 0; k < 8; k++)
		m = fmaxf(m, fabsf(v[k]));
	m = fmaxf(m, __shfl_xor(m, 16, WAVE));
	m = fmaxf(m, __shfl_xor(m, 32, WAVE));
	/* 2^sh * m in [2^13, 2^14); a zero block keeps sh = 0 */
	int sh = 0;
	if (m > 0.0f) {
		const int ex = (int)((__builtin_bit_cast(u32, m) >> 23) & 0xffu) - 127;
		sh = 13 - ex;
		sh = sh > 100 ? 100 : sh < -100 ? -100 : sh;
	}
	const float s = __builtin_bit_cast(float, (u32)(sh + 127) << 23);
#pragma unroll
	for (int k = 0; k < 8; k++) {
		const float y = v[k] * s;
		const _Float16 h = (_Float16)y;
		hi[k] = h;
		lo[k] = (_Float16)(y - (float)h);
	}
	unscale = __builtin_bit_cast(float, (u32)(127 - sh) << 23);
}

/*
 * Grid (ceil(N / 64), ceil(T / 16), K / (64 PZ)), four waves.  PZ: pairs of
 * blocks per workgroup.  part (grid z > 1): [z][T][N] partial sums.
 */
template <int WT, int PZ>
__global__ __launch_bounds__(QMM_WAVES * WAVE) void k_qmm(
	const uint8_t *__restrict__ W, size_t rb, int N, int K, const float *__restrict__ x, int T,
	const float *__restrict__ add, int add_rows, float *__restrict__ out,
	float *__restrict__ part)
{
	typedef qmm_pair<WT> P;
	constexpr int BB = WT == 1 ? 34 : 18, NB = 2 * PZ;
	__shared__ uint4 s_hi[NB][4][QMM_TOK], s_lo[NB][4][QMM_TOK];
	/* read as float4: 16-byte aligned whatever else the LDS holds */
	__shared__ __attribute__((aligned(16))) float s_ts[NB][QMM_TOK];
	const int wave = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
	const int r = lane & 15, g = lane >> 4;
	const int n = blockIdx.x * (QMM_WAVES * QMM_ROWS) + wave * QMM_ROWS + r;
	const int t0 = blockIdx.y * QMM_TOK, z = blockIdx.z;
	/* rows past N repeat the last row (their results are not stored) */
	const uint8_t *row = W + (size_t)min(n, N - 1) * rb + (size_t)z * PZ * 2 * BB;
	u32 w[PZ][P::DW];
#pragma unroll
	for (int p = 0; p < PZ; p++)
		P::load(row + (size_t)p * 2 * BB, g, w[p]);

	/* the tokens' blocks of this stretch, split into LDS: thread item i =
	 * (block, group, token), the token fastest, so a wave's stores are 1 KB
	 * contiguous (with the group fastest every lane of a wave hit the same
	 * banks); all of a thread's loads go out before any is used (a loop
	 * that waited for each made the staging eight round trips) */
	constexpr int IT = QMM_TOK * NB * 4 / (QMM_WAVES * WAVE); /* items per thread */
	float v[IT][8];
#pragma unroll
	for (int u = 0; u < IT; u++) { /* every load first: one round trip */
		const int i = (int)threadIdx.x + u * QMM_WAVES * WAVE;
		const int t = i & 15, gg = (i >> 4) & 3, b = i >> 6;
		float4 p = {0.0f, 0.0f, 0.0f, 0.0f}, q = p;
		if (t0 + t < T) {
			const float *xb = x + (size_t)(t0 + t) * K + (size_t)(z * NB + b) * 32;
			p = WT == 1 ? ((const float4 *)(xb + 8 * gg))[0] : *(const float4 *)(xb + 4 * gg);
			q = WT == 1 ? ((const float4 *)(xb + 8 * gg))[1]
				    : *(const float4 *)(xb + 16 + 4 * gg);
		}
		v[u][0] = p.x; v[u][1] = p.y; v[u][2] = p.z; v[u][3] = p.w;
		v[u][4] = q.x; v[u][5] = q.y; v[u][6] = q.z; v[u][7] = q.w;
	}
#pragma unroll
	for (int u = 0; u < IT; u++) {
		const int i = (int)threadIdx.x + u * QMM_WAVES * WAVE;
		const int t = i & 15, gg = (i >> 4) & 3, b = i >> 6;
		half8_t hi, lo;
		float us;
		qmm_split8(v[u], hi, lo, us);
		s_hi[b][gg][t] = __builtin_bit_cast(uint4, hi);
		s_lo[b][gg][t] = __builtin_bit_cast(uint4, lo);
		if (gg == 0)
			s_ts[b][t] = us;
	}
	__syncthreads();

	floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
	for (int p = 0; p < PZ; p++) {
#pragma unroll
		for (int h = 0; h < 2; h++) {
			const int b = 2 * p + h;
			float d;
			const half8_t bq = P::operand(w[p], h, d);
			const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
			floatx4 blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(
				__builtin_bit_cast(half8_t, s_hi[b][g][r]), bq, zero, 0, 0, 0);
			blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(
				__builtin_bit_cast(half8_t, s_lo[b][g][r]), bq, blk, 0, 0, 0);
			const float4 s = *(const float4 *)&s_ts[b][4 * g];
			acc[0] = __builtin_fmaf(d * s.x, blk[0], acc[0]);
			acc[1] = __builtin_fmaf(d * s.y, blk[1], acc[1]);
			acc[2] = __builtin_fmaf(d * s.z, blk[2], acc[2]);
			acc[3] = __builtin_fmaf(d * s.w, blk[3], acc[3]);
		}
		/* one pair at a time: left to itself the scheduler issued every
		 * MFMA first and held all 64 results (256 AGPRs: one wave per
		 * SIMD) */
		__builtin_amdgcn_sched_barrier(0);
	}
	if (n >= N)
		return;
#pragma unroll
	for (int j = 0; j < 4; j++) {
		const int t = t0 + 4 * g + j;
		if (t >= T)
			continue;
		const size_t o = (size_t)t * N + n;
		if (gridDim.z == 1)
			out[o] = (add ? add[add_rows ? o : (size_t)n] : 0.0f) + acc[j];
		else
			part[(size_t)z * T * N + o] = acc[j];
	}
}

/* out = add + the stretches' partial sums, added in stretch order */
__global__ __launch_bounds__(256) void k_qmm_reduce(const float *__restrict__ part, int KS,
						     size_t TN, int N, const float *__restrict__ add,
						     int add_rows, float *__restrict__ out)
{
	const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
	if (o >= TN)
		return;
	float s = part[o];
	for (int k = 1; k < KS; k++)
		s += part[(size_t)k * TN + o];
	out[o] = (add ? add[add_rows ? o : o % (size_t)N] : 0.0f) + s;
}

/* ---------------------------------------------------------------------- */
/* the product of many tokens                                              */
/* ---------------------------------------------------------------------- */

#define QT_WAVES 8
#define QT_COLS 128 /* columns of K per stage: 4 blocks */

/* geometry of TM 32-token groups and NW column waves: rows, bytes of a row's
 * stage, stage bytes */
template <int WT, int NW, int TM> struct qt_geo {
	static constexpr int TOK = 32 * TM; /* tokens of a tile */
	/* LDS bytes of one 16-byte chunk of every token; the padding starts a
	 * wave's four chunks 16 banks apart */
	static constexpr int CHUNK = TOK * 16 + 64;
	static constexpr int XB = 32 * CHUNK;           /* a stage's tokens: 16 chunks of hi, 16 of lo */
	static constexpr int TPR = QT_WAVES * WAVE / TOK; /* threads that stage a token */
	static constexpr int BB = WT == 1 ? 34 : 18;
	static constexpr int NR = 32 * NW;
	static constexpr int RB = 4 * BB, DW = RB / 4;
	/* dwords a thread loads; the last ones may repeat the last row past the tile */
	static constexpr int J = (NR * DW + QT_WAVES * WAVE - 1) / (QT_WAVES * WAVE);
	static constexpr int WB = J * QT_WAVES * WAVE * 4;
	static constexpr int SB = XB + WB; /* one stage */
	static constexpr int LDS = 2 * SB + 2 * 4 * TOK * 4; /* and the scales of its blocks */
};

/* a lane's share of block b (parity ODD) of its row's stage in LDS: raw
 * dwords, then the unscaled operands (elements 16 kh + 8 h .. + 7, in the order
 * 0 2 1 3 4 6 5 7) and the block scale */
template <int WT, int ODD> struct qt_blk;

template <int ODD> struct qt_blk<2, ODD> {
	u32 q[3], sc;
	__device__ inline void load(const uint8_t *blk, int h)
	{
		const u32 *a = (const u32 *)(blk + 8 * h + (ODD ? 2 : 0));
		q[0] = a[0];
		q[1] = a[1];
		q[2] = ODD ? 0u : a[2];
		sc = *(const u32 *)(blk - (ODD ? 2 : 0));
	}
	__device__ inline void operands(half8_t (&k)[2], float &d) const
	{
		typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
		const half2_t lo = {(_Float16)-1032.0f, (_Float16)-1032.0f};
		const half2_t r16 = {(_Float16)0.0625f, (_Float16)0.0625f};
		const half2_t hi = {(_Float16)-72.0f, (_Float16)-72.0f};
		const u32 q0 = ODD ? q[0] : __builtin_amdgcn_alignbit(q[1], q[0], 16);
		const u32 q1 = ODD ? q[1] : __builtin_amdgcn_alignbit(q[2], q[1], 16);
		const u32 w[4] = {q0, q0 >> 8, q1, q1 >> 8};
		half2_t a[4], b[4];
#pragma unroll
		for (int i = 0; i < 4; i++) { /* 1024 + n, and 1024 + 16 n: both exact */
			a[i] = __builtin_bit_cast(half2_t, (w[i] & 0x000f000fu) | 0x64006400u) + lo;
			b[i] = __builtin_elementwise_fma(
				__builtin_bit_cast(half2_t, (w[i] & 0x00f000f0u) | 0x64006400u), r16, hi);
		}
		k[0] = half8_t{a[0][0], a[0][1], a[1][0], a[1][1], a[2][0], a[2][1], a[3][0], a[3][1]};
		k[1] = half8_t{b[0][0], b[0][1], b[1][0], b[1][1], b[2][0], b[2][1], b[3][0], b[3][1]};
		d = f16_bits_to_f32(ODD ? sc >> 16 : sc & 0xffffu);
	}
};

template <int ODD> struct qt_blk<1, ODD> {
	u32 q[6], sc;
	__device__ inline void load(const uint8_t *blk, int h)
	{
		const u32 *a = (const u32 *)(blk + 8 * h + (ODD ? 2 : 0));
		q[0] = a[0];
		q[1] = a[1];
		q[2] = ODD ? 0u : a[2];
		q[3] = a[4];
		q[4] = a[5];
		q[5] = ODD ? 0u : a[6];
		sc = *(const u32 *)(blk - (ODD ? 2 : 0));
	}
	__device__ inline void operands(half8_t (&k)[2], float &d) const
	{
		typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
		const half2_t off = {(_Float16)-1152.0f, (_Float16)-1152.0f};
#pragma unroll
		for (int kh = 0; kh < 2; kh++) {
			const u32 *p = q + 3 * kh;
			u32 v[2] = {p[0], p[1]};
			if (!ODD) {
				v[0] = __builtin_amdgcn_alignbit(p[1], p[0], 16);
				v[1] = __builtin_amdgcn_alignbit(p[2], p[1], 16);
			}
			half2_t a[4];
#pragma unroll
			for (int i = 0; i < 2; i++) { /* signed bytes: q ^ 0x80 = q + 128 */
				const u32 u = v[i] ^ 0x80808080u;
				a[2 * i] = __builtin_bit_cast(half2_t, qmm_magic(u, 0x04020400u)) + off;
				a[2 * i + 1] = __builtin_bit_cast(half2_t, qmm_magic(u, 0x04030401u)) + off;
			}
			k[kh] = half8_t{a[0][0], a[0][1], a[1][0], a[1][1],
					a[2][0], a[2][1], a[3][0], a[3][1]};
		}
		d = f16_bits_to_f32(ODD ? sc >> 16 : sc & 0xffffu);
	}
};

/*
 * NBK blocks of a stage for one wave: 32 TM tokens x 32 rows, each block's sums
 * scaled by the row's block scale and the tokens' (their product is exact)
 * and added to acc.  In steps of half a block, ordered by hand: a step's MFMAs
 * run beside the next step's LDS reads and the unpacking of the block after
 * (left to itself the compiler reads each operand right before its MFMA and
 * waits out the LDS latency every time).  TM = 2: a step is a group of 32
 * tokens, and the fp32 steps of the last one's sums stand beside its MFMAs.
 * TM = 1: a step is the hi or the lo operands, and the last block's fp32 steps
 * come before the next one's MFMAs (the SIMD's other waves fill in; a second
 * set of sums, beside the 128 registers of two workgroups a CU, spilled).
 */
template <int WT, int NBK, int TM>
__device__ static inline void qt_blocks(const uint8_t *row, const uint8_t *sx, const float *sts, int r,
					int h, floatx16 (&acc)[TM])
{
	constexpr int BB = qt_geo<WT, 8, TM>::BB, CH = qt_geo<WT, 8, TM>::CHUNK, TOK = 32 * TM;
	constexpr int NQ = 2 * TM; /* MFMAs of a step */
	qt_blk<WT, 0> we;
	qt_blk<WT, 1> wo;
	half8_t k[2][2], a[2][NQ]; /* k: [block & 1][kh]; a: [step & 1][kh, and hi or lo] */
	floatx16 s[TM];
	floatx4 ts[TM][4]; /* scales of the lane's tokens 8 i + 4 h .. + 3 of a group */
	float d[2];
	auto reada = [&](int step) {
		const int b = step / 2, u = step % 2;
#pragma unroll
		for (int q = 0; q < NQ; q++) {
			const int p = TM == 2 ? q / 2 : u, kh = q % 2, t = TM == 2 ? u : 0;
			a[step & 1][q] = *(const half8_t *)(sx + (16 * p + 4 * b + 2 * kh + h) * CH +
							    (32 * t + r) * 16);
		}
	};
	auto readts = [&](int b, int t) {
#pragma unroll
		for (int i = 0; i < 4; i++)
			ts[t][i] = *(const floatx4 *)(sts + b * TOK + 32 * t + 8 * i + 4 * h);
	};
	/* acc += the sums of block b and token group t, scaled */
	auto add = [&](int b, int t) {
#pragma unroll
		for (int j = 0; j < 16; j++)
			acc[t][j] = __builtin_fmaf(d[b & 1] * ts[t][j / 4][j % 4], s[t][j], acc[t][j]);
		/* in this step: left to itself the compiler puts every block's fp32
		 * steps behind the last MFMA and spills the sums until then */
		asm volatile("" : "+v"(acc[t]));
	};
	we.load(row, h);
	wo.load(row + BB, h);
	reada(0);
	we.operands(k[0], d[0]);
	__builtin_amdgcn_sched_barrier(0);
#pragma unroll
	for (int step = 0; step < 2 * NBK; step++) {
		const int b = step / 2, u = step % 2, f = b & 1, t = TM == 2 ? u : 0;
		if (step + 1 < 2 * NBK)
			reada(step + 1);
		if (TM == 2)
			readts(b, u);
		else if (u == 0 && b > 0)
			readts(b - 1, 0);
		if (u == 0) { /* block b + 2's bytes, over block b's, which k holds */
			if (b + 2 < NBK) {
				if (f == 0)
					we.load(row + (b + 2) * BB, h);
				else
					wo.load(row + (b + 2) * BB, h);
			}
		} else if (b + 1 < NBK) {
			if (f == 0)
				wo.operands(k[1], d[1]);
			else
				we.operands(k[0], d[0]);
		}
		if (TM == 1 && u == 0 && b > 0)
			add(b - 1, 0);
#pragma unroll
		for (int q = 0; q < NQ; q++) {
			const floatx16 z = {};
			s[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
				a[step & 1][q], k[f][q % 2], q == 0 && (TM == 2 || u == 0) ? z : s[t], 0, 0, 0);
		}
		if (TM == 2 && step > 0) /* the next step's unpacking replaces its d */
			add((step - 1) / 2, (step - 1) % 2);
		__builtin_amdgcn_sched_group_barrier(0x100, 8, 0);
#pragma unroll
		for (int i = 0; i < NQ; i++) {
			__builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
			__builtin_amdgcn_sched_group_barrier(0x2, 16, 0);
		}
		__builtin_amdgcn_sched_barrier(0);
	}
	if (TM == 1)
		readts(NBK - 1, 0);
	add(NBK - 1, TM - 1);
}

/* the maximum over eight neighbouring lanes: lanes ^ 1, ^ 2, the other four
 * mirrored */
__device__ static inline u32 qt_max8(u32 m)
{
	m = max(m, (u32)__builtin_amdgcn_mov_dpp((int)m, 0xb1, 0xf, 0xf, true));
	m = max(m, (u32)__builtin_amdgcn_mov_dpp((int)m, 0x4e, 0xf, 0xf, true));
	return max(m, (u32)__builtin_amdgcn_mov_dpp((int)m, 0x141, 0xf, 0xf, true));
}

/*
 * A token's 128 columns of a stage, held by TPR = 8 or 16 threads (thread i:
 * the float4s i, i + TPR, ...: eight neighbouring threads hold a block), each
 * block scaled by a power of two of its own (its largest magnitude into
 * [2^13, 2^14)) and split into hi and lo.  Scales stop at 2^125: below that
 * all bits of a value fit the two parts, and the inverse times a weight's f16
 * scale is exact in fp32.
 */
template <int TPR, int CH, int TOK>
__device__ static inline void qt_stage(const float4 (&v)[32 / TPR], uint8_t *sx, float *ts, int row, int i)
{
	typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
#pragma unroll
	for (int j = 0; j < 32 / TPR; j++) {
		/* magnitudes compare as their bits do */
		const u32 m = qt_max8(__builtin_bit_cast(
			u32, fmaxf(fmaxf(fabsf(v[j].x), fabsf(v[j].y)), fmaxf(fabsf(v[j].z), fabsf(v[j].w)))));
		/* exponent 13 - m's, 125 at most (a zero block's too) */
		const u32 sb = min((267u << 23) - (m & 0x7f800000u), 252u << 23);
		const float s = __builtin_bit_cast(float, sb);
		/* element order 0, 2, 1, 3: a weight operand's */
		const floatx4 y = {v[j].x * s, v[j].z * s, v[j].y * s, v[j].w * s};
		const half4_t hi = __builtin_convertvector(y, half4_t);
		const half4_t lo = __builtin_convertvector(y - __builtin_convertvector(hi, floatx4), half4_t);
		const int f = i + TPR * j; /* of the token's 32 float4s: block f / 8 */
		uint8_t *o = sx + (f >> 1) * CH + row * 16 + (f & 1) * 8;
		*(half4_t *)o = hi;
		*(half4_t *)(o + 16 * CH) = lo;
		if (f % 8 == 0)
			ts[(f / 8) * TOK + row] = __builtin_bit_cast(float, (254u << 23) - sb);
	}
}

/*
 * out = add + x . W^T, a workgroup of eight waves per (32 TM tokens, 32 NW rows):
 * NW waves side by side on the rows, and 8 / NW groups of them on the blocks
 * of a stage (128 columns of K), whose sums are added at the end in group
 * order.  The raw weights of a stage come by LDS-DMA and the tokens through
 * registers, split on their way into LDS, both one stage ahead in the other
 * of two buffers: one barrier a stage, and no scratch memory, so calls on one
 * matrix may overlap and be captured.
 *
 * Bound: the VALU (the tokens' split, the unpacking, a multiplication and an
 * FMA per block and output) and the MFMAs, which overlap only in part: about
 * 500 and 32 instructions a wave of a 64 x 256 stage, 4,000 and 2,050 of its
 * 7,000 cycles, in a single workgroup per CU (LDS); two 32 x 128 ones fit.
 * Q4_0 6144 x 4096, calls back to back: 333 tokens 926 -> 94 us (the per-token
 * product, which takes the weights once per token), 1024 tokens against
 * k_qmm 908 -> 190; 4096 x 4096, 1024 tokens 608 -> 106.  One scale per token
 * and 128 columns would save the multiplications (333 tokens 88, 1024 tokens
 * 171) but cost the blocks below their neighbours bits.  Tried with that form
 * at 333 tokens (91 there): 32 tokens x 64 rows a wave (half the operand reads,
 * twice the unpacking) 101; splitting the tokens at opposite ends of a stage
 * in a SIMD's two waves 96; without the hand-made order 104.  Tried with this
 * one: the scales as a byte each in LDS (a quarter of their reads, a shift
 * more per output) 128; the tokens' loads where the compiler puts them, right
 * before their use, 103; the split as two mixed FMAs a value (fma_mixlo / hi, a
 * third fewer instructions in the split, the same bits) 2% slower.
 */
template <int WT, int NW, int TM>
__global__ __launch_bounds__(QT_WAVES * WAVE, TM == 1 ? 4 : 2) void k_qmm_tile(
	const uint8_t *__restrict__ W, size_t rb, int N, int K, const float *__restrict__ x, int T,
	const float *__restrict__ add, int add_rows, float *__restrict__ out)
{
	typedef qt_geo<WT, NW, TM> G;
	constexpr int KG = QT_WAVES / NW, GB = 4 / KG; /* K groups; blocks of a stage each takes */
	__shared__ __attribute__((aligned(16))) uint8_t qt_lds[G::LDS];
	float *s_ts = (float *)(qt_lds + 2 * G::SB); /* [2][4][TOK] */
	const int tid = threadIdx.x, lane = tid % WAVE;
	const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
	const int r = lane & 31, h = lane >> 5, wn = wave % NW, wk = wave / NW;
	const int tiles = (T + G::TOK - 1) / G::TOK, cols = (N + G::NR - 1) / G::NR;
	/* class id % 8 (an XCD) takes a contiguous run of items, a column block's
	 * token tiles side by side: they share its weights in that L2 */
	const int per = (tiles * cols + 7) / 8, item = ((int)blockIdx.x % 8) * per + (int)blockIdx.x / 8;
	if ((int)blockIdx.x / 8 >= per || item >= tiles * cols)
		return; /* the whole workgroup */
	const int t0 = item % tiles * G::TOK, n0 = item / tiles * G::NR;
	const int row = tid / G::TPR, i = tid % G::TPR;
	/* tokens past T repeat the last one, rows past N the last row (never stored) */
	const float4 *xp = (const float4 *)(x + (size_t)min(t0 + row, T - 1) * K) + i;
	const uint8_t *wb = W + (size_t)n0 * rb;
	u32 woff[G::J];
#pragma unroll
	for (int j = 0; j < G::J; j++) {
		const int f = (wave * G::J + j) * WAVE + lane, wr = min(f / G::DW, G::NR - 1);
		woff[j] = (u32)min(wr, N - 1 - n0) * (u32)rb + (u32)(f % G::DW) * 4u;
	}
	const u32 l0 = __builtin_amdgcn_readfirstlane(lds_addr(qt_lds));
	auto issue = [&](int s) {
		const u32 lb = l0 + (u32)((s & 1) * G::SB + G::XB + wave * G::J * WAVE * 4);
#pragma unroll
		for (int j = 0; j < G::J; j++)
			dma_dword(wb + (size_t)s * G::RB, woff[j], lb + (u32)(j * WAVE * 4));
	};
	float4 v[32 / G::TPR];
	floatx16 tot[TM] = {};
	const int ns = K / QT_COLS;
	auto fetch = [&](int s) {
#pragma unroll
		for (int j = 0; j < 32 / G::TPR; j++)
			v[j] = xp[(size_t)min(s, ns - 1) * (QT_COLS / 4) + G::TPR * j];
	};
	issue(0);
	fetch(0);
	qt_stage<G::TPR, G::CHUNK, G::TOK>(v, qt_lds, s_ts, row, i);
	for (int s = 0; s < ns;) {
		/* sums of 512 columns first, as k_qmm's: a chain over all of K = 4096
		 * left 1.32e-7 (relative L2 against float64), these 1.06e-7, k_qmm 1.15e-7 */
		floatx16 acc[TM] = {};
#pragma unroll 1
		for (const int e = min(s + 4, ns); s < e; s++) {
			const int b = s & 1;
			const uint8_t *sx = qt_lds + b * G::SB, *sw = sx + G::XB + (wn * 32 + r) * G::RB;
			uint8_t *nx = qt_lds + (b ^ 1) * G::SB;
			wait_vm<0>();    /* this wave's part of the stage's weights */
			__syncthreads(); /* stage s is whole; the other buffer is free */
			if (s + 1 < ns)
				issue(s + 1);
			fetch(s + 1);
			__builtin_amdgcn_sched_barrier(0); /* not down to their use */
			/* group wk: blocks GB wk .. of the stage */
			qt_blocks<WT, GB, TM>(sw + wk * GB * G::BB, sx + wk * 4 * GB * G::CHUNK,
					      s_ts + (4 * b + wk * GB) * G::TOK, r, h, acc);
			/* the last stage's is not read: under a condition the compiler would
			 * move the loads there, and the wait for them */
			qt_stage<G::TPR, G::CHUNK, G::TOK>(v, nx, s_ts + 4 * (b ^ 1) * G::TOK, row, i);
		}
#pragma unroll
		for (int t = 0; t < TM; t++)
			tot[t] += acc[t];
	}
	if constexpr (KG > 1) { /* group 1's sums to group 0 */
		__syncthreads();
		float *p = (float *)qt_lds + (size_t)wn * 16 * TM * WAVE + lane;
		if (wk == 1) {
#pragma unroll
			for (int j = 0; j < 16 * TM; j++)
				p[j * WAVE] = tot[j / 16][j % 16];
		}
		__syncthreads();
		if (wk == 1)
			return;
#pragma unroll
		for (int j = 0; j < 16 * TM; j++)
			tot[j / 16][j % 16] += p[j * WAVE];
	}
	const int n = n0 + wn * 32 + r;
	if (n >= N)
		return;
#pragma unroll
	for (int t = 0; t < TM; t++)
#pragma unroll
		for (int j = 0; j < 16; j++) {
			const int tk = t0 + 32 * t + 8 * (j / 4) + 4 * h + j % 4;
			if (tk >= T)
				continue;
			const size_t o = (size_t)tk * N + n;
			out[o] = (add ? add[add_rows ? o : (size_t)n] : 0.0f) + tot[t][j];
		}
}

/* ---------------------------------------------------------------------- */
/* host                                                                    */
/* ---------------------------------------------------------------------- */

static int qmm_pz(int K)
{
	return K / 64 < QMM_PZ ? K / 64 : QMM_PZ;
}

static bool qmm_supported(int wtype, int K)
{
	return (wtype == 1 || wtype == 2) && K >= 256 && K % 256 == 0 &&
	       (K <= 64 * QMM_PZ ? ((K / 256) & (K / 256 - 1)) == 0 : K % (64 * QMM_PZ) == 0);
}

/* the partial sums of a call with K longer than one stretch */
extern "C" size_t moe_qmm_work_bytes(int T, int N, int K)
{
	const int KS = K / (64 * qmm_pz(K));
	return KS > 1 ? (size_t)KS * T * N * sizeof(float) : 0;
}

/* stretches of 64 * PZ columns the product of K columns splits into (its
 * partial sums are KS slices of T * N floats when KS > 1) */
extern "C" int moe_qmm_stretches(int K)
{
	return K / (64 * qmm_pz(K));
}

/* parts_only: KS > 1 and only the partial sums, left for the caller to add
 * in stretch order (k_qmm_reduce's sum) */
static int launch_qmm(int wtype, const uint8_t *W, int N, int K, const float *x, int T,
		      const float *add, int add_rows, float *out, void *work, bool parts_only,
		      void *stream)
{
	if (!qmm_supported(wtype, K) || N < 1 || T < 1 || (size_t)T * N > 0xffffffffull)
		return (int)hipErrorInvalidValue;
	const int PZ = qmm_pz(K), KS = K / (64 * PZ);
	if ((T + QMM_TOK - 1) / QMM_TOK > 65535 || (KS > 1 && !work) || (parts_only && KS < 2))
		return (int)hipErrorInvalidValue;
	const size_t rb = (size_t)(K / 32) * (wtype == 1 ? 34 : 18);
	const dim3 grid((N + QMM_WAVES * QMM_ROWS - 1) / (QMM_WAVES * QMM_ROWS),
			(T + QMM_TOK - 1) / QMM_TOK, KS),
		blk(QMM_WAVES * WAVE);
	hipStream_t s = (hipStream_t)stream;
	float *part = (float *)work;
	bool done = false;
#define QMM(WTT, PP)                                                                        \
	if (!done && wtype == WTT && PZ == PP) {                                            \
		hipLaunchKernelGGL((k_qmm<WTT, PP>), grid, blk, 0, s, W, rb, N, K, x, T, add,   \
				   add_rows, out, part);                                    \
		done = true;                                                                \
	}
	QMM(1, 4) QMM(1, 8)
	QMM(2, 4) QMM(2, 8)
#undef QMM
	if (!done)
		return (int)hipErrorInvalidValue;
	if (KS > 1 && !parts_only) {
		const size_t TN = (size_t)T * N;
		hipLaunchKernelGGL(k_qmm_reduce, dim3((unsigned)((TN + 255) / 256)), dim3(256), 0, s,
				   part, KS, TN, N, add, add_rows, out);
	}
	return (int)hipGetLastError();
}

extern "C" int moe_launch_qmm(int wtype, const uint8_t *W, int N, int K, const float *x, int T,
			      const float *add, int add_rows, float *out, void *work,
			      void *stream)
{
	return launch_qmm(wtype, W, N, K, x, T, add, add_rows, out, work, false, stream);
}

extern "C" int moe_launch_qmm_parts(int wtype, const uint8_t *W, int N, int K, const float *x,
				    int T, void *work, void *stream)
{
	return launch_qmm(wtype, W, N, K, x, T, NULL, 0, NULL, work, true, stream);
}

/* 256-workgroup rounds (one per CU) of tiles of tok tokens x nr rows */
static long long tile_rounds(int N, int T, int tok, int nr)
{
	return ((long long)((T + tok - 1) / tok) * ((N + nr - 1) / nr) + 255) / 256;
}

#define SMALL_ROUNDS(N, T) tile_rounds(N, T, 32, 128)
#define WIDE_ROUNDS(N, T) tile_rounds(N, T, 64, 256)

/* A round of 64 x 256 tiles (one workgroup per CU) takes 93 us at K = 4096, of
 * 32 x 128 tiles (two fit, each then half as fast) 35.  Small / wide in us
 * (calls back to back), Q4_0: 6144 x 4096 T = 160 47 / 93, T = 256 69 / 94, T =
 * 333 98 / 93, T = 768 168 / 189, T = 1024 213 / 192; 4096 x 4096 T = 512 72 / 94,
 * T = 768 112 / 101, T = 1024 144 / 106; 2048 x 2048 T = 1024 38 / 52; 50304 x 2048
 * T = 32 36 / 52, T = 48 67 / 52; 32000 x 4096 T = 48 70 / 94.  (64 x 128 tiles, one
 * per CU, were never more than a tenth better than both.) */
static bool tile_wide(int N, int T)
{
	return 8 * WIDE_ROUNDS(N, T) < 3 * SMALL_ROUNDS(N, T);
}

/* Whether moe_launch_qmm_tile is faster than moe_launch_qmm: a workgroup of
 * k_qmm (16 tokens, 64 rows, 512 columns) takes about 22 ns of the whole
 * chip, a round of tiles 9.8 (small) or 23 ns (wide) per column of K.  k_qmm /
 * tiles in us, Q4_0, calls back to back: 6144 x 4096 T = 17 36 / 39, T = 33 50 /
 * 40; 4096 x 4096 T = 48 38 / 40, T = 64 48 / 40; 2048 x 2048 T = 64 17 / 22; 6144 x
 * 2048 T = 32 22 / 22, T = 33 30 / 22; 50304 x 2048 T = 2 60 / 36, T = 16 69 / 37;
 * 32000 x 4096 T = 2 73 / 42, T = 16 83 / 43 */
extern "C" int moe_qmm_tile_better(int N, int T)
{
	const long long w = (long long)((T + QMM_TOK - 1) / QMM_TOK) * ((N + 63) / 64);
	return w > 228 * SMALL_ROUNDS(N, T) || w > 540 * WIDE_ROUNDS(N, T);
}

extern "C" size_t moe_qmm_work_most(int T, int N, int K)
{
	while (T > 0 && moe_qmm_tile_better(N, T))
		T--;
	return moe_qmm_work_bytes(T, N, K);
}

template <int WT, int NW, int TM>
static hipError_t launch_tile(const uint8_t *W, size_t rb, int N, int K, const float *x, int T,
			      const float *add, int add_rows, float *out, hipStream_t s)
{
	typedef qt_geo<WT, NW, TM> G;
	const long long items = (long long)((T + G::TOK - 1) / G::TOK) * ((N + G::NR - 1) / G::NR);
	if (items > 0x7fffff00ll)
		return hipErrorInvalidValue;
	hipLaunchKernelGGL((k_qmm_tile<WT, NW, TM>), dim3((unsigned)((items + 7) / 8 * 8)),
			   dim3(QT_WAVES * WAVE), 0, s, W, rb, N, K, x, T, add, add_rows, out);
	return hipGetLastError();
}

extern "C" int moe_launch_qmm_tile(int wtype, const uint8_t *W, int N, int K, const float *x, int T,
				   const float *add, int add_rows, float *out, void *stream)
{
	if (!qmm_supported(wtype, K) || N < 1 || T < 1)
		return (int)hipErrorInvalidValue;
	const size_t rb = (size_t)(K / 32) * (wtype == 1 ? 34 : 18);
	hipStream_t s = (hipStream_t)stream;
	if (tile_wide(N, T))
		return (int)(wtype == 1 ? launch_tile<1, 8, 2>(W, rb, N, K, x, T, add, add_rows, out, s)
					: launch_tile<2, 8, 2>(W, rb, N, K, x, T, add, add_rows, out, s));
	return (int)(wtype == 1 ? launch_tile<1, 4, 1>(W, rb, N, K, x, T, add, add_rows, out, s)
				: launch_tile<2, 4, 1>(W, rb, N, K, x, T, add, add_rows, out, s));
}
