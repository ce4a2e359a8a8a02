// The per-head output projections of a decoder, all heads in one product:
//   o[row][c] = ((o_0 + o_1) + ...) + o_{nh-1},
//   o_h = scale_h[c] * (sum_k code_h[c][k] x[row][h][k])
// with every o_h the value the quantized GEMM (kern_qgemm.hip) computes for
// that head's line (exact integer sums on the line's grid, one rounding, the
// scale; split lines and the reference's loop the same), and the heads added
// in order in f32, as the graph's adds do. The lines' digits are made by the
// GEMM's digit kernels with lines in head-major order (line = h rp + row, rp
// the rows padded to 32), so a head's 32 rows are one MFMA fragment. Written
// head by head the products are nh times the output: 16 heads' 537 MB for a
// prompt of 8192 tokens x 1024 channels, written once and read back once.
#include "tg_kern.h"
#include "tg_qdigits.h"

#include <string.h>

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

namespace {

struct Heads {
	tgk_heads_args a;
	tgk_qdig q;
	const int8_t *w; // [nh Dp / 32][Kp / 32][64][16] (tgk_qweight's int8 layout)
	const float *scale;
	int Kp, nout;
};

// code (head h, channel c, input k)
__device__ inline int head_code(const Heads &d, int h, int c, int k)
{
	const long ch = (long)h * d.a.Dp + c;
	return d.w[((ch >> 5) * (d.Kp / 32) + (k >> 5)) * 1024 + ((ch & 31) + 32 * ((k >> 4) & 1)) * 16 + (k & 15)];
}

// One head's product before its scale: T = sum_l plane_l 256^l, an integer
// below 2^40, times 2^(E - 23), rounded once. The planes' sums are at most
// 2^22 in magnitude (|code|, |digit| <= 128, K <= 256), so the lower two
// combine in int32, and with the upper 16 bits of that added to the third, T
// = A 65536 + B, |A| < 2^23 and 0 <= B < 2^16: both exact in f32, and one
// fused multiply-add rounds T once. The power of two is exact where the
// result is a normal number, which |T| >= 1 and E >= -100 make it; below, in
// f64 (a wave's lines all above, which nearly all are, skip that).
__device__ inline float head_sum(int acc0, int acc1, int acc2, float p2)
{
	const int lo = acc0 + acc1 * 256;
	return __builtin_fmaf((float)(acc2 + (lo >> 16)), 65536.0f, (float)(lo & 0xffff)) * p2;
}
__device__ inline float head_sum64(int acc0, int acc1, int acc2, int E)
{
	return (float)ldexp(__builtin_fma((double)acc2, 65536.0, (double)(acc0 + acc1 * 256)), E - 23);
}

// the same of any line, from the line itself: its grid, a split line's grid and outliers, or the reference's loop
__device__ inline float line_value(const Heads &d, int h, int row, int c, int E, int cls)
{
	if (cls & 1) { // the reference's sequential loop (TGQ_REF, or a candidate no resolve has seen)
		const float *x = d.a.x + (long)row * d.a.xrow + (long)h * d.a.xhead;
		float t = 0.0f;
		for (int k = 0; k < d.a.HD; k++) t += (float)head_code(d, h, c, k) * x[k];
		return t;
	}
	const long line = (long)h * d.a.rp + row;
	const int8_t *q = d.q.dig + (line >> 5) * (d.Kp / 32) * 3072 + (line & 31) * 16;
	int acc[3] = { 0, 0, 0 };
	for (int k = 0; k < d.a.HD; k++) {
		const int code = head_code(d, h, c, k);
		for (int l = 0; l < 3; l++) acc[l] += code * q[(k >> 5) * 3072 + ((k >> 4) & 1) * 512 + l * 1024 + (k & 15)];
	}
	double o = 0.0; // its outliers, in input order
	for (int j = 0; cls != TGQ_GRID && j < d.nout; j++) {
		const int k = d.q.ok[line * d.nout + j];
		if (k < 0) break;
		o += (double)head_code(d, h, c, k) * (double)d.q.ox[line * d.nout + j];
	}
	return (float)(ldexp(__builtin_fma((double)acc[2], 65536.0, (double)(acc[0] + acc[1] * 256)), E - 23) + o);
}

// A step's rows: a block per 16 rows x 16 channels, a wave per head (in
// turns), whose digits and weights all load at once into
// v_mfma_i32_16x16x64_i8's operands; the heads' values meet in LDS, HG heads'
// at a time, and 256 threads add them in order. A head's product is a load's
// latency and six matrix instructions; what bounds the kernel is the bytes a
// compute unit takes in (128 KB a block at 16 heads of 128). 33 steps of 16
// sequences through a layer of 72 heads of 64: 4.0 ms, 25.5 with a product
// per head, as more heads than HG ran before, and 3.3 with 64 heads.
constexpr int HG = 64; // heads whose values fit 64 KiB of LDS
template <int NS>
__global__ __launch_bounds__(1024) void heads_step_k(Heads d)
{
	extern __shared__ float red[]; // [min(nh, HG)][16 rows][16 channels]
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = blockDim.x >> 6;
	const int tc = (d.a.D + 15) / 16, r0 = (int)(blockIdx.x / (unsigned)tc) * 16, c0 = (int)(blockIdx.x % (unsigned)tc) * 16;
	const int r = lane & 15, g = lane >> 4, nkb = d.Kp / 32;
	const int t = threadIdx.x;
	float s = 0.0f; // of threads 0 .. 255: their output's sum so far
	for (int h0 = 0; h0 < d.a.nh; h0 += HG) {
		const int hn = d.a.nh - h0 < HG ? d.a.nh - h0 : HG;
		if (h0) __syncthreads(); // the values before are added
		for (int h = h0 + wave; h < h0 + hn; h += W) {
			const long line0 = (long)h * d.a.rp + r0, ch0 = (long)h * d.a.Dp + c0;
			const int8_t *A = d.q.dig + (line0 >> 5) * nkb * 3072 + ((line0 & 31) + r) * 16 + (g & 1) * 512 + (g >> 1) * 3072;
			const int8_t *B = d.w + (ch0 >> 5) * nkb * 1024 + (g >> 1) * 1024 + ((g & 1) * 32 + (ch0 & 31) + r) * 16;
			v4i af[NS][3], bf[NS];
#pragma unroll
			for (int i = 0; i < NS; i++) {
				bf[i] = *(const v4i *)(B + i * 2048);
#pragma unroll
				for (int l = 0; l < 3; l++) af[i][l] = *(const v4i *)(A + i * 6144 + l * 1024);
			}
			const int c = c0 + r;
			const float sc = d.scale[ch0 + r];
			int E[4], cls[4];
#pragma unroll
			for (int v = 0; v < 4; v++) E[v] = d.q.e[line0 + 4 * g + v], cls[v] = d.q.special[line0 + 4 * g + v];
			v4i acc[3] = { { 0, 0, 0, 0 }, { 0, 0, 0, 0 }, { 0, 0, 0, 0 } };
#pragma unroll
			for (int i = 0; i < NS; i++)
#pragma unroll
				for (int l = 0; l < 3; l++) acc[l] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[i][l], bf[i], acc[l], 0, 0, 0);
#pragma unroll
			for (int v = 0; v < 4; v++) {
				const int row = r0 + 4 * g + v;
				const int cl = row < d.a.rows && c < d.a.D ? cls[v] : 0;
				red[(h - h0) * 256 + (4 * g + v) * 16 + r] = sc * (cl == TGQ_GRID ? head_sum64(acc[0][v], acc[1][v], acc[2][v], E[v]) : line_value(d, h, row, c, E[v], cl));
			}
		}
		__syncthreads();
		if (t >= 256) continue;
		for (int h = 0; h < hn; h++) s = h0 + h ? s + red[h * 256 + t] : red[t];
	}
	const int row = r0 + (t >> 4), c = c0 + (t & 15);
	if (t < 256 && row < d.a.rows && c < d.a.D) d.a.o[(long)row * d.a.orow + c] = s;
}

// A prompt's rows: a block of 8 waves takes 64 rows x 128 channels, a wave 32
// x 32 of them: per head three planes' int32 sums, then their values added to
// the running f32 sums in registers. A stage is CB 32-input blocks of a
// head's digits and weights (40 KiB at 128 inputs) in one of two LDS buffers;
// the next stage's loads are in flight in registers while one is multiplied.
// A wave's loads, matrix instructions and arithmetic (about ten VALU
// instructions per head and output) follow one another, so the kernel lives
// on waves: two blocks a compute unit, four waves a SIMD. 8192 rows x 16 heads
// of 128 x 1024 channels: 129 us and 38 us of digits (138 with a wave's tile
// twice as wide and two waves a SIMD); head by head the products took 244 us,
// their digits 94, and the norm that added them 41 more than it does now.
template <int CB>
__global__ __launch_bounds__(512, 4) void heads_prompt_k(Heads d)
{
	constexpr int AB = 2 * CB * 3, BB = 4 * CB, NP = AB + BB, NL = (NP + 7) / 8; // 1 KiB pieces of a stage, per wave
	__shared__ __align__(16) int8_t lds[2][NL * 8 * 1024];
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = wave & 1, wn = wave >> 1;
	const int tc = d.a.Dp / 128;
	int id = blockIdx.x; // neighbouring tiles of the same rows on one XCD: its L2 serves their digits
	if (gridDim.x % 8 == 0) id = (id % 8) * (gridDim.x / 8) + id / 8;
	const int r0 = id / tc * 64, c0 = id % tc * 128, nkb = d.Kp / 32, nch = nkb / CB, rb = d.a.rp / 32;
	if (c0 >= d.a.D) return;
	// piece p of a stage: digits of row block p / (3 CB), then weights of channel block (p - AB) / CB; its address in
	// the stage to be loaded next (pieces past the last repeat it)
	v4i st[NL];
	const int8_t *src[NL];
#pragma unroll
	for (int i = 0; i < NL; i++) {
		const int p = wave * NL + i < NP ? wave * NL + i : NP - 1;
		const int blk = r0 / 32 + p / (3 * CB), bb = blk < rb ? blk : 0; // (a row block past the rows: not stored)
		src[i] = p < AB ? d.q.dig + (long)bb * nkb * 3072 + p % (3 * CB) * 1024
				: d.w + (long)(c0 / 32 + (p - AB) / CB) * nkb * 1024 + (p - AB) % CB * 1024;
	}
	int nextch = 0; // the chunk of its head that the next stage is
	auto fetch = [&]() {
		const bool head = ++nextch == nch; // then on to the next head's first
		if (head) nextch = 0;
#pragma unroll
		for (int i = 0; i < NL; i++) {
			const bool isA = wave * NL + i < AB;
			st[i] = *(const v4i *)(src[i] + lane * 16);
			const long hs = isA ? (long)rb * nkb * 3072 : (long)d.a.Dp / 32 * nkb * 1024, cs = isA ? CB * 3072 : CB * 1024;
			src[i] += head ? hs - (nch - 1) * cs : cs;
		}
	};
	auto stash = [&](int b) {
#pragma unroll
		for (int i = 0; i < NL; i++) *(v4i *)&lds[b][(wave * NL + i) * 1024 + lane * 16] = st[i];
	};
	const int mrow = r0 + wm * 32, c = c0 + wn * 32 + (lane & 31); // this wave's first row, the lane's channel
	float sum[16];
#pragma unroll
	for (int v = 0; v < 16; v++) sum[v] = 0.0f;
	fetch();
	stash(0);
	int b = 0;
	for (int h = 0; h < d.a.nh; h++) {
		// the lines' exponents and classes (lane: row lane % 32) and the channels' scales, needed after the products
		const int lrow = mrow + (lane & 31);
		const long line = (long)h * d.a.rp + (lrow < d.a.rp ? lrow : 0);
		const int El = d.q.e[line];
		int cl = d.q.special[line];
		if (lrow >= d.a.rows) cl = 0;
		const float p2l = ldexpf(1.0f, El - 23), sc = d.scale[(long)h * d.a.Dp + c];
		v16i acc[3];
		auto mul = [&](int kb, bool first) {
			const v4i bf = *(const v4i *)&lds[b][(AB + wn * CB + kb) * 1024 + lane * 16];
			const v16i zero = { 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0 };
#pragma unroll
			for (int l = 0; l < 3; l++) {
				const v4i af = *(const v4i *)&lds[b][((wm * CB + kb) * 3 + l) * 1024 + lane * 16];
				acc[l] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af, bf, first ? zero : acc[l], 0, 0, 0);
			}
		};
		__syncthreads(); // the stage is in LDS, and the other buffer's readers are done
		if (nch > 1 || h + 1 < d.a.nh) fetch();
#pragma unroll
		for (int kb = 0; kb < CB; kb++) mul(kb, kb == 0);
		b ^= 1;
		for (int ch = 1; ch < nch; ch++) {
			stash(b);
			__syncthreads();
			if (ch + 1 < nch || h + 1 < d.a.nh) fetch();
#pragma unroll
			for (int kb = 0; kb < CB; kb++) mul(kb, false);
			b ^= 1;
		}
		float o[16];
#pragma unroll
		for (int v = 0; v < 16; v++) {
			const float p2 = __shfl(p2l, 8 * (v / 4) + 4 * (lane >> 5) + v % 4);
			o[v] = sc * head_sum(acc[0][v], acc[1][v], acc[2][v], p2);
		}
		// lines off their grid (or far below 1), one after another: a channel's value per lane, handed to those that hold the line
		for (unsigned bad = (unsigned)__ballot(cl != 0 || (El < -100 && lrow < d.a.rows)); bad; bad &= bad - 1) {
			const int lr = __builtin_ctz(bad);
			const float t = line_value(d, h, mrow + lr, c < d.a.D ? c : d.a.D - 1, __shfl(El, lr), __shfl(cl, lr));
#pragma unroll
			for (int v = 0; v < 16; v++)
				if (8 * (v / 4) + 4 * (lane >> 5) + v % 4 == lr) o[v] = sc * t;
		}
#pragma unroll
		for (int v = 0; v < 16; v++) sum[v] = h ? sum[v] + o[v] : o[v];
		if (h + 1 < d.a.nh) stash(b);
	}
#pragma unroll
	for (int v = 0; v < 16; v++) {
		const int row = mrow + 8 * (v / 4) + 4 * (lane >> 5) + v % 4;
		if (row < d.a.rows && c < d.a.D) d.a.o[(long)row * d.a.orow + c] = sum[v];
	}
}

} // namespace

bool tgk_heads(hipStream_t st, const tgk_heads_args *a, void *scratch)
{
	const tgk_qweight *w = a->w;
	if (!w || w->bits != 8 || a->rows <= 0 || a->nh <= 0 || a->HD <= TGK_REFLOOP_K || a->HD > TGK_HEADS_MAX || a->rp % 32 || a->rp < a->rows ||
	    a->Dp % 256)
		return false;
	tgk_qgemm_args g;
	memset(&g, 0, sizeof g);
	g.w = w, g.x = a->x, g.xr = a->xhead, g.xj = a->xrow, g.xk = 1, g.ni = a->rp, g.M = a->nh * a->rp;
	if (!a->digits) tgk_qgemm_digits(st, &g, scratch);
	const Heads d{ *a, tgk_qgemm_digit_area(scratch, g.M, w->Kp), (const int8_t *)w->w, w->scale, w->Kp, tgq_nout(w->Kp) };
	// from 1024 rows 64 x 128 tiles fill a quarter of the chip and more; below, 16 x 16 tiles with the heads side by side
	if (a->rows >= 1024) {
		const unsigned grid = (unsigned)((a->rows + 63) / 64 * (a->Dp / 128));
		if (w->Kp % 128 == 0) heads_prompt_k<4><<<grid, 512, 0, st>>>(d);
		else heads_prompt_k<2><<<grid, 512, 0, st>>>(d);
		return true;
	}
	const unsigned grid = (unsigned)((a->rows + 15) / 16 * ((a->D + 15) / 16));
	const int W = a->nh < 4 ? 4 : a->nh < 16 ? a->nh : 16;
	const size_t lds = (size_t)(a->nh < HG ? a->nh : HG) * 1024;
	switch (w->Kp / 64) {
	case 1: heads_step_k<1><<<grid, W * 64, lds, st>>>(d); break;
	case 2: heads_step_k<2><<<grid, W * 64, lds, st>>>(d); break;
	case 3: heads_step_k<3><<<grid, W * 64, lds, st>>>(d); break;
	default: heads_step_k<4><<<grid, W * 64, lds, st>>>(d); break;
	}
	return true;
}
