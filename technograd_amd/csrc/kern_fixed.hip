// Q16.16 row programs one instruction at a time: every instruction of a row
// program (tg_kern.h: rp_ins) as a launch over all (element, row) pairs of a
// pass, on the interpreter's arena ([slot][R], consecutive rows in
// consecutive words). For programs without think loops, whose rows all run
// the same instructions, that are too large to compile: the interpreter
// (kern_rowprog.hip) gives a row to one lane, so a pass there is one lane's
// chain of loads per term, whatever the rows. The element functions
// (tg_rowdev.h) are the interpreter's, and sums of products are exact
// integers, so the results are the same.
#include "tg_kern.h"
#include "tg_rowdev.h"
#include "tgm.h"

using namespace tgrd;

namespace {

// unary and binary functions by op; each op's loop is chosen once per launch
template <class F>
__device__ inline void fx_un_each(int op, F f)
{
	switch (op) {
#define UN(K, fn) \
	case K: f([](int x) { return fn(x); }); break;
		UN(TGM_NEG, negq) UN(TGM_TANH, tanhq) UN(TGM_RELU, reluq) UN(TGM_SIGMOID, sigmoidq) UN(TGM_EXP, expq) UN(TGM_SQRT, sqrtq)
		UN(TGM_GELU, geluq) UN(TGM_SILU, siluq) UN(TGM_SOFTPLUS, softplusq) UN(TGM_LOG, logq) UN(TGM_SIN, sinq) UN(TGM_COS, cosq)
		UN(TGM_FLOOR, floorq)
#undef UN
	case -1: f([](int x) { return x; }); break;
	default: f([](int x) { return stepq(x); }); break;
	}
}

__device__ inline int fx_bin(int op, int x, int y)
{
	switch (op) {
	case TGK_ADD: return addq(x, y);
	case TGK_SUB: return subq(x, y);
	case TGK_MUL: return fmulq(x, y);
	case TGK_DIV: return fdivq(x, y);
	case TGK_MAX: return maxq(x, y);
	default: return minq(x, y);
	}
}

__device__ inline int at(const tgk_fx &x, long i, int r) { return x.p[i * x.st + r * x.ls]; }

// words that no kernel writes while this one runs: read through scalar loads when the address is the wave's
typedef const int __attribute__((address_space(4))) *cword;

// Products with shared weights: a lane per row, so an input is one coalesced
// load, and CH channels per lane, whose weights are the same for the whole
// wave: they come through scalar loads, CH words at a time from the packed
// copy [C/16][K][16], and a term is one v_mad_i64_i32 with a scalar operand.
// Four waves of a block take neighbouring channels of the same 64 rows. It is
// bound by VALU issue and, for the rest, by loads: at 16384 rows, 64 inputs to
// 256 channels and 256 to 256, a SIMD issues an instruction (four cycles,
// v_mad_i64_i32 too) in 70 % of its cycles, and its four waves wait 41 % of
// theirs. 16384 rows x 256 inputs x 256 channels take 65 us, a 64-256-256-16
// MLP's pass of those rows 138 us; the interpreter took 12.5 ms for it.
template <int CH>
__global__ __launch_bounds__(256) void fx_mm_k(tgk_fx_mm d)
{
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int cb = (blockIdx.y * 4 + wave) * CH;
	if (cb >= d.C) return;
	const int row = blockIdx.x * 64 + lane, rc = row < d.rows ? row : d.rows - 1;
	cword w = (cword)(d.w + (long)(cb / 16) * d.K * 16 + cb % 16);
	for (int q = blockIdx.z; q < d.nq; q += gridDim.z) {
		const int *xq = d.x.p + rc * d.x.ls + q * d.xq * d.x.st;
		const long xs = d.xp * d.x.st;
		long acc[CH];
#pragma unroll
		for (int c = 0; c < CH; c++) acc[c] = 0;
		constexpr int U = 4; // terms whose loads are in flight together
		int p = 0;
		for (; p + U <= d.K; p += U) {
			int x[U];
#pragma unroll
			for (int u = 0; u < U; u++) x[u] = xq[(p + u) * xs];
#pragma unroll
			for (int u = 0; u < U; u++)
#pragma unroll
				for (int c = 0; c < CH; c++) acc[c] += (long)w[(p + u) * 16 + c] * x[u];
		}
		for (; p < d.K; p++) {
			const int x = xq[p * xs];
#pragma unroll
			for (int c = 0; c < CH; c++) acc[c] += (long)w[p * 16 + c] * x;
		}
		if (row >= d.rows) continue;
		fx_un_each(d.uop, [&](auto f) {
#pragma unroll
			for (int c = 0; c < CH; c++)
				if (cb + c < d.C) {
					const int v = d.qscale ? qscaleq(acc[c], d.qscale[cb + c]) : sat((acc[c] + 32768) >> 16);
					d.o[((cb + c) * d.oc + q * d.oq) * d.R + row] = f(v);
				}
		});
	}
}

// products of two row values (attention): one output per thread
__global__ __launch_bounds__(256) void fx_mmrow_k(int *o, long R, tgk_fx a, tgk_fx b, int G, int M, int K, int N, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (int g = blockIdx.z; g < G; g += gridDim.z)
		for (long e = blockIdx.y; e < (long)M * N; e += gridDim.y) {
			const long i = e / N, j = e - i * N, ai = ((long)g * M + i) * K, bj = (long)g * K * N + j;
			long s = 0;
#pragma unroll 4
			for (int p = 0; p < K; p++) s += (long)at(a, ai + p, row) * at(b, bj + (long)p * N, row);
			o[((long)g * M * N + e) * R + row] = sat((s + 32768) >> 16);
		}
}

__global__ __launch_bounds__(256) void fx_bin_k(int op, int *o, long R, tgk_fx a, int am, const int *amap, tgk_fx b, int bm, const int *bmap,
						int n, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (int i = blockIdx.y; i < n; i += gridDim.y)
		o[i * R + row] = fx_bin(op, at(a, am == 0 ? i : am == 1 ? 0 : amap[i], row), at(b, bm == 0 ? i : bm == 1 ? 0 : bmap[i], row));
}

__global__ __launch_bounds__(256) void fx_un_k(int op, int *o, long R, tgk_fx a, int n, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	fx_un_each(op, [&](auto f) {
		for (int i = blockIdx.y; i < n; i += gridDim.y) o[i * R + row] = f(at(a, i, row));
	});
}

// softmax or rmsnorm: a lane per line and row
__global__ __launch_bounds__(256) void fx_row_k(int op, int *o, long R, tgk_fx a, int nrow, int cols, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (int q = blockIdx.y; q < nrow; q += gridDim.y) {
		const long base = (long)q * cols;
		int *y = o + base * R + row;
		if (op == TGM_SOFTMAX) {
			int mx = at(a, base, row);
			for (int i = 1; i < cols; i++) mx = maxq(mx, at(a, base + i, row));
			long s = 0;
			for (int i = 0; i < cols; i++) {
				const int e = expq_neg(subq(at(a, base + i, row), mx)); // x - max <= 0
				y[i * R] = e;
				s += e;
			}
			for (int i = 0; i < cols; i++) y[i * R] = softq(y[i * R], s);
		} else {
			unsigned long ss = 0;
			for (int i = 0; i < cols; i++) {
				const long x = at(a, base + i, row);
				ss += (unsigned long)(x * x);
			}
			const int rms = rmsq(ss, cols);
			for (int i = 0; i < cols; i++) y[i * R] = fdivq(at(a, base + i, row), rms);
		}
	}
}

__global__ __launch_bounds__(256) void fx_red_k(int op, int *o, tgk_fx a, int n, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	long s = 0;
#pragma unroll 4
	for (int i = 0; i < n; i++) s += at(a, i, row);
	o[row] = op == TGM_SUM ? sat(s) : sat(s / n);
}

__global__ __launch_bounds__(256) void fx_trans_k(int *o, long R, tgk_fx a, int RR, int C, long n, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (long e = blockIdx.y; e < n; e += gridDim.y) {
		const long z = e / ((long)RR * C), rem = e - z * RR * C, i = rem / C, j = rem - i * C;
		o[(z * RR * C + j * RR + i) * R + row] = at(a, e, row);
	}
}

__global__ __launch_bounds__(256) void fx_outer_k(int *o, long R, tgk_fx a, int m, tgk_fx b, int n, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (long e = blockIdx.y; e < (long)m * n; e += gridDim.y) o[e * R + row] = fmulq(at(a, e / n, row), at(b, e % n, row));
}

__global__ __launch_bounds__(256) void fx_copy_k(int *o, long R, long ooff, tgk_fx a, long aoff, int n, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (int i = blockIdx.y; i < n; i += gridDim.y) o[(ooff + i) * R + row] = at(a, aoff + i, row);
}

__global__ __launch_bounds__(256) void fx_take_k(int *o, long R, tgk_fx w, tgk_fx idx, int cnt, int d, int h, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row >= rows) return;
	for (long e = blockIdx.y; e < (long)cnt * h; e += gridDim.y) {
		const long i = e / h, rr = ((long)at(idx, i, row) + 32768) >> 16;
		o[e * R + row] = rr >= 0 && rr < d ? at(w, rr * h + (e - i * h), row) : 0;
	}
}

__global__ __launch_bounds__(256) void fx_fill_k(int *o, int stride, int v, int rows)
{
	const int row = blockIdx.x * 256 + threadIdx.x;
	if (row < rows) o[(long)row * stride] = v;
}

// [rows][n] <-> [n][R] in tiles of 64 x 64 through LDS: both sides move whole runs of 64 words
constexpr int FT = 64;
__global__ __launch_bounds__(256) void fx_in_k(int *o, long R, const int *in, int n, int rows)
{
	__shared__ int z[FT][FT + 1];
	const int r0 = blockIdx.x * FT, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	for (int i0 = blockIdx.y * FT; i0 < n; i0 += gridDim.y * FT) {
		for (int r = w; r < FT; r += 4)
			if (r0 + r < rows && i0 + lane < n) z[lane][r] = in[(long)(r0 + r) * n + i0 + lane];
		__syncthreads();
		for (int i = w; i < FT; i += 4)
			if (i0 + i < n && r0 + lane < rows) o[(long)(i0 + i) * R + r0 + lane] = z[i][lane];
		__syncthreads();
	}
}

__global__ __launch_bounds__(256) void fx_out_k(int *out, tgk_fx a, int n, int rows)
{
	__shared__ int z[FT][FT + 1];
	const int r0 = blockIdx.x * FT, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	for (int i0 = blockIdx.y * FT; i0 < n; i0 += gridDim.y * FT) {
		for (int i = w; i < FT; i += 4)
			if (i0 + i < n && r0 + lane < rows) z[lane][i] = at(a, i0 + i, r0 + lane);
		__syncthreads();
		for (int r = w; r < FT; r += 4)
			if (r0 + r < rows && i0 + lane < n) out[(long)(r0 + r) * n + i0 + lane] = z[r][lane];
		__syncthreads();
	}
}

inline unsigned blk(long n, int per) { return (unsigned)((n + per - 1) / per); }
// rows in x, elements in y (the kernels walk what lies past the grid)
inline dim3 grid2(int rows, long n) { return dim3(blk(rows, 256), (unsigned)(n < 65535 ? n : 65535)); }

} // namespace

void tgk_fx_mul(hipStream_t s, const tgk_fx_mm *d)
{
	if (d->rows <= 0 || d->C <= 0 || d->nq <= 0) return;
	const unsigned nz = d->nq < 65535 ? (unsigned)d->nq : 65535u;
	// 16 channels a lane use an input 16 times; with too few waves for that to fill the chip, four
	if ((long)blk(d->rows, 64) * blk(d->C, 16) * d->nq >= 1024) fx_mm_k<16><<<dim3(blk(d->rows, 64), blk(d->C, 64), nz), 256, 0, s>>>(*d);
	else fx_mm_k<4><<<dim3(blk(d->rows, 64), blk(d->C, 16), nz), 256, 0, s>>>(*d);
}

void tgk_fx_mulrow(hipStream_t s, int *o, long R, tgk_fx a, tgk_fx b, int G, int M, int K, int N, int rows)
{
	dim3 g = grid2(rows, (long)M * N);
	g.z = (unsigned)(G < 65535 ? G : 65535);
	fx_mmrow_k<<<g, 256, 0, s>>>(o, R, a, b, G, M, K, N, rows);
}

void tgk_fx_binary(hipStream_t s, int op, int *o, long R, tgk_fx a, int am, const int *amap, tgk_fx b, int bm, const int *bmap, int n, int rows)
{
	fx_bin_k<<<grid2(rows, n), 256, 0, s>>>(op, o, R, a, am, amap, b, bm, bmap, n, rows);
}

void tgk_fx_unary(hipStream_t s, int op, int *o, long R, tgk_fx a, int n, int rows) { fx_un_k<<<grid2(rows, n), 256, 0, s>>>(op, o, R, a, n, rows); }

void tgk_fx_rowop(hipStream_t s, int op, int *o, long R, tgk_fx a, int nrow, int cols, int rows)
{
	fx_row_k<<<grid2(rows, nrow), 256, 0, s>>>(op, o, R, a, nrow, cols, rows);
}

void tgk_fx_reduce(hipStream_t s, int op, int *o, tgk_fx a, int n, int rows) { fx_red_k<<<blk(rows, 256), 256, 0, s>>>(op, o, a, n, rows); }

void tgk_fx_transpose(hipStream_t s, int *o, long R, tgk_fx a, int g, int r, int c, int rows)
{
	const long n = (long)g * r * c;
	fx_trans_k<<<grid2(rows, n), 256, 0, s>>>(o, R, a, r, c, n, rows);
}

void tgk_fx_outer(hipStream_t s, int *o, long R, tgk_fx a, int m, tgk_fx b, int n, int rows)
{
	fx_outer_k<<<grid2(rows, (long)m * n), 256, 0, s>>>(o, R, a, m, b, n, rows);
}

void tgk_fx_copy(hipStream_t s, int *o, long R, long ooff, tgk_fx a, long aoff, int n, int rows)
{
	fx_copy_k<<<grid2(rows, n), 256, 0, s>>>(o, R, ooff, a, aoff, n, rows);
}

void tgk_fx_take(hipStream_t s, int *o, long R, tgk_fx w, tgk_fx idx, int cnt, int d, int h, int rows)
{
	fx_take_k<<<grid2(rows, (long)cnt * h), 256, 0, s>>>(o, R, w, idx, cnt, d, h, rows);
}

void tgk_fx_fill(hipStream_t s, int *o, int stride, int v, int rows) { fx_fill_k<<<blk(rows, 256), 256, 0, s>>>(o, stride, v, rows); }

void tgk_fx_in(hipStream_t s, int *o, long R, const int *in, int n, int rows)
{
	if (n > 0) fx_in_k<<<dim3(blk(rows, FT), blk(n, FT) < 65535 ? blk(n, FT) : 65535), 256, 0, s>>>(o, R, in, n, rows);
}

void tgk_fx_out(hipStream_t s, int *out, tgk_fx a, int n, int rows)
{
	if (n > 0) fx_out_k<<<dim3(blk(rows, FT), blk(n, FT) < 65535 ? blk(n, FT) : 65535), 256, 0, s>>>(out, a, n, rows);
}
