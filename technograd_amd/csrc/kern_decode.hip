// Kernels of the KV-cache decoder (tg_decode.cpp) for models in the Qwen3
// importer's layout (examples/qwen3/import.py). Each computes the values the
// fixed-length graph computes, with the same f32 operations in the same
// order (this file is compiled with -ffp-contract=off), so a decoded token's
// logits equal the fixed-length forward's at that position bit for bit.
#include "tg_kern.h"
#include "tg_devmath.h"
#include "tg_qdigits.h"

#include <math.h>

namespace {

// RoPE on the normed, scaled q and k lines of a chunk of token rows (row =
// s * T0 + i at position p0 + i): v = x * cos[p] + (x @ Rot) * sin[p], as the
// graph's `x * cosT + (x @ Rot) * sinT`. q lines go to qr [rows][NQ][HD], k
// lines to the K cache; the chunk's v vectors (columns after q and k of the
// projection output) go to the V cache.
__global__ void rope_cache_k(tgk_dec_rope_args a, long total)
{
	const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
	if (t >= total) return;
	const int NL = a.NQ + 2 * a.NKV; // lines per token row: q, k, v
	const long row = t / ((long)NL * a.HD);
	const int rem = (int)(t - row * NL * a.HD), line = rem / a.HD, d = rem - line * a.HD;
	const int s = (int)(row / a.T0), p = a.p0 + (int)(row - (long)s * a.T0);
	float *kv_s = (float *)0;
	if (line >= a.NQ) kv_s = (line < a.NQ + a.NKV ? a.K : a.V) + (long)s * a.kv_seq + a.kv_layer;
	if (line < a.NQ + a.NKV) {
		const long i = (row * (a.NQ + a.NKV) + line) * a.HD + d;
		const float x = a.hq[i], r = a.rt[i];
		const float c = a.cosT[(long)p * a.HD + d], sn = a.sinT[(long)p * a.HD + d];
		const float v = x * c + r * sn;
		if (line < a.NQ) a.qr[(row * a.NQ + line) * a.HD + d] = v;
		else kv_s[((long)(line - a.NQ) * a.P + p) * a.HD + d] = v;
	} else {
		const int j = line - a.NQ - a.NKV;
		kv_s[((long)j * a.P + p) * a.HD + d] = a.qkv[row * a.ctot + (long)(a.NQ + a.NKV) * a.HD + (long)j * a.HD + d];
	}
}

// The same values four at a time: block y takes token rows y, y + gridDim.y,
// ..., a thread four consecutive d of one line (HD % 4 == 0, every operand
// 16-byte aligned: the launcher checks), so a row's sequence and position
// come from one 32-bit division, not two 64-bit ones per element.
__global__ __launch_bounds__(256) void rope_cache4_k(tgk_dec_rope_args a, int rows)
{
	const int NL = a.NQ + 2 * a.NKV, HD4 = a.HD / 4;
	const int e = blockIdx.x * 256 + threadIdx.x; // (line, quad) of a token row
	if (e >= NL * HD4) return;
	const int line = e / HD4, d = (e - line * HD4) * 4;
	auto rot = [](float x, float c, float r, float sn) { return x * c + r * sn; };
	for (int row = blockIdx.y; row < rows; row += gridDim.y) {
		const int s = row / a.T0, p = a.p0 + (row - s * a.T0);
		float *kv_s = nullptr;
		if (line >= a.NQ) kv_s = (line < a.NQ + a.NKV ? a.K : a.V) + (long)s * a.kv_seq + a.kv_layer;
		if (line < a.NQ + a.NKV) {
			const long i = ((long)row * (a.NQ + a.NKV) + line) * a.HD + d;
			const float4 x = *(const float4 *)(a.hq + i), r = *(const float4 *)(a.rt + i);
			const float4 c = *(const float4 *)(a.cosT + (long)p * a.HD + d), sn = *(const float4 *)(a.sinT + (long)p * a.HD + d);
			const float4 v = make_float4(rot(x.x, c.x, r.x, sn.x), rot(x.y, c.y, r.y, sn.y), rot(x.z, c.z, r.z, sn.z),
						     rot(x.w, c.w, r.w, sn.w));
			if (line < a.NQ) *(float4 *)(a.qr + ((long)row * a.NQ + line) * a.HD + d) = v;
			else *(float4 *)(kv_s + ((long)(line - a.NQ) * a.P + p) * a.HD + d) = v;
		} else {
			const int j = line - a.NQ - a.NKV;
			*(float4 *)(kv_s + ((long)j * a.P + p) * a.HD + d) =
				*(const float4 *)(a.qkv + (long)row * a.ctot + (long)(a.NQ + a.NKV) * a.HD + (long)j * a.HD + d);
		}
	}
}

// Digits, exponent, class and sum of q of line L of K <= 256 inputs by one
// wave, inputs 4 lane .. 4 lane + 3 in v (zeros from K on); z holds the line
// in LDS for the resolve of a candidate that the coarse test leaves.
__device__ inline void wave_digits(const float *v, const float *z, int K, int Kp, const tgk_qdig &q, int L, TgqHist *hist)
{
	const int lane = threadIdx.x & 63;
	unsigned mb = 0;
	tgq_scan4(v, mb);
	mb = tgq_wave_umax(mb);
	float amax;
	int nan;
	tgq_scan_end(mb, amax, nan);
	const int special = tgq_special(nan, amax), E = tgq_exponent(amax, special);
	int8_t *blk = tgq_row_base(q.dig, L, Kp);
	TgqRowSums s{};
	tgq_quad(blk, 4 * lane, 4 * lane < Kp, v, E, special, s);
	const int cls = tgq_row_class(s, special);
	if (lane == 0) q.e[L] = E, q.special[L] = cls, q.qsum[L] = s.qs;
	if (cls != TGQ_CAND) return;
	tgq_wave_sync();
	const int nout = tgq_nout(Kp);
	auto ld = [&](int g, float *x) {
		for (int u = 0; u < 16; u++) x[u] = 16 * g + u < K ? z[16 * g + u] : 0.0f;
	};
	tgq_resolve_row(hist, ld, K, Kp, E, blk, &q.qsum[L], &q.e[L], &q.special[L], q.ok + (long)L * nout, q.ox + (long)L * nout, nout, lane);
}

// One decode step's attention: one block per (sequence, KV head) for the GRP
// query heads sharing it, keys at positions 0 .. p. Per query head and key:
// score = sum_d q[d] k[d] in order from 0.0f, times the scale, plus the mask's
// 0; softmax with the reference's max rule, expf, a sequential sum and a
// division; out[d] = sum over keys of prob * v[d] in key order. The
// fixed-length graph's row for this position has further keys whose masked
// scores give probabilities of exactly 0: they change neither the max nor the
// sums. K, then V, stream through LDS in chunks of ck keys: every thread
// loads its share of the next chunk (16-byte loads) before the current one is
// used, so a chunk's loads are in flight while the previous chunk's chains
// run. Each score, each sum and each output stays one thread's sum in order:
// a (key, head) thread per score, a (head, d) thread per output, carried
// across chunks. LDS rows are HD + 4 floats apart: 16-byte reads of
// consecutive rows by consecutive lanes hit distinct banks. HD % 16 == 0.
// With Kp, a wave per query head then makes the digits of its outputs for the
// output projections (line head rp + s): they are at hand, and a launch of
// their own took a step 6.0 us a layer for 768 lines of 128; the attention
// takes 2 more (26.4 to 28.4 us, 48 sequences at 232 positions on average).
constexpr int ATT_TPB = 512, ATT_R = 4; // threads; float4 loads per thread and chunk

int attn_chunk(int HD) // keys per chunk: ATT_R float4 loads per thread, at most 64
{
	int ck = 64;
	while (ck > 1 && ck * (HD / 4) > ATT_R * ATT_TPB) ck >>= 1;
	return ck;
}

template <int GRP>
__global__ __launch_bounds__(ATT_TPB) void dec_attn_k(tgk_dec_attn_args a, int ck)
{
	extern __shared__ float4 sh4[];
	const int n = a.p + 1, HD = a.HD, H4 = HD / 4, KS = H4 + 1, nst = (n + 3) & ~3, per = ck * H4;
	float4 *kv = sh4;                  // [ck][KS] the staged chunk of K or V
	float *q = (float *)(kv + ck * KS); // [GRP][HD]
	float *sc = q + GRP * HD;           // [GRP][nst] scores, then probabilities
	float *lv = sc + GRP * nst;         // [GRP] max, then sum
	const int tid = threadIdx.x, s = blockIdx.x / a.NKV, j = blockIdx.x - s * a.NKV;
	const float *K = a.K + (long)s * a.kv_seq + a.kv_layer + (long)j * a.P * HD;
	const float *V = a.V + (long)s * a.kv_seq + a.kv_layer + (long)j * a.P * HD;
	float4 rg[ATT_R];
	auto fetch = [&](const float *base, int c0) { // chunk of keys c0 .. c0 + ck - 1 into registers
		for (int u = 0; u < ATT_R; u++) {
			const int e = tid + u * ATT_TPB, key = c0 + e / H4;
			rg[u] = e < per && key < n ? ((const float4 *)(base + (long)key * HD))[e % H4] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		}
	};
	auto stash = [&]() {
		for (int u = 0; u < ATT_R; u++) {
			const int e = tid + u * ATT_TPB;
			if (e < per) kv[(e / H4) * KS + e % H4] = rg[u];
		}
	};
	for (int e = tid; e < GRP * HD; e += ATT_TPB) q[e] = a.qr[((long)s * a.NQ + j * GRP) * HD + e];
	fetch(K, 0);
	for (int c0 = 0; c0 < n; c0 += ck) {
		__syncthreads(); // the previous chunk's chains are done with kv
		stash();
		__syncthreads();
		fetch(c0 + ck < n ? K : V, c0 + ck < n ? c0 + ck : 0); // next chunk (or V's first) in flight meanwhile
		for (int it = tid; it < ck * GRP; it += ATT_TPB) {
			const int g = it / ck, kk = it - g * ck;
			if (c0 + kk >= n) continue;
			const float4 *kr = kv + kk * KS, *qg = (const float4 *)(q + g * HD);
			float acc = 0.0f;
			for (int d4 = 0; d4 < H4; d4++) {
				const float4 k4 = kr[d4], q4 = qg[d4];
				acc = acc + q4.x * k4.x;
				acc = acc + q4.y * k4.y;
				acc = acc + q4.z * k4.z;
				acc = acc + q4.w * k4.w;
			}
			sc[g * nst + c0 + kk] = acc * a.scale + 0.0f;
		}
	}
	__syncthreads(); // the score chains are done with kv
	stash();         // V's first chunk (fetched during the last K chunk) into kv,
	if (ck < n) fetch(V, ck); // and its second in flight, both during the softmax
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
	for (int g = wave; g < GRP; g += ATT_TPB >> 6) { // max: a wave per query head
		const float *r = sc + g * nst;
		float m = -INFINITY;
		for (int key = 1 + lane; key < n; key += 64) m = fmaxf(m, r[key]);
		for (int w = 32; w > 0; w >>= 1) m = fmaxf(m, __shfl_xor(m, w));
		if (lane == 0) lv[g] = isnan(r[0]) ? r[0] : fmaxf(r[0], m);
	}
	__syncthreads();
	for (int e = tid; e < GRP * nst; e += ATT_TPB) {
		const int g = e / nst;
		if (e - g * nst < n) sc[e] = expf(sc[e] - lv[g]);
	}
	__syncthreads();
	if (tid < GRP) lv[tid] = tg_ordered_sum_pp<6>(sc + tid * nst, n);
	__syncthreads();
	for (int e = tid; e < GRP * nst; e += ATT_TPB) {
		const int g = e / nst;
		if (e - g * nst < n) sc[e] = sc[e] / lv[g];
	}
	constexpr int OI = (GRP * 256 + ATT_TPB - 1) / ATT_TPB; // outputs per thread (HD <= 256)
	float acc[OI];
	for (int u = 0; u < OI; u++) acc[u] = 0.0f;
	for (int c0 = 0; c0 < n; c0 += ck) {
		__syncthreads(); // probabilities final; the previous chunk's chains are done with kv
		if (c0 > 0) {    // (the first chunk is in kv already)
			stash();
			__syncthreads();
			if (c0 + ck < n) fetch(V, c0 + ck);
		}
		const int m = min(ck, n - c0);
		const float *vb = (const float *)kv;
		for (int u = 0; u < OI; u++) {
			const int it = tid + u * ATT_TPB;
			if (it >= GRP * HD) break;
			const int g = it / HD, d = it - g * HD;
			const float *r = sc + g * nst + c0;
			float x = acc[u];
			for (int kk = 0; kk < m; kk++) x = x + r[kk] * vb[kk * (HD + 4) + d];
			acc[u] = x;
		}
	}
	for (int u = 0; u < OI; u++) {
		const int it = tid + u * ATT_TPB;
		if (it >= GRP * HD) break;
		const int g = it / HD, d = it - g * HD;
		a.att[((long)s * a.NQ + j * GRP + g) * HD + d] = acc[u];
		q[it] = acc[u];
	}
	if (!a.Kp) return;
	__syncthreads(); // the heads' outputs are in q; kv is read, its room goes to the resolves (tgk_dec_attn_digits)
	if (wave >= GRP) return;
	const float4 o = 4 * lane < HD ? *(const float4 *)(q + wave * HD + 4 * lane) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	const float v[4] = { o.x, o.y, o.z, o.w };
	wave_digits(v, q + wave * HD, HD, a.Kp, a.q, (j * GRP + wave) * a.rp + s, (TgqHist *)kv + wave);
}

// four consecutive values of a line that starts at any float
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

// values i .. i + 3 of a line of n: one load, or single ones where the line ends within them (zeros past it)
__device__ inline void ld4(float *v, const float *p, int i, int n)
{
	if (i + 4 <= n) {
		const f4u f = *(const f4u *)(p + i);
		v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
	} else {
		for (int u = 0; u < 4; u++) v[u] = i + u < n ? p[i + u] : 0.0f;
	}
}
__device__ inline void st4(float *p, int i, int n, const float *v)
{
	if (i + 4 <= n) *(f4u *)(p + i) = f4u{ v[0], v[1], v[2], v[3] };
	else
		for (int u = 0; u < 4; u++)
			if (i + u < n) p[i + u] = v[u];
}

// a block's partial results, one entry per wave
struct BlkDigits {
	uint4 mb[4];                   // max |x| bits, 16 waves
	unsigned long long s[16][5]; // TgqRowSums
};

// Digits, exponent, class and sum of q of row m of K inputs, values z[0 .. Kp)
// in LDS (zero from K on; written before the call, its first barrier orders
// them), from this thread's scan mb of its share (tgq_scan4). Four inputs a
// thread and pass (tgq_quad); the waves' sums meet in LDS, where five lanes
// of the first wave add one quantity each. A candidate that the coarse test
// leaves is resolved by that wave (the row is in z).
__device__ inline void blk_digits(const float *z, int K, int Kp, unsigned mb, const tgk_qdig &q, int m, BlkDigits *red, TgqHist *hist)
{
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
	mb = tgq_wave_umax(mb);
	if (lane == 0) ((unsigned *)red->mb)[wave] = mb;
	if (tid >= nw && tid < 16) ((unsigned *)red->mb)[tid] = 0;
	__syncthreads();
	mb = 0;
	for (int i = 0; i < 4; i++) {
		const uint4 t = red->mb[i];
		mb = max(max(max(mb, t.x), max(t.y, t.z)), t.w);
	}
	mb = (unsigned)__builtin_amdgcn_readfirstlane((int)mb);
	float amax;
	int nan;
	tgq_scan_end(mb, amax, nan);
	const int special = tgq_special(nan, amax), E = tgq_exponent(amax, special);
	int8_t *blk = tgq_row_base(q.dig, m, Kp);
	TgqRowSums s{};
	for (int j0 = 0; j0 < Kp; j0 += 4 * blockDim.x) {
		const int k0 = j0 + 4 * tid;
		const bool in = k0 < Kp;
		const float4 f = in ? *(const float4 *)(z + k0) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		const float v[4] = { f.x, f.y, f.z, f.w };
		tgq_quad(blk, k0, in, v, E, special, s);
	}
	if (lane == 0) {
		unsigned long long *r = red->s[wave];
		r[0] = (unsigned long long)s.qs, r[1] = (unsigned long long)s.tl, r[2] = s.co.cnt, r[3] = s.co.s0, r[4] = s.co.s1;
	}
	__syncthreads();
	if (wave) return;
	unsigned long long t = 0;
#pragma unroll
	for (int w = 0; w < 16; w++) {
		const unsigned long long x = red->s[w < nw ? w : 0][lane < 5 ? lane : 0]; // (16 loads in flight, not one after another)
		t += w < nw ? x : 0ull;
	}
	auto of = [&](int l) {
		return (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)t, l) |
		       (unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)(unsigned)(t >> 32), l) << 32;
	};
	s.qs = (long long)of(0), s.tl = (long long)of(1), s.co = TgqCoarse{ of(2), of(3), of(4) };
	const int cls = tgq_row_class(s, special);
	if (lane == 0) q.e[m] = E, q.special[m] = cls, q.qsum[m] = s.qs;
	if (cls != TGQ_CAND) return;
	const int nout = tgq_nout(Kp);
	auto ld = [&](int g, float *v) {
		for (int i = 0; i < 16; i++) v[i] = z[16 * g + i];
	};
	tgq_resolve_row(hist, ld, K, Kp, E, blk, &q.qsum[m], &q.e[m], &q.special[m], q.ok + (long)m * nout, q.ox + (long)m * nout, nout, lane);
}

// tgk_dec_norm: one block per token row, a thread per four elements. The
// row's sum of squares is the reference's sequential loop over the squares
// (computed in parallel), the scale 1 / sqrtf(sum / D + 1e-6) as the row-op
// kernel, then (h * inv) * g.
// A few blocks of one row each, so latency is all: a load, the dependent adds
// of the row's sum, the digits' reductions. 48 rows of 1024 in 9.3 us; 13.6
// with 1024 threads of single elements, 16 inputs' digits a lane in one wave,
// the sums by shuffles and one thread's reads after them.
constexpr int NORM_MAX_TPB = TGK_DEC_NORM_MAX / 4;
__global__ __launch_bounds__(NORM_MAX_TPB) void dec_norm_k(tgk_dec_norm_args a)
{
	extern __shared__ float4 zs4[]; // [Kp] values, [Kp] squares (16-byte aligned)
	float *zs = (float *)zs4;
	__shared__ float inv_s;
	__shared__ BlkDigits red;
	__shared__ TgqHist hist;
	const int t = blockIdx.x, D = a.D, Kp = a.Kp, tid = threadIdx.x, i = 4 * tid;
	float *z = zs, *sq = zs + Kp, *hr = a.h + (long)t * a.hs;
	float v[4], g[4];
	ld4(v, hr, i, D);
	ld4(g, a.g, i, D);
	if (a.mode == 1) {
		float b[4];
		ld4(b, a.add + (long)t * a.adds, i, D);
		for (int u = 0; u < 4; u++) v[u] = v[u] + b[u];
	} else if (a.mode == 2) { // v + ((o_0 + o_1) + ... + o_{nh-1}), eight heads' loads at a time
		const float *o = a.o + (long)t * D;
		float acc[4];
		ld4(acc, o, i, D);
		for (int k0 = 1; k0 < a.nh; k0 += 8) {
			float b[8][4];
			for (int k = 0; k < 8; k++) ld4(b[k], o + (long)(k0 + k < a.nh ? k0 + k : 0) * a.ohead, i, D);
			for (int k = 0; k < 8 && k0 + k < a.nh; k++)
				for (int u = 0; u < 4; u++) acc[u] = acc[u] + b[k][u];
		}
		for (int u = 0; u < 4; u++) v[u] = v[u] + acc[u];
	}
	if (a.mode) st4(hr, i, D, v);
	if (i < Kp) *(float4 *)(sq + i) = make_float4(v[0] * v[0], v[1] * v[1], v[2] * v[2], v[3] * v[3]);
	__syncthreads();
	if (tid == 0) inv_s = 1.0f / sqrtf(tg_ordered_sum<8>(sq, D) / (float)D + 1e-6f);
	__syncthreads();
	const float inv = inv_s;
	float nv[4];
	for (int u = 0; u < 4; u++) nv[u] = i + u < D ? v[u] * inv * g[u] : 0.0f;
	st4(a.out + (long)t * a.outs, i, D, nv);
	if (i < Kp) *(float4 *)(z + i) = make_float4(nv[0], nv[1], nv[2], nv[3]);
	unsigned mb = 0;
	tgq_scan4(nv, mb);
	blk_digits(z, D, Kp, mb, a.q, t, &red, &hist);
}

// tgk_dec_hnorm: one wave per head line (4 per block, no block barrier:
// lines past the end leave at once), four elements a lane. Same operations
// as tgk_dec_norm. HD <= 256. 1152 lines of 128 in 5.8 us (8.1 with 16
// inputs' digits a lane, in 8 lanes of a wave).
__global__ __launch_bounds__(256) void dec_hnorm_k(tgk_dec_hnorm_args a)
{
	extern __shared__ float4 hs4[]; // per wave: [Kp] squares, then values (16-byte aligned)
	__shared__ TgqHist hist[4];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, L = blockIdx.x * 4 + w, HD = a.HD, Kp = a.Kp, i = 4 * lane;
	if (L >= a.rows * a.NH) return;
	const int t = L / a.NH, j = L - t * a.NH;
	float *z = (float *)hs4 + (long)w * Kp;
	float v[4], g[4];
	ld4(v, a.x + (long)t * a.xs + (long)j * HD, i, HD);
	ld4(g, a.g + (long)j * HD, i, HD);
	if (i < Kp) *(float4 *)(z + i) = make_float4(v[0] * v[0], v[1] * v[1], v[2] * v[2], v[3] * v[3]);
	tgq_wave_sync();
	const float inv = 1.0f / sqrtf(tg_ordered_sum_pp<8>(z, HD) / (float)HD + 1e-6f); // (every lane the same sum)
	tgq_wave_sync(); // the squares are read
	float nv[4];
	for (int u = 0; u < 4; u++) nv[u] = i + u < HD ? v[u] * inv * g[u] : 0.0f;
	st4(a.out + (long)L * HD, i, HD, nv);
	if (i < Kp) *(float4 *)(z + i) = make_float4(nv[0], nv[1], nv[2], nv[3]);
	wave_digits(nv, z, HD, Kp, a.q, L, &hist[w]);
}

// Many lines at once (a prompt's token rows, or its head lines). Line L = t
// npr + j reads h + t hs + j D (updated in place by modes 1 and 2, which need
// npr == 1), takes gain g + j gs, writes out + L D and the digits of row L.
// The values are the same as tgk_dec_norm's and tgk_dec_hnorm's: (h * inv) *
// g with inv = 1 / sqrtf(sum / D + 1e-6), sum the ordered sum of the squares.
struct NormLines {
	float *h;
	long hs;
	int mode;
	const float *add;
	long adds;
	const float *o;
	long ohead;
	int nh;
	const float *g;
	long gs;
	float *out;
	int D, npr;
	int lines;
	tgk_qdig q;
};

// sums (or the max) over the LPL lanes of a line, in the last of them
template <int LPL> __device__ inline int line_add(int v)
{
	v += tgq_dpp<0x111, 0xf>(v);
	v += tgq_dpp<0x112, 0xf>(v);
	v += tgq_dpp<0x114, 0xf>(v);
	v += tgq_dpp<0x118, 0xf>(v);
	if (LPL >= 32) v += tgq_dpp<0x142, 0xa>(v);
	if (LPL >= 64) v += tgq_dpp<0x143, 0xc>(v);
	return v;
}
template <int LPL> __device__ inline unsigned line_umax(unsigned v)
{
	v = max(v, (unsigned)tgq_dpp<0x111, 0xf>((int)v));
	v = max(v, (unsigned)tgq_dpp<0x112, 0xf>((int)v));
	v = max(v, (unsigned)tgq_dpp<0x114, 0xf>((int)v));
	v = max(v, (unsigned)tgq_dpp<0x118, 0xf>((int)v));
	if (LPL >= 32) v = max(v, (unsigned)tgq_dpp<0x142, 0xa>((int)v));
	if (LPL >= 64) v = max(v, (unsigned)tgq_dpp<0x143, 0xc>((int)v));
	return v;
}
// the same of lanes' sums of at most 64 |q|, which 64 lanes may take past 32 bits: by halves
template <int LPL, int QPL> __device__ inline long long line_add_q(int v)
{
	if (LPL * QPL <= 64) return line_add<LPL>(v);
	return (long long)line_add<LPL>(v >> 16) * 65536 + line_add<LPL>(v & 0xffff);
}

// A line is LPL lanes' with QPL quads a lane (quad s + LPL q is lane s's),
// Kp = 4 LPL QPL; a wave holds 64 / LPL of them NL times over, in registers
// from the load to the digits. Only the squares go through LDS, for the
// ordered sums: one lane a line, the block's lines side by side in one wave,
// another in each block (a block's first waves tend to share a SIMD, and the
// sums' adds bound the kernel together with the memory). The digits go by
// quads as in tgq_quad, a line's sums by data-parallel moves within its
// lanes. FULL: D == Kp, no quad ends past the line.
// 8192 rows of 1024 in 35 us (88 with one element a lane and access, every
// value through LDS twice), 4.5 TB/s of 159 MB; 196,608 head lines of 128 in
// 73 (118).
template <int LPL, int QPL, int NL, bool FULL>
__global__ __launch_bounds__(256) void norm_lines_k(NormLines a)
{
	constexpr int KP = 4 * LPL * QPL, G = 64 / LPL, LW = G * NL, R = 4 * LW, ZS = KP + 4;
	extern __shared__ float4 sh4[];
	float *z = (float *)sh4; // [R][ZS] squares; consecutive lines 4 banks apart
	float *linv = z + R * ZS;
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), sub = lane % LPL, grp = lane / LPL;
	const int D = FULL ? KP : a.D, L0 = blockIdx.x * R, l0 = wave * LW + grp; // slot n: line L0 + l0 + n G
	auto ld = [&](float *v, const float *p, int i) {
		if (FULL) {
			const f4u f = *(const f4u *)(p + i);
			v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
		} else
			ld4(v, p, i, D);
	};
	auto st = [&](float *p, int i, const float *v) {
		if (FULL) *(f4u *)(p + i) = f4u{ v[0], v[1], v[2], v[3] };
		else st4(p, i, D, v);
	};
	float v[NL][QPL][4], g[NL][QPL][4];
#pragma unroll
	for (int n = 0; n < NL; n++) {
		const int L = min(L0 + l0 + n * G, a.lines - 1), t = L / a.npr, j = L - t * a.npr; // (lines past the end read the last)
#pragma unroll
		for (int q = 0; q < QPL; q++) ld(v[n][q], a.h + (long)t * a.hs + (long)j * D, 4 * (sub + q * LPL));
#pragma unroll
		for (int q = 0; q < QPL; q++) ld(g[n][q], a.g + (long)j * a.gs, 4 * (sub + q * LPL));
		if (a.mode == 1) { // npr == 1: line L is token row L
			float b[QPL][4];
#pragma unroll
			for (int q = 0; q < QPL; q++) ld(b[q], a.add + (long)L * a.adds, 4 * (sub + q * LPL));
#pragma unroll
			for (int q = 0; q < QPL; q++)
				for (int u = 0; u < 4; u++) v[n][q][u] = v[n][q][u] + b[q][u];
		} else if (a.mode == 2) { // v + ((o_0 + o_1) + ... + o_{nh-1})
#pragma unroll
			for (int q = 0; q < QPL; q++) {
				const float *o = a.o + (long)L * D;
				float acc[4];
				ld(acc, o, 4 * (sub + q * LPL));
				for (int k = 1; k < a.nh; k++) {
					float b[4];
					ld(b, o + (long)k * a.ohead, 4 * (sub + q * LPL));
					for (int u = 0; u < 4; u++) acc[u] = acc[u] + b[u];
				}
				for (int u = 0; u < 4; u++) v[n][q][u] = v[n][q][u] + acc[u];
			}
		}
	}
#pragma unroll
	for (int n = 0; n < NL; n++) {
		const int l = l0 + n * G;
#pragma unroll
		for (int q = 0; q < QPL; q++) {
			const int i = 4 * (sub + q * LPL);
			const float *x = v[n][q];
			if (a.mode && L0 + l < a.lines) st(a.h + (long)(L0 + l) * a.hs, i, x);
			*(float4 *)(z + l * ZS + i) = make_float4(x[0] * x[0], x[1] * x[1], x[2] * x[2], x[3] * x[3]);
		}
	}
	__syncthreads();
	if (wave == (int)(blockIdx.x & 3) && lane < R) linv[lane] = 1.0f / sqrtf(tg_ordered_sum_pp<6>(z + lane * ZS, D) / (float)D + 1e-6f);
	__syncthreads();
#pragma unroll
	for (int n = 0; n < NL; n++) {
		const int L = L0 + l0 + n * G;
		const bool ok = L < a.lines;
		const float inv = linv[l0 + n * G];
		unsigned mb = 0;
#pragma unroll
		for (int q = 0; q < QPL; q++) {
			const int i = 4 * (sub + q * LPL);
			float *x = v[n][q];
			for (int u = 0; u < 4; u++) x[u] = FULL || i + u < D ? x[u] * inv * g[n][q][u] : 0.0f;
			if (ok) st(a.out + (long)L * D, i, x);
			tgq_scan4(x, mb);
		}
		mb = (unsigned)__shfl((int)line_umax<LPL>(mb), lane | (LPL - 1));
		float amax;
		int nan;
		tgq_scan_end(mb, amax, nan);
		const int special = tgq_special(nan, amax), E = tgq_exponent(amax, special);
		int8_t *blk = tgq_row_base(a.q.dig, L, KP);
		int qs = 0, aq = 0, nx = 0; // a lane's at most 64 inputs: below 2^29
#pragma unroll
		for (int q = 0; q < QPL; q++) {
			float *x = v[n][q];
			unsigned u[4], w0, w1, w2;
			for (int i = 0; i < 4; i++) {
				if (special) x[i] = 0.0f; // zero digits, nothing to add up
				const float sv = ldexpf(x[i], 23 - E), rq = rintf(sv);
				const int qi = (int)rq;
				qs += qi;
				aq += abs(qi);
				nx += rq != sv;
				u[i] = (unsigned)(qi + 0x808080);
			}
			tgq_pack4(u, w0, w1, w2);
			const int k0 = 4 * (sub + q * LPL);
			int8_t *p = blk + (k0 >> 5) * 3072 + ((k0 >> 4) & 1) * 512 + (k0 & 15);
			if (ok) *(unsigned *)p = w0, *(unsigned *)(p + 1024) = w1, *(unsigned *)(p + 2048) = w2;
		}
		TgqRowSums s{}; // (right in a line's last lane)
		s.qs = line_add_q<LPL, QPL>(qs);
		const long long ta = LPL * QPL <= 64 ? (long long)(unsigned)line_add<LPL>(aq) : line_add_q<LPL, QPL>(aq);
		s.tl = ta + ((long long)line_add<LPL>(nx) << TGQ_TALLY_SHIFT);
		const bool last = sub == LPL - 1;
		if (__any(last && !special && tgq_candidate(s.tl))) { // the coarse test of candidate lines before any resolve
			int n0 = 0, n1 = 0, nz = 0, a0 = 0, a1 = 0;
#pragma unroll
			for (int q = 0; q < QPL; q++)
				for (int i = 0; i < 4; i++) {
					const unsigned m = (unsigned)abs((int)rintf(ldexpf(v[n][q][i], 23 - E)));
					const bool g0 = m >= (1u << 22), g1 = !g0 && m >= (1u << 21);
					n0 += g0, n1 += g1, nz += v[n][q][i] != 0.0f;
					a0 += g0 ? (int)m : 0, a1 += g1 ? (int)m : 0;
				}
			const int c01 = line_add<LPL>(n0 | n1 << 16), cz = line_add<LPL>(nz); // at most 4096 each
			s.co.cnt = (unsigned long long)(c01 & 0xffff) + ((unsigned long long)(c01 >> 16) << 21) + ((unsigned long long)cz << 42);
			s.co.s0 = LPL * QPL <= 64 ? (unsigned long long)(unsigned)line_add<LPL>(a0) : (unsigned long long)line_add_q<LPL, QPL>(a0);
			s.co.s1 = LPL * QPL <= 64 ? (unsigned long long)(unsigned)line_add<LPL>(a1) : (unsigned long long)line_add_q<LPL, QPL>(a1);
		}
		if (last && ok) a.q.e[L] = E, a.q.special[L] = tgq_row_class(s, special), a.q.qsum[L] = s.qs;
	}
}

template <int LPL, int QPL, int NL> void norm_lines(hipStream_t s, const NormLines &n)
{
	constexpr int KP = 4 * LPL * QPL, R = 256 / LPL * NL;
	const unsigned grid = (unsigned)(((long)n.lines + R - 1) / R);
	const size_t lds = (size_t)R * (KP + 5) * sizeof(float);
	if (n.D == KP) norm_lines_k<LPL, QPL, NL, true><<<grid, 256, lds, s>>>(n);
	else norm_lines_k<LPL, QPL, NL, false><<<grid, 256, lds, s>>>(n);
}

// whether lines padded to Kp run there, and the launch (4096: a line's quads
// are a block's registers; dec_norm_k, a line a block, takes 320 us for 4096
// rows of 4096 and 1.27 ms for 16384)
bool norm_lines_for(hipStream_t s, int Kp, const NormLines &n)
{
	switch (Kp) {
	case 64: norm_lines<16, 1, 4>(s, n); return true;
	case 128: norm_lines<32, 1, 4>(s, n); return true;
	case 256: norm_lines<64, 1, 4>(s, n); return true;
	case 512: norm_lines<64, 2, 2>(s, n); return true;
	case 1024: norm_lines<64, 4, 1>(s, n); return true;
	case 2048: norm_lines<64, 8, 1>(s, n); return true;
	default: return false;
	}
}

// tgk_dec_silu: one block per row, four elements a thread and pass; silu as
// the element-wise kernels compute it. 48 rows of 3072 in 7.1 us (11.5 with
// 16 inputs' digits a lane: three of 16 waves had any).
__global__ __launch_bounds__(1024) void dec_silu_k(tgk_dec_silu_args a)
{
	extern __shared__ float4 zs4[]; // [Kp]
	float *zs = (float *)zs4;
	__shared__ BlkDigits red;
	__shared__ TgqHist hist;
	const int t = blockIdx.x, FF = a.FF;
	const float *g = a.gu + (long)t * a.gus, *u = g + FF;
	unsigned mb = 0;
	for (int i = 4 * threadIdx.x; i < a.Kp; i += 4 * blockDim.x) {
		float x[4], y[4], v[4];
		ld4(x, g, i, FF);
		ld4(y, u, i, FF);
		for (int e = 0; e < 4; e++) v[e] = i + e < FF ? x[e] / (1.0f + expf(-x[e])) * y[e] : 0.0f;
		st4(a.out + (long)t * FF, i, FF, v);
		tgq_scan4(v, mb);
		*(float4 *)(zs + i) = make_float4(v[0], v[1], v[2], v[3]);
	}
	blk_digits(zs, FF, a.Kp, mb, a.q, t, &red, &hist);
}

// out = silu(g) * u for a prompt's many rows [g (FF) | u (FF)] (gus apart),
// the operations dec_silu_k applies, streamed four values a thread (when FF,
// gus and the pointers allow 16-byte accesses); the GEMM's own digit kernel
// makes the digits after it. Block y takes rows y, y + gridDim.y, ...
__global__ __launch_bounds__(256) void silu_mul_k(const float *gu, long gus, float *out, int FF, int rows, int vec)
{
	const int i = (blockIdx.x * 256 + threadIdx.x) * 4;
	if (i >= FF) return;
	auto one = [](float x, float u) { return x / (1.0f + expf(-x)) * u; };
	for (int t = blockIdx.y; t < rows; t += gridDim.y) {
		const float *g = gu + (long)t * gus, *u = g + FF;
		float *o = out + (long)t * FF;
		if (vec) {
			const float4 gv = *(const float4 *)(g + i), uv = *(const float4 *)(u + i);
			*(float4 *)(o + i) = make_float4(one(gv.x, uv.x), one(gv.y, uv.y), one(gv.z, uv.z), one(gv.w, uv.w));
		} else
			for (int k = i; k < i + 4 && k < FF; k++) o[k] = one(g[k], u[k]);
	}
}

// A prompt chunk's causal softmax, line (sequence, head, t) of sc = q_t . k_u
// for u <= t (the products above the diagonal are not computed). The graph's
// operations on the valid part: x_u = s_u * scale + 0 (the mask's 0), the row
// op's max rule, expf(x_u - max), the sum in key order, e_u / sum. Above the
// diagonal the graph adds -1e9: for finite scores that entry never wins the
// max and its expf is exactly 0, which leaves the sum unchanged and gives
// p_u = 0, written here directly, up to the end of the line's tile of ztile
// positions. lpb lines per block (a power of two >= 4) staged in LDS, stride
// T0 + 4 floats (16-byte aligned); 256 / lpb lanes of one wave take a line, V
// consecutive elements each, so its max and its exponentials need no barrier,
// and only the ordered sums, one thread per line, side by side in one wave,
// do. A line's sum is one chain of adds: eight lines a block leave room for
// eight blocks a compute unit, whose chains overlap (16 x 16 lines of 512
// positions: 111 us; 193 when the block's lanes went through its lines one after
// another, 279 so at 32 lines a block, and 448 a head at a time).
template <int V>
__global__ __launch_bounds__(256) void causal_softmax_k(float *sc, int T0, long nlines, float scale, int ztile, int lpb, int stride)
{
	extern __shared__ float4 sh4[];
	float *z = (float *)sh4, *lv = z + lpb * stride; // lv: per line its sum
	const long L0 = (long)blockIdx.x * lpb;
	const int tid = threadIdx.x, tpl = 256 / lpb, l = tid / tpl, sub = tid - l * tpl;
	const long L = L0 + l;
	const int t = L < nlines ? (int)((unsigned)L % (unsigned)T0) : -1; // the line's position (none: no elements)
	float *y = z + l * stride, *line = sc + L * T0, m = -INFINITY, y0 = 0.0f;
	constexpr int U = 4;
	const int step = tpl * V;
	for (int u0 = sub * V; u0 <= t; u0 += U * step) { // U loads in flight
		float x[U][V];
#pragma unroll
		for (int q = 0; q < U; q++) {
			const int u = u0 + q * step <= t ? u0 + q * step : u0;
			if constexpr (V == 4) {
				const float4 s4 = *(const float4 *)(line + u);
				x[q][0] = s4.x, x[q][1] = s4.y, x[q][2] = s4.z, x[q][3] = s4.w;
			} else
				x[q][0] = line[u];
		}
#pragma unroll
		for (int q = 0; q < U; q++) {
			const int u = u0 + q * step;
			if (u > t) break;
#pragma unroll
			for (int i = 0; i < V; i++) {
				x[q][i] = x[q][i] * scale + 0.0f;
				y[u + i] = x[q][i];
				if (u + i == 0) y0 = x[q][i];
				else if (u + i <= t) m = fmaxf(m, x[q][i]);
			}
		}
	}
	for (int w = tpl / 2; w > 0; w >>= 1) m = fmaxf(m, __shfl_xor(m, w));
	y0 = __shfl(y0, (tid & 63) - sub); // the lane that holds the line's first element
	m = isnan(y0) ? y0 : fmaxf(y0, m);
	for (int u = sub * V; u <= t; u += step)
#pragma unroll
		for (int i = 0; i < V; i++) y[u + i] = expf(y[u + i] - m);
	__syncthreads();
	if (tid < lpb && L0 + tid < nlines) lv[tid] = tg_ordered_sum_pp<6>(z + tid * stride, (int)((unsigned)(L0 + tid) % (unsigned)T0) + 1);
	__syncthreads();
	const float sum = lv[l];
	const int zend = t < 0 ? 0 : min(T0, (t / ztile + 1) * ztile);
	for (int u = sub * V; u < zend; u += step) {
		float p[V];
#pragma unroll
		for (int i = 0; i < V; i++) p[i] = u + i <= t ? y[u + i] / sum : 0.0f;
		if constexpr (V == 4) *(float4 *)(line + u) = make_float4(p[0], p[1], p[2], p[3]);
		else line[u] = p[0];
	}
}

// Greedy choice per row: the index of the largest logit, the first one on
// ties, a nan counting as largest (numpy's argmax). (nan-ness, value, -index)
// is a total order, so any grouping of the comparisons finds the same index:
// argmax_part_k takes the best of each of a row's parts (blocks of `chunk`
// columns, loads in batches of 8 per thread), argmax_fin_k the best of the
// parts, written as an f32 token id (the model's input format) and as an int.
__device__ inline bool am_better(float a, int ia, float b, int ib) // is (a, ia) the better candidate?
{
	if (ib < 0) return ia >= 0;
	if (ia < 0) return false;
	const bool na = isnan(a), nb = isnan(b);
	if (na != nb) return na;
	if (!na && a != b) return a > b;
	return ia < ib;
}

__device__ inline void am_wave(float &v, int &i)
{
	for (int w = 32; w > 0; w >>= 1) {
		const float ov = __shfl_xor(v, w);
		const int oi = __shfl_xor(i, w);
		if (am_better(ov, oi, v, i)) v = ov, i = oi;
	}
}

__global__ __launch_bounds__(256) void argmax_part_k(const float *x, long xrs, int V, int chunk, int nparts, float *pv, int *pi)
{
	__shared__ float bv[4];
	__shared__ int bi[4];
	const int row = blockIdx.x / nparts, part = blockIdx.x - row * nparts;
	const float *r = x + (long)row * xrs;
	const int k0 = part * chunk, k1 = min(V, k0 + chunk);
	float v = 0.0f;
	int i = -1;
	for (int b = k0; b < k1; b += 8 * 256) {
		float u[8];
		for (int j = 0; j < 8; j++) {
			const int k = b + j * 256 + (int)threadIdx.x;
			u[j] = r[k < k1 ? k : k1 - 1];
		}
		for (int j = 0; j < 8; j++) {
			const int k = b + j * 256 + (int)threadIdx.x;
			if (k < k1 && am_better(u[j], k, v, i)) v = u[j], i = k;
		}
	}
	am_wave(v, i);
	if ((threadIdx.x & 63) == 0) bv[threadIdx.x >> 6] = v, bi[threadIdx.x >> 6] = i;
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < 4; w++)
			if (am_better(bv[w], bi[w], v, i)) v = bv[w], i = bi[w];
		pv[blockIdx.x] = v;
		pi[blockIdx.x] = i;
	}
}

__global__ __launch_bounds__(64) void argmax_fin_k(const float *pv, const int *pi, int nparts, float *idf, int *idi, long idi_stride)
{
	const int row = blockIdx.x, l = threadIdx.x;
	float v = l < nparts ? pv[(long)row * nparts + l] : 0.0f;
	int i = l < nparts ? pi[(long)row * nparts + l] : -1;
	am_wave(v, i);
	if (l == 0) {
		idf[row] = (float)i;
		if (idi) idi[(long)row * idi_stride] = i;
	}
}

constexpr int TPB = 256;
inline unsigned blocks(long n) { return (unsigned)((n + TPB - 1) / TPB); }

} // namespace

size_t tgk_dec_attn_lds(int GRP, int HD, int n)
{
	const long nst = (n + 3) & ~3;
	return (size_t)((long)attn_chunk(HD) * (HD + 4) + (long)GRP * HD + GRP * nst + GRP) * sizeof(float);
}

bool tgk_dec_attn_digits(int GRP, int HD)
{
	return HD <= 256 && (size_t)GRP * sizeof(TgqHist) <= (size_t)attn_chunk(HD) * (HD + 4) * sizeof(float);
}


void tgk_dec_rope(hipStream_t s, const tgk_dec_rope_args *a, int rows)
{
	const long total = (long)rows * (a->NQ + 2 * a->NKV) * a->HD;
	if (total <= 0) return;
	auto al = [](const void *p) { return ((size_t)p & 15) == 0; };
	if (a->HD % 4 == 0 && a->ctot % 4 == 0 && a->kv_seq % 4 == 0 && a->kv_layer % 4 == 0 && al(a->hq) && al(a->rt) && al(a->qkv) &&
	    al(a->cosT) && al(a->sinT) && al(a->qr) && al(a->K) && al(a->V)) {
		const int per = (a->NQ + 2 * a->NKV) * (a->HD / 4);
		const dim3 grid((unsigned)((per + 255) / 256), (unsigned)(rows < 65535 ? rows : 65535));
		rope_cache4_k<<<grid, 256, 0, s>>>(*a, rows);
	} else
		rope_cache_k<<<blocks(total), TPB, 0, s>>>(*a, total);
}

void tgk_dec_attn(hipStream_t s, const tgk_dec_attn_args *a, int seqs)
{
	const int GRP = a->NQ / a->NKV, ck = attn_chunk(a->HD);
	const size_t lds = tgk_dec_attn_lds(GRP, a->HD, a->p + 1);
	const unsigned grid = (unsigned)(seqs * a->NKV);
	if (seqs <= 0) return;
	switch (GRP) { // the decoder checks GRP, HD and the LDS size when it is created
	case 1: dec_attn_k<1><<<grid, ATT_TPB, lds, s>>>(*a, ck); break;
	case 2: dec_attn_k<2><<<grid, ATT_TPB, lds, s>>>(*a, ck); break;
	case 4: dec_attn_k<4><<<grid, ATT_TPB, lds, s>>>(*a, ck); break;
	case 8: dec_attn_k<8><<<grid, ATT_TPB, lds, s>>>(*a, ck); break;
	default: break;
	}
}

// many lines (a prompt): norm_lines_k; few (a step): a block per row or a wave per head line
constexpr long NL_MIN_LINES = 2048;
// threads of a block that takes a row of Kp values by fours
inline unsigned quad_tpb(int Kp) { return Kp >= 4096 ? 1024u : (unsigned)(Kp + 255) / 256 * 64; }

bool tgk_dec_norm(hipStream_t s, const tgk_dec_norm_args *a)
{
	if (a->rows <= 0) return true;
	if (a->rows >= NL_MIN_LINES && a->outs == a->D &&
	    norm_lines_for(s, a->Kp, NormLines{ a->h, a->hs, a->mode, a->add, a->adds, a->o, a->ohead, a->nh, a->g, 0, a->out, a->D, 1, a->rows, a->q }))
		return false; // candidates left for tgk_qgemm_split
	dec_norm_k<<<(unsigned)a->rows, quad_tpb(a->Kp), (size_t)a->Kp * 2 * sizeof(float), s>>>(*a);
	return true;
}

bool tgk_dec_hnorm(hipStream_t s, const tgk_dec_hnorm_args *a)
{
	const long lines = (long)a->rows * a->NH;
	if (lines <= 0) return true;
	if (lines >= NL_MIN_LINES &&
	    norm_lines_for(s, a->Kp, NormLines{ (float *)a->x, a->xs, 0, nullptr, 0, nullptr, 0, 0, a->g, a->HD, a->out, a->HD, a->NH, (int)lines, a->q }))
		return false; // candidates left for tgk_qgemm_split
	dec_hnorm_k<<<(unsigned)((lines + 3) / 4), TPB, (size_t)a->Kp * 4 * sizeof(float), s>>>(*a);
	return true;
}

void tgk_dec_silu_mul(hipStream_t s, const float *gu, long gus, float *out, int FF, int rows)
{
	if (rows <= 0 || FF <= 0) return;
	const int vec = FF % 4 == 0 && gus % 4 == 0 && ((size_t)gu & 15) == 0 && ((size_t)out & 15) == 0;
	const dim3 grid((unsigned)((FF + 1023) / 1024), (unsigned)(rows < 65535 ? rows : 65535));
	silu_mul_k<<<grid, 256, 0, s>>>(gu, gus, out, FF, rows, vec);
}

bool tgk_dec_silu(hipStream_t s, const tgk_dec_silu_args *a)
{
	if (a->rows > 0) dec_silu_k<<<(unsigned)a->rows, quad_tpb(a->Kp), (size_t)a->Kp * sizeof(float), s>>>(*a);
	return true;
}

void tgk_dec_causal_softmax(hipStream_t s, float *sc, int T0, long nlines, float scale, int ztile)
{
	if (nlines <= 0 || T0 <= 0) return;
	const int stride = (T0 + 3) / 4 * 4 + 4;
	int lpb = 8; // a power of two >= 4: lines per block, more of short lines so that every lane has elements
	while (lpb < 64 && lpb * T0 < 1024) lpb <<= 1;
	while (lpb > 4 && (long)lpb * stride * 4 + lpb * 4 > 65536) lpb >>= 1;
	const unsigned grid = (unsigned)((nlines + lpb - 1) / lpb);
	const size_t lds = (size_t)lpb * stride * 4 + lpb * 4;
	if (T0 % 4 == 0 && ((size_t)sc & 15) == 0) causal_softmax_k<4><<<grid, 256, lds, s>>>(sc, T0, nlines, scale, ztile ? ztile : T0, lpb, stride);
	else causal_softmax_k<1><<<grid, 256, lds, s>>>(sc, T0, nlines, scale, ztile ? ztile : T0, lpb, stride);
}

void tgk_dec_argmax(hipStream_t s, const float *x, long xrs, int V, int rows, float *idf, int *idi, long idi_stride, float *pv, int *pi)
{
	if (rows <= 0 || V <= 0) return;
	const int np0 = (V + 2047) / 2048, nparts = np0 < TGK_AM_PARTS ? np0 : TGK_AM_PARTS, chunk = (V + nparts - 1) / nparts;
	argmax_part_k<<<(unsigned)(rows * nparts), TPB, 0, s>>>(x, xrs, V, chunk, nparts, pv, pi);
	argmax_fin_k<<<(unsigned)rows, 64, 0, s>>>(pv, pi, nparts, idf, idi, idi_stride);
}
