// Quantisation kernels for reduced-precision storage of A (see quant.hpp for the formats).
#include "quant.hpp"

#include <algorithm>

#include "../../include/ttvx.h"
#include "runtime.hpp"

namespace ttvx
{

// 8 values per thread: two 16-byte loads, one 16-byte store (element alignment suffices on gfx950).  Bound by HBM;
// the scalar form had 4-byte loads and 2-byte stores: 1 GiB of FP32 on MI355X, 402 us -> 260 us (6.2 TB/s).
__global__ __launch_bounds__(kBlock) void k_quant_bf16(const float* __restrict__ src, uint16_t* __restrict__ dst, int64_t n)
{
	int64_t const i = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * 8;
	if(i + 8 <= n) {
		u32x4_b const lo = __builtin_nontemporal_load(TTVX_GLOBAL(u32x4_b, src + i));
		u32x4_b const hi = __builtin_nontemporal_load(TTVX_GLOBAL(u32x4_b, src + i + 4));
		uint32_t const w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
		uint32_t h[8];
#pragma unroll
		for(int e = 0; e < 8; ++e) h[e] = f32_to_bf16_rne(__uint_as_float(w[e]));
		u32x4_b q;
		q.x = h[0] | (h[1] << 16);
		q.y = h[2] | (h[3] << 16);
		q.z = h[4] | (h[5] << 16);
		q.w = h[6] | (h[7] << 16);
		__builtin_nontemporal_store(q, TTVX_GLOBAL_W(u32x4_b, dst + i));
	} else {
		for(int64_t j = i; j < n; ++j) dst[j] = f32_to_bf16_rne(src[j]);
	}
}

// ---- FP8 -------------------------------------------------------------------------------------
// Group g holds the fibers j in [g*fps, (g+1)*fps) (fiber j = o*I + i), all K elements of each.  Its scale needs
// every element before the first code can be written, so a kernel either keeps the group's elements in registers
// between the two (k_quant_rows, k_quant_tile: A is read once) or, where a group or a piece of rows worth a
// cache line does not fit a block's registers, the maxima are collected first and A is read again
// (k_quant_long, k_quant_cols).  MI355X, 128^4 FP32 (1 GiB read, 256 MiB written): 1188 us -> 240 us (5.6 TB/s),
// rows of 128 220 us; the general kernel below divides 64-bit indices twice per element and reads A twice.

// the four codes of x * inv: the gfx950 converter rounds to nearest even and, on clamped operands, gives what
// f32_to_e4m3_rne_sat gives for every float but a positive NaN (checked over all 2^32 patterns)
__device__ __forceinline__ uint32_t encode4(const float (&x)[4])
{
	if(__builtin_isunordered(x[0], x[1]) || __builtin_isunordered(x[2], x[3])) {
		uint32_t w = 0;
#pragma unroll
		for(int e = 0; e < 4; ++e) w |= static_cast<uint32_t>(f32_to_e4m3_rne_sat(x[e])) << (8 * e);
		return w;
	}
	float y[4];
#pragma unroll
	for(int e = 0; e < 4; ++e) y[e] = __builtin_amdgcn_fmed3f(x[e], -448.0f, 448.0f);
	int w = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false);
	return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], w, true));
}

__device__ __forceinline__ uint8_t encode1(float x)
{
	if(x != x) return f32_to_e4m3_rne_sat(x);
	float const y = __builtin_amdgcn_fmed3f(x, -448.0f, 448.0f);
	return static_cast<uint8_t>(__builtin_amdgcn_cvt_pk_fp8_f32(y, y, 0, false) & 0xff);
}

__device__ __forceinline__ float scale_of(float amax) { return amax > 0.f ? amax / 448.0f : 1.0f; }
__device__ __forceinline__ float inv_of(float amax) { return amax > 0.f ? 448.0f / amax : 1.0f; }

// VEC consecutive values, absolute maximum, codes
template<int VEC>
struct QVec {
	float x[VEC];
	__device__ __forceinline__ void load(const float* p)
	{
		if constexpr(VEC == 4) {
			u32x4_b const v = __builtin_nontemporal_load(TTVX_GLOBAL(u32x4_b, p));
			x[0] = __uint_as_float(v.x); x[1] = __uint_as_float(v.y);
			x[2] = __uint_as_float(v.z); x[3] = __uint_as_float(v.w);
		} else {
			x[0] = __builtin_nontemporal_load(TTVX_GLOBAL(float, p));
		}
	}
	__device__ __forceinline__ void store(uint8_t* q, const float (&inv)[VEC]) const
	{
		float y[VEC];
#pragma unroll
		for(int e = 0; e < VEC; ++e) y[e] = x[e] * inv[e];
		if constexpr(VEC == 4) __builtin_nontemporal_store(encode4(y), TTVX_GLOBAL_W(u32_b, q));
		else                   *TTVX_GLOBAL_W(uint8_t, q) = encode1(y[0]);
	}
};

// maximum over the TG threads of a group of threads (64, or the whole block through LDS)
template<int TG>
__device__ __forceinline__ float group_max(float m, float* wmax)
{
#pragma unroll
	for(int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
	if constexpr(TG > 64) {
		if((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
		__syncthreads();
		m = wmax[0];
#pragma unroll
		for(int w = 1; w < TG / 64; ++w) m = fmaxf(m, wmax[w]);
	}
	return m;
}

// Rows (I == 1, dense): a group is E = fps*K contiguous values, held by TG threads (R vectors of 4 each,
// E <= 4*TG*R) between its maximum and its codes.
template<int TG, int R>
__global__ __launch_bounds__(TG < kBlock ? kBlock : TG) void k_quant_rows(const float* __restrict__ A, uint8_t* __restrict__ Q,
                                                                          float* __restrict__ scales, QuantArgs P)
{
	constexpr int PER = TG < kBlock ? kBlock / TG : 1;       // groups per block
	__shared__ float wmax[TG / 64];
	int const t = static_cast<int>(threadIdx.x) & (TG - 1);
	int64_t const g = static_cast<int64_t>(blockIdx.x) * PER + (TG < kBlock ? threadIdx.x / TG : 0);
	if(g >= P.groups) return;                                // whole waves (TG = 64) or never (one group a block)
	int64_t const e0 = g * P.fps * P.K;
	int64_t const left = P.O * P.K - e0;
	int const E = static_cast<int>(left < P.fps * P.K ? left : P.fps * P.K);
	QVec<4> v[R];
	float m = 0.f;
#pragma unroll
	for(int r = 0; r < R; ++r) {
		int const e = (r * TG + t) * 4;
		if(e + 4 <= E) v[r].load(A + e0 + e);
		else
#pragma unroll
			for(int c = 0; c < 4; ++c) v[r].x[c] = e + c < E ? A[e0 + e + c] : 0.f;
	}
#pragma unroll
	for(int r = 0; r < R; ++r)
#pragma unroll
		for(int c = 0; c < 4; ++c) m = fmaxf(m, fabsf(v[r].x[c]));
	m = group_max<TG>(m, wmax);
	if(t == 0) scales[g] = scale_of(m);
	float const i1 = inv_of(m);
	float const inv[4] = {i1, i1, i1, i1};
#pragma unroll
	for(int r = 0; r < R; ++r) {
		int const e = (r * TG + t) * 4;
		if(e + 4 <= E) v[r].store(Q + e0 + e, inv);
		else
#pragma unroll
			for(int c = 0; c < 4; ++c)
				if(e + c < E) Q[e0 + e + c] = encode1(v[r].x[c] * i1);
	}
}

// Columns: block b holds the fibers [b*nf, (b+1)*nf), whole groups, in registers.  LV lanes along the fibers
// (VEC = 4 columns each when 4 divides I, so that a vector stays in its slab), KS = TB / LV along k; when a
// group has more fibers than a block has lanes (short contractions) a thread takes F fiber vectors in turn.
// F * steps <= R loads, all issued before the first use.  Maxima meet in LDS.
template<int VEC, int TB, int R>
__global__ __launch_bounds__(TB) void k_quant_tile(const float* __restrict__ A, uint8_t* __restrict__ Q,
                                                   float* __restrict__ scales, QuantArgs P)
{
	extern __shared__ uint32_t gmax[];                       // bits of the groups' maxima (ordered like the floats)
	int const t = static_cast<int>(threadIdx.x);
	int64_t const fibers = P.O * P.I;
	int64_t const j0 = static_cast<int64_t>(blockIdx.x) * P.nf;
	int64_t const g0 = static_cast<int64_t>(blockIdx.x) * P.tile_groups;
	for(int g = t; g < P.tile_groups; g += TB) gmax[g] = 0u;
	__syncthreads();
	int const l = t % P.LV, ks = t / P.LV;
	int64_t const kstep = static_cast<int64_t>(P.KS) * P.sAk;
	// fiber vector of set s: first fiber, and its offset in A (-1: nothing there)
	auto place = [&](int s, int& f) -> int64_t {
		f = (s * P.LV + l) * VEC;
		int64_t const j = j0 + f;
		if(ks >= P.KS || f >= P.nf || j >= fibers) return -1;
		int64_t const o = j / P.I;
		return o * P.sAo + (j - o * P.I) + ks * P.sAk;
	};
	QVec<VEC> v[R];
	int s = 0, kk = 0, f = 0;
	int64_t off = place(0, f);
#pragma unroll
	for(int r = 0; r < R; ++r) {
		if(s < P.F) {
			bool const ok = off >= 0 && ks + kk * P.KS < P.K;
			if(ok) v[r].load(A + off + kk * kstep);
			else
#pragma unroll
				for(int e = 0; e < VEC; ++e) v[r].x[e] = 0.f;
			if(++kk == P.steps) {
				kk = 0;
				if(++s < P.F) off = place(s, f);
			}
		}
	}
	float m[VEC];
#pragma unroll
	for(int e = 0; e < VEC; ++e) m[e] = 0.f;
	s = 0;
	kk = 0;
#pragma unroll
	for(int r = 0; r < R; ++r) {
		if(s < P.F) {
#pragma unroll
			for(int e = 0; e < VEC; ++e) m[e] = fmaxf(m[e], fabsf(v[r].x[e]));
			if(++kk == P.steps) {
				int const fs = (s * P.LV + l) * VEC;
				if(ks < P.KS && fs < P.nf) {
					uint32_t const ga = static_cast<uint32_t>(fs) / static_cast<uint32_t>(P.fps);
					uint32_t const gb = static_cast<uint32_t>(fs + VEC - 1) / static_cast<uint32_t>(P.fps);
					if(ga == gb) {
						float mm = m[0];
#pragma unroll
						for(int e = 1; e < VEC; ++e) mm = fmaxf(mm, m[e]);
						atomicMax(&gmax[ga], __float_as_uint(mm));
					} else {
#pragma unroll
						for(int e = 0; e < VEC; ++e)
							atomicMax(&gmax[static_cast<uint32_t>(fs + e) / static_cast<uint32_t>(P.fps)], __float_as_uint(m[e]));
					}
				}
#pragma unroll
				for(int e = 0; e < VEC; ++e) m[e] = 0.f;
				kk = 0;
				++s;
			}
		}
	}
	__syncthreads();
	for(int g = t; g < P.tile_groups; g += TB)
		if(g0 + g < P.groups) scales[g0 + g] = scale_of(__uint_as_float(gmax[g]));
	s = 0;
	kk = 0;
	float inv[VEC];
	off = place(0, f);
	if constexpr(VEC == 4) {
#pragma unroll
		for(int r = 0; r < R; ++r) {
			if(s < P.F) {
				if(kk == 0 && off >= 0)
#pragma unroll
					for(int e = 0; e < VEC; ++e)
						inv[e] = inv_of(__uint_as_float(gmax[static_cast<uint32_t>(f + e) / static_cast<uint32_t>(P.fps)]));
				if(off >= 0 && ks + kk * P.KS < P.K) v[r].store(Q + off + kk * kstep, inv);
				if(++kk == P.steps) {
					kk = 0;
					if(++s < P.F) off = place(s, f);
				}
			}
		}
	} else {
		// four steps encode together
#pragma unroll
		for(int r0 = 0; r0 < R; r0 += 4) {
			float y[4] = {0.f, 0.f, 0.f, 0.f};
			int64_t at[4] = {-1, -1, -1, -1};
#pragma unroll
			for(int c = 0; c < 4; ++c) {
				if(s < P.F) {
					if(kk == 0 && off >= 0)
						inv[0] = inv_of(__uint_as_float(gmax[static_cast<uint32_t>(f) / static_cast<uint32_t>(P.fps)]));
					if(off >= 0 && ks + kk * P.KS < P.K) {
						at[c] = off + kk * kstep;
						y[c] = v[r0 + c].x[0] * inv[0];
					}
					if(++kk == P.steps) {
						kk = 0;
						if(++s < P.F) off = place(s, f);
					}
				}
			}
			uint32_t const w = encode4(y);
#pragma unroll
			for(int c = 0; c < 4; ++c)
				if(at[c] >= 0) Q[at[c]] = static_cast<uint8_t>(w >> (8 * c));
		}
	}
}

// Dense slabs too narrow for lanes along i: the tile's fibers [j0, j0 + nf) lie in the contiguous values of the
// slabs that they touch, and a thread takes R vectors of 4 consecutive values, whatever slabs and columns these
// belong to.  Value e (counted from the first slab) is of slab e / (K*I) and column e % I.  Values of fibers that
// belong to the neighbouring blocks (partial first and last slab) are read and left alone.
template<int TB, int R>
__global__ __launch_bounds__(TB) void k_quant_slabs(const float* __restrict__ A, uint8_t* __restrict__ Q,
                                                    float* __restrict__ scales, QuantArgs P)
{
	extern __shared__ uint32_t gmax[];
	int const t = static_cast<int>(threadIdx.x);
	int64_t const fibers = P.O * P.I;
	int64_t const j0 = static_cast<int64_t>(blockIdx.x) * P.nf;
	int const nf = static_cast<int>(j0 + P.nf < fibers ? P.nf : fibers - j0);
	int64_t const g0 = static_cast<int64_t>(blockIdx.x) * P.tile_groups;
	int64_t const o0 = j0 / P.I;
	int const skip = static_cast<int>(j0 - o0 * P.I);         // fibers of the first slab before j0
	int const I = static_cast<int>(P.I);
	int64_t const a0 = o0 * P.K * P.I;
	int const E = static_cast<int>(div_by(static_cast<uint32_t>(skip + nf + I - 1), P.by_I)) * I * static_cast<int>(P.K);
	for(int g = t; g < P.tile_groups; g += TB) gmax[g] = 0u;
	__syncthreads();
	QVec<4> v[R];
#pragma unroll
	for(int r = 0; r < R; ++r) {
		int const e = (r * TB + t) * 4;
		if(e + 4 <= E) v[r].load(A + a0 + e);
		else
#pragma unroll
			for(int c = 0; c < 4; ++c) v[r].x[c] = e + c < E ? A[a0 + e + c] : 0.f;
	}
	// group of value e inside the tile, -1 outside
	auto group = [&](int e) -> int {
		if(e >= E) return -1;
		int const o = static_cast<int>(div_by(static_cast<uint32_t>(e), P.by_slab));
		int const i = e - static_cast<int>(div_by(static_cast<uint32_t>(e), P.by_I)) * I;
		int const f = o * I + i - skip;
		return f >= 0 && f < nf ? static_cast<int>(div_by(static_cast<uint32_t>(f), P.by_fps)) : -1;
	};
	// the one group that every fiber of the vector's slabs is in, -1 when there are several or some lie outside
	auto common = [&](int e) -> int {
		if(e + 4 > E) return -1;
		int const fa = static_cast<int>(div_by(static_cast<uint32_t>(e), P.by_slab)) * I - skip;
		int const fb = (static_cast<int>(div_by(static_cast<uint32_t>(e + 3), P.by_slab)) + 1) * I - 1 - skip;
		if(fa < 0 || fb >= nf) return -1;
		int const g = static_cast<int>(div_by(static_cast<uint32_t>(fa), P.by_fps));
		return g == static_cast<int>(div_by(static_cast<uint32_t>(fb), P.by_fps)) ? g : -1;
	};
	int run = -1;                                             // group of the running maximum
	float m = 0.f;
#pragma unroll
	for(int r = 0; r < R; ++r) {
		int const e = (r * TB + t) * 4;
		int const g = common(e);
		if(g >= 0) {
			if(g != run) {
				if(run >= 0) atomicMax(&gmax[run], __float_as_uint(m));
				run = g;
				m = 0.f;
			}
#pragma unroll
			for(int c = 0; c < 4; ++c) m = fmaxf(m, fabsf(v[r].x[c]));
		} else {
#pragma unroll
			for(int c = 0; c < 4; ++c) {
				int const ge = group(e + c);
				if(ge >= 0) atomicMax(&gmax[ge], __float_as_uint(fmaxf(0.f, fabsf(v[r].x[c]))));
			}
		}
	}
	if(run >= 0) atomicMax(&gmax[run], __float_as_uint(m));
	__syncthreads();
	for(int g = t; g < P.tile_groups; g += TB)
		if(g0 + g < P.groups) scales[g0 + g] = scale_of(__uint_as_float(gmax[g]));
#pragma unroll
	for(int r = 0; r < R; ++r) {
		int const e = (r * TB + t) * 4;
		int const g = common(e);
		if(g >= 0) {
			float const i1 = inv_of(__uint_as_float(gmax[g]));
			float const inv[4] = {i1, i1, i1, i1};
			v[r].store(Q + a0 + e, inv);
		} else {
#pragma unroll
			for(int c = 0; c < 4; ++c) {
				int const ge = group(e + c);
				if(ge >= 0) Q[a0 + e + c] = encode1(v[r].x[c] * inv_of(__uint_as_float(gmax[ge])));
			}
		}
	}
}

// The two passes of groups that no block holds: PASS 0 leaves each group's maximum in `scales` (zeroed before),
// PASS 1 writes the codes from it; k_quant_scales then turns the maxima into scales.
// Columns: LV lanes along fiber vectors, KS along k, block (x, y): fiber tile x, k chunk y.
template<int VEC, int PASS>
__global__ __launch_bounds__(kBlock) void k_quant_cols(const float* __restrict__ A, uint8_t* __restrict__ Q,
                                                       float* __restrict__ scales, QuantArgs P)
{
	constexpr int KL = 8;                                    // loads in flight per lane
	int const t = static_cast<int>(threadIdx.x);
	int const l = t % P.LV, ks = t / P.LV;
	int64_t const j = static_cast<int64_t>(blockIdx.x) * P.nf + l * VEC;
	if(ks >= P.KS || j >= P.O * P.I) return;
	int64_t const o = j / P.I;
	int64_t const kb = static_cast<int64_t>(blockIdx.y) * P.kchunk;
	int64_t const ke = kb + P.kchunk < P.K ? kb + P.kchunk : P.K;
	int64_t const base = o * P.sAo + (j - o * P.I);
	float w[VEC];                                            // PASS 0: maxima, PASS 1: 448 / maximum
	int64_t g[VEC];
#pragma unroll
	for(int e = 0; e < VEC; ++e) {
		g[e] = (j + e) / P.fps;
		w[e] = PASS == 0 ? 0.f : inv_of(scales[g[e]]);
	}
	for(int64_t k = kb + ks; k < ke; k += KL * P.KS) {
		QVec<VEC> v[KL];
#pragma unroll
		for(int r = 0; r < KL; ++r) {
			// steps past the end re-read the round's first row
			int64_t const kr = k + r * P.KS < ke ? k + r * P.KS : k;
			v[r].load(A + base + kr * P.sAk);
		}
#pragma unroll
		for(int r = 0; r < KL; ++r) {
			if constexpr(PASS == 0) {
#pragma unroll
				for(int e = 0; e < VEC; ++e) w[e] = fmaxf(w[e], fabsf(v[r].x[e]));
			} else if(k + r * P.KS < ke) {
				v[r].store(Q + base + (k + r * P.KS) * P.sAk, w);
			}
		}
	}
	if constexpr(PASS == 0)
#pragma unroll
		for(int e = 0; e < VEC; ++e) atomicMax(reinterpret_cast<uint32_t*>(scales + g[e]), __float_as_uint(w[e]));
}

// Dense rows whose groups (E = fps*K contiguous values) exceed a block: block (x, y) takes piece x of group y's values
template<int PASS>
__global__ __launch_bounds__(kBlock) void k_quant_long(const float* __restrict__ A, uint8_t* __restrict__ Q,
                                                       float* __restrict__ scales, QuantArgs P)
{
	__shared__ float wmax[kBlock / 64];
	int64_t const E = P.fps * P.K;
	for(int64_t g = blockIdx.y; g < P.groups; g += gridDim.y) {
		int64_t const e0 = g * E;
		int64_t const end = e0 + E < P.O * P.K ? e0 + E : P.O * P.K;
		int64_t const pb = e0 + static_cast<int64_t>(blockIdx.x) * P.kchunk;
		int64_t const pe = pb + P.kchunk < end ? pb + P.kchunk : end;
		float const i1 = PASS == 0 ? 0.f : inv_of(scales[g]);
		float const inv[4] = {i1, i1, i1, i1};
		float m = 0.f;
		constexpr int KL = 4;
		for(int64_t e = pb + static_cast<int64_t>(threadIdx.x) * 4; e < pe; e += KL * kBlock * 4) {
			QVec<4> v[KL];
#pragma unroll
			for(int r = 0; r < KL; ++r) {
				int64_t const er = e + static_cast<int64_t>(r) * kBlock * 4;
				if(er + 4 <= pe) v[r].load(A + er);
				else
#pragma unroll
					for(int c = 0; c < 4; ++c) v[r].x[c] = er + c < pe ? A[er + c] : 0.f;
			}
#pragma unroll
			for(int r = 0; r < KL; ++r) {
				int64_t const er = e + static_cast<int64_t>(r) * kBlock * 4;
				if constexpr(PASS == 0) {
#pragma unroll
					for(int c = 0; c < 4; ++c) m = fmaxf(m, fabsf(v[r].x[c]));
				} else {
					if(er + 4 <= pe) v[r].store(Q + er, inv);
					else
#pragma unroll
						for(int c = 0; c < 4; ++c)
							if(er + c < pe) Q[er + c] = encode1(v[r].x[c] * i1);
				}
			}
		}
		if constexpr(PASS == 0) {
			m = group_max<kBlock>(m, wmax);
			if(threadIdx.x == 0 && pb < pe) atomicMax(reinterpret_cast<uint32_t*>(scales + g), __float_as_uint(m));
			__syncthreads();
		}
	}
}

// zero: scales = 0; otherwise scales = the scales of the maxima that they hold
__global__ __launch_bounds__(kBlock) void k_quant_scales(float* __restrict__ scales, int64_t groups, int zero)
{
	int64_t const g = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
	if(g < groups) scales[g] = zero ? 0.f : scale_of(scales[g]);
}

// Strides that none of the above takes (no unit stride along i, rows with gaps): one block per scale group, absmax
// over the group's fibers, then encode.
// Element e of group g: fiber j = g*fps + e % nf, k = e / nf (consecutive threads walk
// consecutive fibers, i.e. consecutive i for a fixed k, so loads are coalesced when sAi == 1).
__global__ __launch_bounds__(kBlock) void k_quant_fp8(const float* __restrict__ A, uint8_t* __restrict__ Q,
                                                      float* __restrict__ scales, QuantArgs P)
{
	__shared__ float wmax[kBlock / 64];
	int64_t const fibers = P.O * P.I;
	for(int64_t g = blockIdx.x; g < P.groups; g += gridDim.x) {
		int64_t const j0 = g * P.fps;
		int64_t const nf = std::min(P.fps, fibers - j0);
		int64_t const total = nf * P.K;
		float m = 0.f;
		for(int64_t e = threadIdx.x; e < total; e += kBlock) {
			int64_t const k = e / nf, j = j0 + (e - k * nf);
			int64_t const o = j / P.I, i = j - o * P.I;
			m = fmaxf(m, fabsf(A[o * P.sAo + k * P.sAk + i * P.sAi]));
		}
		for(int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
		if((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
		__syncthreads();
		float amax = wmax[0];
		for(int w = 1; w < kBlock / 64; ++w) amax = fmaxf(amax, wmax[w]);
		__syncthreads();
		float const scale = amax > 0.f ? amax / 448.0f : 1.0f;
		float const inv   = amax > 0.f ? 448.0f / amax : 1.0f;
		if(threadIdx.x == 0) scales[g] = scale;
		for(int64_t e = threadIdx.x; e < total; e += kBlock) {
			int64_t const k = e / nf, j = j0 + (e - k * nf);
			int64_t const o = j / P.I, i = j - o * P.I;
			int64_t const off = o * P.sAo + k * P.sAk + i * P.sAi;
			Q[off] = f32_to_e4m3_rne_sat(A[off] * inv);
		}
	}
}

int quantize_bf16(std::size_t count, const float* src, uint16_t* dst, hipStream_t stream)
{
	if(count == 0) return TTVX_OK;
	int64_t const per = kMaxLeanBlocks * kBlock * 8;          // values of one launch
	for(int64_t at = 0, n = static_cast<int64_t>(count); at < n; at += per) {
		int64_t const len = std::min(per, n - at);
		unsigned const grid = static_cast<unsigned>((len + kBlock * 8 - 1) / (kBlock * 8));
		hipLaunchKernelGGL(k_quant_bf16, dim3(grid), dim3(kBlock), 0, stream, src + at, dst + at, len);
	}
	hipError_t e = hipGetLastError();
	return e == hipSuccess ? TTVX_OK : hip_fail(e, "bf16 quantisation launch");
}

namespace
{
int64_t up(int64_t a, int64_t b) { return (a + b - 1) / b; }

// k_quant_tile's tile for blocks of tb threads with r loads each: the most whole groups that a block holds; false
// when not even one fits
bool tile_shape(QuantArgs& P, int vec, int tb, int r)
{
	int64_t const fibers = P.O * P.I;
	int64_t const unit = vec == 4 && P.fps % 4 != 0 ? (P.fps % 2 != 0 ? 4 : 2) : 1;   // groups that end on a vector
	int64_t gs = std::min<int64_t>(static_cast<int64_t>(tb) * vec * r / (P.K * P.fps), up(up(fibers, P.fps), unit) * unit);
	for(gs = gs / unit * unit; gs >= unit; gs -= unit) {
		int64_t const lanes = gs * P.fps / vec;
		P.LV = static_cast<int>(std::min<int64_t>(lanes, tb));
		P.F  = static_cast<int>(up(lanes, P.LV));
		P.KS = static_cast<int>(P.F > 1 ? 1 : std::min<int64_t>(tb / P.LV, P.K));
		P.steps = static_cast<int>(up(P.K, P.KS));
		if(static_cast<int64_t>(P.F) * P.steps <= r && gs <= 8192) {
			P.nf = gs * P.fps;
			P.tile_groups = static_cast<int>(gs);
			return up(fibers, P.nf) <= kMaxLeanBlocks / 4;
		}
	}
	return false;
}
} // namespace

int quantize_fp8(const Fold& f, const float* a, uint8_t* aq, float* scales, int64_t fps, hipStream_t stream)
{
	QuantArgs P{};
	P.O = f.O; P.K = f.K; P.I = f.I;
	P.sAo = f.sAo; P.sAk = f.sAk; P.sAi = f.sAi;
	// more fibers per scale than there are: one group
	P.fps = std::min<int64_t>(fps, f.O * f.I);
	P.groups = up(f.O * f.I, P.fps);
	auto const launched = []() {
		hipError_t e = hipGetLastError();
		return e == hipSuccess ? TTVX_OK : hip_fail(e, "fp8 quantisation launch");
	};
	auto const scales_pass = [&](int zero) {
		hipLaunchKernelGGL(k_quant_scales, dim3(static_cast<unsigned>(up(P.groups, kBlock))), dim3(kBlock), 0, stream, scales,
		                   P.groups, zero);
	};
	bool const rows = f.I == 1 && (f.sAk == 1 || f.K == 1) && (f.sAo == f.K || f.O == 1);
	if(rows && P.groups <= kMaxLeanBlocks) {
		// a wave, a block of 256 or one of 1024 threads per group, by its size; 8 vectors of 4 per thread at most
		int64_t const E = P.fps * P.K;
		unsigned const g1 = static_cast<unsigned>(P.groups), g4 = static_cast<unsigned>(up(P.groups, kBlock / 64));
		if(E <= 4 * 64 * 2)         hipLaunchKernelGGL((k_quant_rows<64, 2>), dim3(g4), dim3(kBlock), 0, stream, a, aq, scales, P);
		else if(E <= 4 * 256 * 4)   hipLaunchKernelGGL((k_quant_rows<256, 4>), dim3(g1), dim3(kBlock), 0, stream, a, aq, scales, P);
		else if(E <= 4 * 256 * 8)   hipLaunchKernelGGL((k_quant_rows<256, 8>), dim3(g1), dim3(kBlock), 0, stream, a, aq, scales, P);
		else if(E <= 4 * 1024 * 8)  hipLaunchKernelGGL((k_quant_rows<1024, 8>), dim3(g1), dim3(1024), 0, stream, a, aq, scales, P);
		else {
			scales_pass(1);
			P.kchunk = 4 * kBlock * 16;                      // 64 KiB pieces: a few rounds of loads per block
			int64_t pieces = up(E, P.kchunk);
			if(pieces > 65536) {
				pieces = 65536;
				P.kchunk = up(up(E, pieces), 4) * 4;
			}
			dim3 const grid(static_cast<unsigned>(up(E, P.kchunk)), static_cast<unsigned>(std::min<int64_t>(P.groups, 32768)));
			hipLaunchKernelGGL((k_quant_long<0>), grid, dim3(kBlock), 0, stream, a, aq, scales, P);
			hipLaunchKernelGGL((k_quant_long<1>), grid, dim3(kBlock), 0, stream, a, aq, scales, P);
			scales_pass(0);
		}
		return launched();
	}
	if(f.I > 1 && f.sAi == 1) {
		// narrow slabs (rows of less than a cache line): whole groups as contiguous values, when the two slabs that a
		// tile's ends may cut do not cost much
		int64_t const slab = f.K * f.I, E = P.fps * f.K;
		if(f.I < 32 && f.sAk == f.I && (f.sAo == slab || f.O == 1) && slab <= 4096) {
			int64_t const fibers = f.O * f.I;
			auto const tile = [&](int64_t capacity) -> int64_t {
				int64_t const gs = std::min<int64_t>({(capacity - 2 * slab) / E, P.groups, 4096});
				return gs >= 1 ? gs : 0;
			};
			int64_t const g256 = tile(4 * 256 * 8), g1024 = tile(4 * 1024 * 8);
			int64_t const gs = 2 * g256 * E >= 4 * 256 * 8 ? g256 : g1024;
			if(gs > 0 && up(P.groups, gs) <= kMaxLeanBlocks / 4) {
				P.nf = gs * P.fps;
				P.tile_groups = static_cast<int>(gs);
				P.by_slab = fast_div(slab);
				P.by_I = fast_div(f.I);
				P.by_fps = fast_div(P.fps);
				unsigned const grid = static_cast<unsigned>(up(fibers, P.nf));
				if(gs == g256)
					hipLaunchKernelGGL((k_quant_slabs<256, 8>), dim3(grid), dim3(256), gs * sizeof(uint32_t), stream, a, aq, scales, P);
				else
					hipLaunchKernelGGL((k_quant_slabs<1024, 8>), dim3(grid), dim3(1024), gs * sizeof(uint32_t), stream, a, aq, scales, P);
				return launched();
			}
		}
		int const vec = f.I % 4 == 0 ? 4 : 1;
		// blocks of 256 threads where their tiles still write whole 128-byte lines of codes, else of 1024 (128^4:
		// tiles of 64 fibers 283 us, of 256 fibers 240 us).  A tile is worth its single read of A while its rows come near a cache line (24 fibers)
		auto const wide = [&](bool ok) { return ok && P.nf >= std::min<int64_t>(24, f.O * f.I); };
		if(vec == 4 && wide(tile_shape(P, 4, 256, 8)) && P.nf >= 128) {
			hipLaunchKernelGGL((k_quant_tile<4, 256, 8>), dim3(static_cast<unsigned>(up(f.O * f.I, P.nf))), dim3(256),
			                   P.tile_groups * sizeof(uint32_t), stream, a, aq, scales, P);
			return launched();
		}
		if(vec == 4 && wide(tile_shape(P, 4, 1024, 8))) {
			hipLaunchKernelGGL((k_quant_tile<4, 1024, 8>), dim3(static_cast<unsigned>(up(f.O * f.I, P.nf))), dim3(1024),
			                   P.tile_groups * sizeof(uint32_t), stream, a, aq, scales, P);
			return launched();
		}
		if(vec == 1 && wide(tile_shape(P, 1, 256, 32)) && P.nf >= 128) {
			hipLaunchKernelGGL((k_quant_tile<1, 256, 32>), dim3(static_cast<unsigned>(up(f.O * f.I, P.nf))), dim3(256),
			                   P.tile_groups * sizeof(uint32_t), stream, a, aq, scales, P);
			return launched();
		}
		if(vec == 1 && wide(tile_shape(P, 1, 1024, 32))) {
			hipLaunchKernelGGL((k_quant_tile<1, 1024, 32>), dim3(static_cast<unsigned>(up(f.O * f.I, P.nf))), dim3(1024),
			                   P.tile_groups * sizeof(uint32_t), stream, a, aq, scales, P);
			return launched();
		}
		int64_t const lanes = up(f.O * f.I, vec);
		P.LV = static_cast<int>(std::min<int64_t>(lanes, 64));
		P.KS = kBlock / P.LV;
		P.nf = static_cast<int64_t>(P.LV) * vec;
		int64_t const tiles = up(f.O * f.I, P.nf);
		if(tiles <= kMaxLeanBlocks) {
			// k chunks while the fiber tiles leave the chip short of blocks, each with some rounds of loads
			int64_t const chunks = std::max<int64_t>(1, std::min<int64_t>({up(4096, tiles), P.K / (P.KS * 16), 16384}));
			P.kchunk = up(P.K, chunks);
			dim3 const grid(static_cast<unsigned>(tiles), static_cast<unsigned>(up(P.K, P.kchunk)));
			scales_pass(1);
			if(vec == 4) {
				hipLaunchKernelGGL((k_quant_cols<4, 0>), grid, dim3(kBlock), 0, stream, a, aq, scales, P);
				hipLaunchKernelGGL((k_quant_cols<4, 1>), grid, dim3(kBlock), 0, stream, a, aq, scales, P);
			} else {
				hipLaunchKernelGGL((k_quant_cols<1, 0>), grid, dim3(kBlock), 0, stream, a, aq, scales, P);
				hipLaunchKernelGGL((k_quant_cols<1, 1>), grid, dim3(kBlock), 0, stream, a, aq, scales, P);
			}
			scales_pass(0);
			return launched();
		}
	}
	unsigned const grid = static_cast<unsigned>(std::min<int64_t>(P.groups, 65536));
	hipLaunchKernelGGL(k_quant_fp8, dim3(grid), dim3(kBlock), 0, stream, a, aq, scales, P);
	return launched();
}

} // namespace ttvx
