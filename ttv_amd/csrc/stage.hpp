// Column products whose slabs are a few KiB (few columns, short contractions), staged through LDS.
//
// With I columns narrower than a cache line the column tiles lose lanes to the row width and fetch lines in
// pieces.  Slabs that follow one another in memory (sAk == I, sAo == K*I) need neither: a block reads OS whole
// slabs as one contiguous run of 16-byte vectors (at most kStageBytes, all loads in flight at once), lays them
// into LDS, and every thread sums the K values of its outputs from there.  Bound by HBM: LDS moves each byte
// twice, at a tenth of its rate; the unaligned rows of 2- and 1-byte storage cost nothing extra, because only
// the LDS reads are of element size.  Tiles of 16 KiB (8 blocks per CU) reach 4.1-5.3 TB/s where 32 KiB reach 5.9.
//
// MI355X, 256 MiB, GB/s of this kernel against the best of the direct column tiles:
//   columns x contraction   FP32          FP64          BF16          FP8
//   2 x 8                   5988 / 3488   6179 / 4618   5601 / 2108   4508 / 1237
//   8 x 8                   6179 / 4740   6367 / 5716   6023 / 1745   5187 / 978
//   11 x 13                 4793 / 3403   5467 / 4229   4204 / 2903   3279 / 895
//   45 x 32                 6258 / 6013   6523 / 5150   5840 / 5186   3898 / 3906
//   128 x 32                6327 / 6141   6373 / 5885   6373 / 6069   5849 / 4919
// (odd rows of FP8 read single bytes from LDS, which is what bounds them).
#pragma once

#include "kernels.hpp"

namespace ttvx
{

constexpr int kStageBytes = 32 * 1024;       // LDS per block: 5 blocks of 4 waves per CU, 8 loads per lane
constexpr int kStageMaxPV = 4;               // most columns per thread

// PV consecutive elements in LDS (aligned to PV elements)
template<typename S, int PV>
__device__ __forceinline__ void stage_read(const unsigned char* p, typename Traits<S>::acc (&x)[PV])
{
	Vec<S, PV> v;
	constexpr int BYTES = PV * static_cast<int>(sizeof(S));
	if constexpr(BYTES == 1)       v.w[0] = *p;
	else if constexpr(BYTES == 2)  v.w[0] = *reinterpret_cast<const uint16_t*>(p);
	else if constexpr(BYTES == 4)  v.w[0] = *reinterpret_cast<const uint32_t*>(p);
	else if constexpr(BYTES == 8) {
		u32x2 const q = *reinterpret_cast<const u32x2*>(p);
		v.w[0] = q.x; v.w[1] = q.y;
	} else {
#pragma unroll
		for(int c = 0; c < BYTES / 16; ++c) {
			u32x4 const q = reinterpret_cast<const u32x4*>(p)[c];
			v.w[4 * c] = q.x; v.w[4 * c + 1] = q.y; v.w[4 * c + 2] = q.z; v.w[4 * c + 3] = q.w;
		}
	}
	decode(v, x);
}

// SWZ: LDS holds byte a at a + 16 * (a / 256), so that rows of nearly a multiple of 256 bytes do not all start in
// the same banks
template<bool SWZ> __device__ __forceinline__ int stage_at(int a) { return SWZ ? a + ((a >> 8) << 4) : a; }

// The block's `bytes` contiguous bytes from src into LDS, slabs of `slab` bytes P.pitch apart
template<typename S, bool SWZ = false>
__device__ __forceinline__ void stage_load(const unsigned char* src, int bytes, int slab, const Args& P, unsigned char* lds)
{
	constexpr int R = kStageBytes / (16 * kBlock);
	int const t = static_cast<int>(threadIdx.x);
	int const nv = bytes >> 4;
	if(nv > 0) {
		u32x4_b v[R];
#pragma unroll
		for(int r = 0; r < R; ++r) {
			// lanes past the end re-read the first vector (no branch between the loads)
			int const idx = r * kBlock + t;
			v[r] = __builtin_nontemporal_load(TTVX_GLOBAL(u32x4_b, src) + (idx < nv ? idx : 0));
		}
		__builtin_amdgcn_sched_barrier(0);
		// P.pitch == slab, or slab + 16 (slabs of an even number of vectors: their starts then spread over the banks)
#pragma unroll
		for(int r = 0; r < R; ++r) {
			int const idx = r * kBlock + t;
			if(idx < nv) {
				int const at = SWZ ? idx + (idx >> 4)
				                   : (P.pitch == slab ? idx : idx + static_cast<int>(div_by(static_cast<uint32_t>(idx), P.by_slab)));
				reinterpret_cast<u32x4*>(lds)[at] = v[r];
			}
		}
	}
	// the end of the last block's run (no padding there: a padded slab is whole vectors)
#pragma unroll 1
	for(int e = nv * 16 + t * static_cast<int>(sizeof(S)); e < bytes; e += kBlock * static_cast<int>(sizeof(S)))
		*reinterpret_cast<S*>(lds + stage_at<SWZ>(e)) = *reinterpret_cast<const S*>(src + e);
}

// Item: slabs [item*OS, item*OS + OS).  Thread t: outputs t % JL (+ JL, ...), contraction group t / JL of KG = 256 / JL
// (JL = 1 << itShift lanes; several groups only when one round of lanes covers the item's outputs).
template<typename S, int PV, bool KAHAN>
__device__ __forceinline__ void stage_item(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                           void* __restrict__ C, const Args& P, int64_t item, unsigned char* lds)
{
	using Acc = typename Traits<S>::acc;
	int const t = static_cast<int>(threadIdx.x);
	int64_t const o0 = item * P.OS;
	int const slabs = static_cast<int>(P.O - o0 < P.OS ? P.O - o0 : P.OS);
	int const K = static_cast<int>(P.K), I = static_cast<int>(P.I);
	int const slab = K * I * static_cast<int>(sizeof(S));
	int const bytes = slabs * slab;
	const unsigned char* const src = reinterpret_cast<const unsigned char*>(A) + o0 * slab;
	stage_load<S>(src, bytes, slab, P, lds);
	__syncthreads();

	int const JL = 1 << P.itShift, KG = kBlock >> P.itShift;
	int const jl = t & (JL - 1), kg = t >> P.itShift;
	int const ipv = I / PV;
	int const n = slabs * ipv;
	int const row = I * static_cast<int>(sizeof(S));
	int const step = KG * row;
	bool const uniform = JL >= 64;           // one k for a whole wave: b through the scalar cache
	const Acc* const bu = b + __builtin_amdgcn_readfirstlane(kg);
	const Acc* const bl = b + kg;
#pragma unroll 1
	for(int j = jl; j < n || KG > 1; j += JL) {
		int const jc = j < n ? j : n - 1;    // spare lanes repeat the last output and store nothing
		int const o = static_cast<int>(div_by(static_cast<uint32_t>(jc), P.by_i));
		int const i = (jc - o * ipv) * PV;
		const unsigned char* p = lds + o * P.pitch + i * static_cast<int>(sizeof(S)) + kg * row;
		Sum<Acc, KAHAN> acc[PV];
		auto sum = [&](const Acc* bp) {
			int left = kg < K ? (K - 1 - kg) / KG + 1 : 0;
			auto round = [&](auto n_) {
				constexpr int N = decltype(n_)::value;
				Acc x[N][PV];
#pragma unroll
				for(int u = 0; u < N; ++u) stage_read<S, PV>(p + u * step, x[u]);
#pragma unroll
				for(int u = 0; u < N; ++u)
#pragma unroll
					for(int e = 0; e < PV; ++e) acc[e].fma(x[u][e], bp[u * KG]);
				p += N * step;
				bp += N * KG;
				left -= N;
			};
#pragma unroll 1
			while(left >= 8) round(std::integral_constant<int, 8>{});
			if(left >= 4) round(std::integral_constant<int, 4>{});
			if(left >= 2) round(std::integral_constant<int, 2>{});
			if(left >= 1) round(std::integral_constant<int, 1>{});
		};
		if(uniform) sum(bu);
		else        sum(bl);
		Acc v[PV];
#pragma unroll
		for(int e = 0; e < PV; ++e) v[e] = acc[e].value();
		if(KG > 1) {
			// lanes of one output: jl + JL*g inside the wave, then the waves' sums in LDS
			for(int d = JL; d < 64; d <<= 1)
#pragma unroll
				for(int e = 0; e < PV; ++e) v[e] += __shfl_xor(v[e], d, 64);
			int const w = JL < 64 ? 64 : JL;         // threads that hold one partial sum of every output
			int const parts = kBlock / w;
			Acc* const red = reinterpret_cast<Acc*>(lds);
			__syncthreads();                         // every read of the slabs is done
			if((t & (w - 1)) < JL)
#pragma unroll
				for(int e = 0; e < PV; ++e) red[((t / w) * PV + e) * JL + jl] = v[e];
			__syncthreads();
			if(t >= JL || j >= n) return;
			for(int g = 1; g < parts; ++g)
#pragma unroll
				for(int e = 0; e < PV; ++e) v[e] += red[(g * PV + e) * JL + jl];
		}
		int64_t const oo = o0 + o;
		if constexpr(kScaled<S>) {
			if(P.scales != nullptr && P.fps32) {
				// outputs fit 31 bits: no 64-bit division (a third of the time of short contractions)
				uint32_t const j0 = static_cast<uint32_t>(oo) * static_cast<uint32_t>(I) + static_cast<uint32_t>(i);
				uint32_t const ga = div_by(j0, P.by_fps), gb = div_by(j0 + (PV - 1), P.by_fps);
				if(ga == gb) {
					float const s = P.scales[ga];
#pragma unroll
					for(int e = 0; e < PV; ++e) v[e] *= s;
				} else {
#pragma unroll
					for(int e = 0; e < PV; ++e) v[e] *= P.scales[div_by(j0 + e, P.by_fps)];
				}
			} else {
				scale_vec<Acc, PV>(P.scales, P.fps, oo * P.I + i, v);
			}
		}
		Acc* const dst = static_cast<Acc*>(C) + oo * P.sCo + i;
		// consecutive lanes write consecutive outputs: whole lines, non-temporal
		constexpr int BYTES = PV * static_cast<int>(sizeof(Acc));
		if constexpr(BYTES >= 16) {
#pragma unroll
			for(int c = 0; c < BYTES / 16; ++c) {
				u32x4_b q;
				uint32_t const* w = reinterpret_cast<const uint32_t*>(v) + 4 * c;
				q.x = w[0]; q.y = w[1]; q.z = w[2]; q.w = w[3];
				__builtin_nontemporal_store(q, TTVX_GLOBAL_W(u32x4_b, dst) + c);
			}
		} else {
#pragma unroll
			for(int e = 0; e < PV; ++e) __builtin_nontemporal_store(v[e], TTVX_GLOBAL_W(Acc, dst) + e);
		}
		if(KG > 1) return;
	}
}

// MI355X, 256 MiB, GB/s of k_stage_rows against the best direct row kernel (k_rows, k_dot):
//   row length   FP64          BF16          FP8
//   33           6061 / 5627   5962 / 4471   4775 / 3096
//   129          6292 / 3437   5300 / 4344   5743 / 3273
//   255          6126 / 4356   5011 / 4711   4536 / 4334
//   513          5576 / 4390   4471 / 3213   4194 / 2955
// Rows of whole 16-byte vectors of the 4-, 2- and 1-byte types stay with k_rows (FP8 rows of 128: 5678 / 5797), and
// the swizzle is for rows whose starts would collide (FP8 rows of 511 without it 2.8 TB/s).
// Rows (q fastest) of FP64, BF16 and FP8 in the same way: item = rows [item*OS, item*OS + OS), G = 1 << itShift neighbouring lanes per row,
// which take its words (of 4 bytes; 8 for FP64) in turn.  Words are read from the aligned ones that hold them, so
// rows of 2- and 1-byte storage may start anywhere.
template<typename S, bool KAHAN, bool SWZ>
__device__ __forceinline__ void stage_rows_item(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                void* __restrict__ C, const Args& P, int64_t item, unsigned char* lds)
{
	using Acc = typename Traits<S>::acc;
	constexpr int WB = sizeof(S) == 8 ? 8 : 4;                        // bytes of a word
	constexpr int E = WB / static_cast<int>(sizeof(S));               // elements of a word
	int const t = static_cast<int>(threadIdx.x);
	int64_t const o0 = item * P.OS;
	int const rows = static_cast<int>(P.O - o0 < P.OS ? P.O - o0 : P.OS);
	int const K = static_cast<int>(P.K);
	int const row = K * static_cast<int>(sizeof(S));
	int const G = 1 << P.itShift;
	// with several lanes per row b comes from LDS too (through the vector cache it took as long as A: BF16 rows of
	// 256 4.3 TB/s)
	Acc* const lb = reinterpret_cast<Acc*>(lds + P.red);
	if(G > 1)
		for(int k = t; k < K; k += kBlock) lb[k] = b[k];
	stage_load<S, SWZ>(reinterpret_cast<const unsigned char*>(A) + o0 * row, rows * row, row, P, lds);
	__syncthreads();

	int const g = t & (G - 1);
	int const words = K / E;                                          // whole words of a row
#pragma unroll 1
	for(int r0 = 0; r0 < rows; r0 += kBlock >> P.itShift) {
		int const r = r0 + (t >> P.itShift);
		bool const live = r < rows;
		int const at = (live ? r : 0) * P.pitch;
		int const at0 = at & ~(WB - 1);                               // the word at or below the row's first element
		uint32_t const m = static_cast<uint32_t>(at & 3);
		Sum<Acc, KAHAN> acc;
		// N words w, w + step, ... of the row into x; those of 2- and 1-byte storage are funnel-shifted from the two
		// aligned words that hold them
		auto words_at = [&](auto n_, int w, int step, auto& x) {
			constexpr int N = decltype(n_)::value;
			if constexpr(sizeof(S) == 8) {
#pragma unroll
				for(int u = 0; u < N; ++u) x[u] = *reinterpret_cast<const double*>(lds + stage_at<SWZ>(at0 + 8 * (w + u * step)));
			} else {
				uint32_t lo[N], hi[N];
#pragma unroll
				for(int u = 0; u < N; ++u) {
					int const a = at0 + 4 * (w + u * step);
					lo[u] = *reinterpret_cast<const uint32_t*>(lds + stage_at<SWZ>(a));
					hi[u] = *reinterpret_cast<const uint32_t*>(lds + stage_at<SWZ>(a + 4));
				}
#pragma unroll
				for(int u = 0; u < N; ++u) {
					Vec<S, E> v;
					v.w[0] = __builtin_amdgcn_alignbyte(hi[u], lo[u], m);
					Acc y[E];
					decode(v, y);
#pragma unroll
					for(int e = 0; e < E; ++e) x[u * E + e] = y[e];
				}
			}
		};
		auto run = [&](auto lds_b, const Acc* bp, int w, int step) {
			constexpr bool kLds = decltype(lds_b)::value;
			int left = w < words ? (words - 1 - w) / step + 1 : 0;
			auto round = [&](auto n_) {
				constexpr int N = decltype(n_)::value;
				Acc x[N * E], bv[N * E];
#pragma unroll
				for(int u = 0; u < N; ++u) {
					struct alignas(E * sizeof(Acc)) Word { Acc v[E]; };
					if constexpr(kLds) {
						Word const q = *reinterpret_cast<const Word*>(bp + u * step * E);
#pragma unroll
						for(int e = 0; e < E; ++e) bv[u * E + e] = q.v[e];
					} else {
#pragma unroll
						for(int e = 0; e < E; ++e) bv[u * E + e] = bp[u * step * E + e];
					}
				}
				words_at(n_, w, step, x);
#pragma unroll
				for(int u = 0; u < N * E; ++u) acc.fma(x[u], bv[u]);
				w += N * step;
				bp += N * step * E;
				left -= N;
			};
#pragma unroll 1
			while(left >= 8) round(std::integral_constant<int, 8>{});
			if(left >= 4) round(std::integral_constant<int, 4>{});
			if(left >= 2) round(std::integral_constant<int, 2>{});
			if(left >= 1) round(std::integral_constant<int, 1>{});
		};
		if(G == 1) run(std::false_type{}, b, 0, 1);   // one k for a whole wave: b through the scalar cache
		else       run(std::true_type{}, lb + g * E, g, G);
		if constexpr(E > 1) {
			// the last elements of a row whose length a word does not divide
			if(g == 0)
				for(int k = words * E; k < K; ++k) {
					Acc x[1];
					stage_read<S, 1>(lds + stage_at<SWZ>(at + k * static_cast<int>(sizeof(S))), x);
					acc.fma(x[0], b[k]);
				}
		}
		Acc v = acc.value();
		for(int d = G >> 1; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
		if(live && g == 0) {
			int64_t const o = o0 + r;
			if constexpr(kScaled<S>)
				if(P.scales != nullptr) v *= P.fps32 ? P.scales[div_by(static_cast<uint32_t>(o), P.by_fps)] : P.scales[o / P.fps];
			static_cast<Acc*>(C)[o * P.sCo] = v;
		}
	}
}

template<typename S, bool KAHAN, bool SWZ>
__global__ __launch_bounds__(kBlock, 5) void k_stage_rows(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                          void* __restrict__ C, Args P)
{
	extern __shared__ __attribute__((aligned(16))) unsigned char stage_lds[];
	stage_rows_item<S, KAHAN, SWZ>(A, b, C, P, blockIdx.x, stage_lds);
}

// FP64 slabs that no tile holds, in chunks of OS whole rows (dense slabs: a chunk is one contiguous run, whatever the
// row length).  Block (x, y): slab x, contraction rows [y*kchunk, (y+1)*kchunk).  A lane keeps its outputs (vector
// t % JL) over all chunks; the 5 blocks of a CU overlap each other's loads and sums.
// MI355X, 256 MiB, GB/s against the best direct column tile, contractions of 300 and 1000: rows of 64 5879 / 5280,
// 5258 / 5321; of 100 5065 / 4346, 5180 / 3813; of 255 5436 / 4556, 5071 / 4042; of 256 5045 / 5173, 4587 / 5189.
template<int PV>
__global__ __launch_bounds__(kBlock, 5) void k_stage_chunks(const double* __restrict__ A, const double* __restrict__ b,
                                                            void* __restrict__ C, Args P)
{
	extern __shared__ __attribute__((aligned(16))) unsigned char stage_lds[];
	unsigned char* const lds = stage_lds;
	constexpr int SZ = 8;
	int const t = static_cast<int>(threadIdx.x);
	int64_t const o = blockIdx.x;
	int const I = static_cast<int>(P.I), row = I * SZ;
	int64_t const kb = static_cast<int64_t>(blockIdx.y) * P.kchunk;
	int64_t const ke = kb + P.kchunk < P.K ? kb + P.kchunk : P.K;
	double* const lb = reinterpret_cast<double*>(lds + P.pitch);      // the chunk's b (lanes of a wave on several rows)
	int const JL = 1 << P.itShift, KG = kBlock >> P.itShift;
	int const jl = t & (JL - 1), kg = t >> P.itShift;
	int const n = I / PV;
	int const j = jl < n ? jl : n - 1;       // spare lanes repeat the last output and store nothing
	int const step = KG * row;
	bool const uniform = JL >= 64;           // one k for a whole wave: b through the scalar cache
	Sum<double, false> acc[PV];
	for(int64_t k = kb; k < ke; k += P.OS) {
		int const rows = static_cast<int>(ke - k < P.OS ? ke - k : P.OS);
		stage_load<double>(reinterpret_cast<const unsigned char*>(A + (o * P.K + k) * I), rows * row, P.pitch, P, lds);
		if(!uniform)
			for(int q = t; q < rows; q += kBlock) lb[q] = b[k + q];
		__syncthreads();
		const unsigned char* p = lds + j * PV * SZ + kg * row;
		auto sum = [&](const double* bp) {
			int left = kg < rows ? (rows - 1 - kg) / KG + 1 : 0;
			auto round = [&](auto n_) {
				constexpr int N = decltype(n_)::value;
				double x[N][PV];
#pragma unroll
				for(int u = 0; u < N; ++u) stage_read<double, PV>(p + u * step, x[u]);
#pragma unroll
				for(int u = 0; u < N; ++u)
#pragma unroll
					for(int e = 0; e < PV; ++e) acc[e].fma(x[u][e], bp[u * KG]);
				p += N * step;
				bp += N * KG;
				left -= N;
			};
#pragma unroll 1
			while(left >= 8) round(std::integral_constant<int, 8>{});
			if(left >= 4) round(std::integral_constant<int, 4>{});
			if(left >= 2) round(std::integral_constant<int, 2>{});
			if(left >= 1) round(std::integral_constant<int, 1>{});
		};
		if(uniform) sum(b + k + __builtin_amdgcn_readfirstlane(kg));
		else        sum(lb + kg);
		__syncthreads();
	}
	double s[PV];
#pragma unroll
	for(int e = 0; e < PV; ++e) s[e] = acc[e].value();
	if(KG > 1) {
		for(int d = JL; d < 64; d <<= 1)
#pragma unroll
			for(int e = 0; e < PV; ++e) s[e] += __shfl_xor(s[e], d, 64);
		int const w = JL < 64 ? 64 : JL;
		int const parts = kBlock / w;
		double* const red = reinterpret_cast<double*>(lds);
		if((t & (w - 1)) < JL)
#pragma unroll
			for(int e = 0; e < PV; ++e) red[((t / w) * PV + e) * JL + jl] = s[e];
		__syncthreads();
		if(t >= JL) return;
		for(int g = 1; g < parts; ++g)
#pragma unroll
			for(int e = 0; e < PV; ++e) s[e] += red[(g * PV + e) * JL + jl];
	}
	if(jl >= n) return;
#pragma unroll
	for(int e = 0; e < PV; ++e) store_out<double, false>(C, P, o, static_cast<int64_t>(jl) * PV + e, s[e]);
}

// (at most 96 registers: 5 waves per SIMD, as many as the LDS leaves room for)
template<typename S, int PV, bool KAHAN>
__global__ __launch_bounds__(kBlock, 5) void k_stage(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                  void* __restrict__ C, Args P)
{
	extern __shared__ __attribute__((aligned(16))) unsigned char stage_lds[];
	stage_item<S, PV, KAHAN>(A, b, C, P, blockIdx.x, stage_lds);
}

} // namespace ttvx
