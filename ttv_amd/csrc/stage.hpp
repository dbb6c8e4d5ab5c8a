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

// Item: slabs [item*OS, item*OS + OS).  Thread t: outputs t % JL (+ JL, ...), contraction group t / JL of KG = 256 / JL
// (JL = 1 << itShift lanes; several groups only when one round of lanes covers the item's outputs).
template<typename S, int PV, bool KAHAN>
__device__ __forceinline__ void stage_item(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                           void* __restrict__ C, const Args& P, int64_t item, unsigned char* lds)
{
	using Acc = typename Traits<S>::acc;
	constexpr int R = kStageBytes / (16 * kBlock);
	int const t = static_cast<int>(threadIdx.x);
	int64_t const o0 = item * P.OS;
	int const slabs = static_cast<int>(P.O - o0 < P.OS ? P.O - o0 : P.OS);
	int const K = static_cast<int>(P.K), I = static_cast<int>(P.I);
	int const slab = K * I * static_cast<int>(sizeof(S));
	int const bytes = slabs * slab;
	const unsigned char* const src = reinterpret_cast<const unsigned char*>(A) + o0 * slab;
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
				int const at = P.pitch == slab ? idx : idx + static_cast<int>(div_by(static_cast<uint32_t>(idx), P.by_slab));
				reinterpret_cast<u32x4*>(lds)[at] = v[r];
			}
		}
	}
	// the end of the last block's run (no padding there: a padded slab is whole vectors)
#pragma unroll 1
	for(int e = nv * 16 + t * static_cast<int>(sizeof(S)); e < bytes; e += kBlock * static_cast<int>(sizeof(S)))
		*reinterpret_cast<S*>(lds + e) = *reinterpret_cast<const S*>(src + e);
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

// (at most 96 registers: 5 waves per SIMD, as many as the LDS leaves room for)
template<typename S, int PV, bool KAHAN>
__global__ __launch_bounds__(kBlock, 5) void k_stage(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                  void* __restrict__ C, Args P)
{
	extern __shared__ __attribute__((aligned(16))) unsigned char stage_lds[];
	stage_item<S, PV, KAHAN>(A, b, C, P, blockIdx.x, stage_lds);
}

} // namespace ttvx
