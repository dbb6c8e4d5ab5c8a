// Products on views whose free modes do not fold to three dimensions (blocks of a larger tensor).
//
// The free dimension 0 or the contraction has unit stride; every other free dimension is an outer index
// whose A and C offsets a thread finds once, by mixed-radix division, before its contraction loop.
//
//   k_view_cols  dimension 0 has unit stride in A and C: a lane owns one vector of VEC columns of one outer
//                index and walks k; the lanes of a wave take consecutive vectors, so a wave reads runs of
//                whole rows whatever the row length (no lanes are lost to a row width that is no power of two)
//   k_view_rows, k_view_long_rows  the contraction has unit stride: rows of at most 64 vectors take exactly
//                their vectors' lanes (20 vectors: 3 rows per wave; a power of two of lanes with steps over a
//                row measured 71 us below), longer ones a wave or a block each
//
// All are bound by HBM: every line of A that the view touches is read once, with 8 vectors in flight per
// lane.  MI355X, the interior 96x90x84x80 FP32 of a tensor 4 larger in every mode (235 MB a product):
// columns 96-101 us -> 44-48 us (5.0-5.4 TB/s), rows 998 us -> 47 us, against k_strided (one thread per
// output, one 4-byte load in flight), which is kept for views in which nothing has unit stride.
#pragma once

#include "kernels.hpp"

namespace ttvx
{

// A and C offsets of outer index o over the dimensions first .. nd-1 (fastest first)
__device__ __forceinline__ void view_offsets(const StridedArgs& G, int first, int64_t o, int64_t& offa, int64_t& offc)
{
	offa = 0;
	offc = 0;
	if(G.idx32) {
		uint32_t rest = static_cast<uint32_t>(o);
		for(int d = first; d < G.nd; ++d) {
			uint32_t const q = div_by(rest, G.div[d]);
			uint32_t const idx = rest - q * static_cast<uint32_t>(G.n[d]);
			rest = q;
			offa += static_cast<int64_t>(idx) * G.sa[d];
			offc += static_cast<int64_t>(idx) * G.sc[d];
		}
	} else {
		int64_t rest = o;
		for(int d = first; d < G.nd; ++d) {
			int64_t const q = rest / G.n[d];
			int64_t const idx = rest - q * G.n[d];
			rest = q;
			offa += idx * G.sa[d];
			offc += idx * G.sc[d];
		}
	}
}

// Thread t of a block: vector unit t % UL of the block (UL = kBlock / ks), contraction group t / UL, which
// takes k = group, group + ks, ...; ks > 1 (few outputs) meets in LDS.
template<typename S, int VEC, bool KAHAN>
__global__ __launch_bounds__(kBlock) void k_view_cols(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                      void* __restrict__ C, StridedArgs G)
{
	using Acc = typename Traits<S>::acc;
	extern __shared__ unsigned char smem_raw[];
	Acc* const red = reinterpret_cast<Acc*>(smem_raw);       // [ks][VEC][UL] when ks > 1
	constexpr int KL = 8;                                    // loads in flight per lane
	int const t  = static_cast<int>(threadIdx.x);
	int const ul = kBlock / G.ks;
	int const l  = t & (ul - 1);
	int const kg = t / ul;
	int64_t const I = G.n[0];
	int64_t const iv = (I + VEC - 1) / VEC;
	int64_t const unit = static_cast<int64_t>(blockIdx.x) * ul + l;
	bool const live = unit < G.units;
	int64_t const uc = live ? unit : G.units - 1;            // tail lanes re-read live data and store nothing
	int64_t const o = G.idx32 ? static_cast<int64_t>(div_by(static_cast<uint32_t>(uc), G.div[0])) : uc / iv;
	int64_t const i  = (uc - o * iv) * VEC;
	int64_t const ic = i + VEC <= I ? i : I - VEC;           // a row's last vector is clamped to its end
	int64_t offa, offc;
	view_offsets(G, 1, o, offa, offc);
	const S* pa = A + offa + ic + kg * G.sAk;
	const Acc* pb = b + kg;
	int64_t const step = static_cast<int64_t>(G.ks) * G.sAk;
	int64_t nk = kg < G.K ? (G.K - 1 - kg) / G.ks + 1 : 0;
	Sum<Acc, KAHAN> acc[VEC];
	auto round = [&](auto n_) {
		constexpr int N = decltype(n_)::value;
		Vec<S, VEC> raw[N];
		Acc bk[N];
#pragma unroll
		for(int j = 0; j < N; ++j) raw[j].load(pa + j * step);
#pragma unroll
		for(int j = 0; j < N; ++j) bk[j] = pb[j * G.ks];
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for(int j = 0; j < N; ++j) {
			Acc x[VEC];
			decode(raw[j], x);
#pragma unroll
			for(int e = 0; e < VEC; ++e) acc[e].fma(x[e], bk[j]);
		}
		pa += N * step;
		pb += N * G.ks;
		nk -= N;
	};
	while(nk >= KL) round(std::integral_constant<int, KL>{});
	if(nk >= 4) round(std::integral_constant<int, 4>{});
	if(nk >= 2) round(std::integral_constant<int, 2>{});
	if(nk >= 1) round(std::integral_constant<int, 1>{});

	Acc v[VEC];
#pragma unroll
	for(int e = 0; e < VEC; ++e) v[e] = acc[e].value();
	if(G.ks > 1) {
#pragma unroll
		for(int e = 0; e < VEC; ++e) red[(kg * VEC + e) * ul + l] = v[e];
		__syncthreads();
		if(kg != 0) return;
		for(int g = 1; g < G.ks; ++g)
#pragma unroll
			for(int e = 0; e < VEC; ++e) v[e] += red[(g * VEC + e) * ul + l];
	}
	if(!live) return;
	if constexpr(kScaled<S>) scale_vec<Acc, VEC>(G.scales, G.fps, o * I + ic, v);
	Acc* const dst = static_cast<Acc*>(C) + offc + ic;
	constexpr int PER = 16 / static_cast<int>(sizeof(Acc));
	if(VEC >= PER && ic == i) {
#pragma unroll
		for(int c = 0; c < VEC / PER; ++c) {
			u32x4_a4 q;
			uint32_t const* src = reinterpret_cast<const uint32_t*>(v) + 4 * c;
			q.x = src[0]; q.y = src[1]; q.z = src[2]; q.w = src[3];
			*TTVX_GLOBAL_W(u32x4_a4, dst + c * PER) = q;
		}
	} else {
		// element ic + e; the ones before i belong to the vector before
#pragma unroll
		for(int e = 0; e < VEC; ++e)
			if(ic + e >= i) dst[e] = v[e];
	}
}

// Rows of at most 64 vectors at the offsets of the outer index: a row takes exactly its vectors' lanes, 64 / lpr
// rows per wave and U row sets, every load issued before the first use; sums by segmented shifts.  Row r of set
// u of wave w: (w*U + u)*rpw + r.
template<typename S, int VEC, int U, bool KAHAN>
__global__ __launch_bounds__(kBlock) void k_view_rows(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                      void* __restrict__ C, StridedArgs G)
{
	using Acc = typename Traits<S>::acc;
	int const lane = static_cast<int>(threadIdx.x) & 63;
	int const lpr  = G.lpr;
	int const rpw  = 64 / lpr;
	int const r    = lane / lpr;
	int const kl   = lane - r * lpr;
	int64_t const k0 = static_cast<int64_t>(kl) * VEC;
	bool const live = r < rpw;
	int64_t const kc = live ? row_clamp(k0, G.K, VEC) : 0;
	int64_t const wave = static_cast<int64_t>(blockIdx.x) * (kBlock / 64) + (threadIdx.x >> 6);
	int64_t const row0 = wave * U * rpw + (live ? r : 0);
	Acc bb[VEC];
	load_b_vec<Acc, VEC>(b, kc, bb);
	Vec<S, VEC> raw[U];
	int64_t offc[U];
#pragma unroll
	for(int u = 0; u < U; ++u) {
		int64_t const row = row0 + static_cast<int64_t>(u) * rpw;
		int64_t offa;
		view_offsets(G, 0, row < G.outputs ? row : G.outputs - 1, offa, offc[u]);
		raw[u].load(A + offa + kc);
	}
	Acc v[U];
#pragma unroll
	for(int u = 0; u < U; ++u) {
		Sum<Acc, KAHAN> acc;
		Acc x[VEC];
		decode(raw[u], x);
		if(kc != k0) mask_head<Acc, VEC>(x, k0 - kc);
#pragma unroll
		for(int e = 0; e < VEC; ++e) acc.fma(x[e], bb[e]);
		v[u] = acc.value();
	}
	segment_sum<Acc, U>(v, kl, lpr);
	if(kl != 0 || !live) return;
#pragma unroll
	for(int u = 0; u < U; ++u) {
		int64_t const row = row0 + static_cast<int64_t>(u) * rpw;
		if(row >= G.outputs) continue;
		if constexpr(kScaled<S>)
			if(G.scales != nullptr) v[u] *= static_cast<Acc>(G.scales[row / G.fps]);
		static_cast<Acc*>(C)[offc[u]] = v[u];
	}
}

// Longer rows: one wave per row, or the whole block when rows are few (lpr = 64 or kBlock)
template<typename S, int VEC, bool KAHAN>
__global__ __launch_bounds__(kBlock) void k_view_long_rows(const S* __restrict__ A,
                                                           const typename Traits<S>::acc* __restrict__ b,
                                                           void* __restrict__ C, StridedArgs G)
{
	using Acc = typename Traits<S>::acc;
	__shared__ Acc red[kBlock / 64];
	constexpr int KL = VEC >= 8 ? 4 : 8;                     // vectors in flight per lane
	int const t   = static_cast<int>(threadIdx.x);
	int const lpr = G.lpr;
	int const kl  = t & (lpr - 1);
	int64_t const row = static_cast<int64_t>(blockIdx.x) * (kBlock / lpr) + t / lpr;
	int64_t offa, offc;
	view_offsets(G, 0, row < G.outputs ? row : G.outputs - 1, offa, offc);
	const S* const pa = A + offa;
	int64_t const kstride = static_cast<int64_t>(lpr) * VEC;
	Sum<Acc, KAHAN> acc;
	for(int64_t k = static_cast<int64_t>(kl) * VEC; k < G.K; k += KL * kstride) {
		Vec<S, VEC> raw[KL];
		Acc bv[KL][VEC];
		// steps past the row's end re-read the round's first vector and are not added
#pragma unroll
		for(int j = 0; j < KL; ++j) {
			int64_t const kc = row_clamp(k + j * kstride < G.K ? k + j * kstride : k, G.K, VEC);
			raw[j].load(pa + kc);
			load_b_vec<Acc, VEC>(b, kc, bv[j]);
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for(int j = 0; j < KL; ++j) {
			int64_t const ks = k + j * kstride;
			if(ks < G.K) {
				int64_t const kc = row_clamp(ks, G.K, VEC);
				Acc x[VEC];
				decode(raw[j], x);
				if(kc != ks) mask_head<Acc, VEC>(x, ks - kc);
#pragma unroll
				for(int e = 0; e < VEC; ++e) acc.fma(x[e], bv[j][e]);
			}
		}
	}
	Acc v = acc.value();
	for(int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
	if(lpr > 64) {
		if((t & 63) == 0) red[t >> 6] = v;
		__syncthreads();
		v = red[0];
		for(int w = 1; w < kBlock / 64; ++w) v += red[w];
	}
	if(kl != 0 || row >= G.outputs) return;
	if constexpr(kScaled<S>)
		if(G.scales != nullptr) v *= static_cast<Acc>(G.scales[row / G.fps]);
	static_cast<Acc*>(C)[offc] = v;
}

} // namespace ttvx
