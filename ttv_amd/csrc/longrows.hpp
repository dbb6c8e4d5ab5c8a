// Rows (q fastest) longer than one vector per lane, with b in registers.
//
// A lane of the looping row kernels re-reads its values of b for every vector of A.  For 1-byte storage these are
// 64 bytes, 64 bytes apart from lane to lane, against 16 bytes of A: the vector cache serves one lane a cycle, and
// that, not HBM, set 2.5 TB/s (BF16: half of it, 4-5 TB/s).  Here a wave keeps the b of its piece of the row (4 KiB of A
// at most) and walks over the rows instead, so b is read once for all of them.  KS waves of a block take
// neighbouring pieces, the other 4 / KS further rows; what a block does not cover of the contraction is split over
// gridDim.y, with partial sums as in the split column kernel.
//
// MI355X, 256 MiB (rows of 4001: 240-480 MB), GB/s, before (the best looping row kernel) -> here:
//   row length   FP32           FP64           BF16           FP8
//   1000         5548 -> 5837   4220 -> 5311   5258 -> 5415   -
//   4000         5595 -> 5915   3697 -> 4755   4956 -> 5985   3542 -> 4676
//   4001         -              -              3915 -> 5698   2872 -> 3902
//   20000        5418 -> 5530   4051 -> 4897   4139 -> 5516   3693 -> 4441
//   100003       4877 -> 5069   3506 -> 4195   3433 -> 5575   2507 -> 3846
// 21 rows of 4000037 FP32: 64.7 -> 58.7 us with rows in even shares (20 + 1 rows: 76 us).
#pragma once

#include "kernels.hpp"

namespace ttvx
{

constexpr int kLongMaxRows = 256;                 // rows per wave (their sums meet in LDS)
// elements of a row per wave: N vectors of each lane (4, or 2 for rows that these hold)
constexpr int long_piece(int vec, int n) { return 64 * vec * n; }

template<typename S, int VEC, int N, bool KAHAN>
__global__ __launch_bounds__(kBlock) void k_long_rows(const S* __restrict__ A, const typename Traits<S>::acc* __restrict__ b,
                                                      void* __restrict__ C, Args P)
{
	using Acc = typename Traits<S>::acc;
	__shared__ Acc red[kBlock / 64][kLongMaxRows];
	int const lane = static_cast<int>(threadIdx.x) & 63;
	int const w    = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
	int const wk   = w & (P.KS - 1), wr = w / P.KS;               // piece of the chunk, rows of the block (KS = WK waves)
	int64_t const r0 = (static_cast<int64_t>(blockIdx.x) * (kBlock / 64 / P.KS) + wr) * P.OS;
	int const rows = static_cast<int>(r0 >= P.O ? 0 : (P.O - r0 < P.OS ? P.O - r0 : P.OS));
	for(int it = 0; it < P.kiter; ++it) {
		int64_t const k0 = static_cast<int64_t>(blockIdx.y) * P.kchunk +
		                   static_cast<int64_t>(it * P.KS + wk) * long_piece(VEC, N);
		// element of step s: k0 + s*64*VEC + lane*VEC; the row's last vector is clamped, lanes past it load the row's
		// first vector and add nothing
		int64_t kc[N];
		int head[N];                                              // leading elements of the vector that are not this lane's
		bool edge[N];                                             // the next lane does not hold the row's next vector
		Acc bv[N][VEC];
		bool const whole = k0 + long_piece(VEC, N) <= P.K;
#pragma unroll
		for(int s = 0; s < N; ++s) {
			int64_t const k = k0 + (static_cast<int64_t>(s) * 64 + lane) * VEC;
			bool const live = k < P.K;
			kc[s] = live ? row_clamp(k, P.K, VEC) : 0;
			head[s] = live ? static_cast<int>(k - kc[s]) : VEC;
			edge[s] = lane == 63 || k + 2 * VEC > P.K;
			load_b_vec<Acc, VEC>(b, kc[s], bv[s]);
		}
		// H rows at once (two in flight; an odd last one alone)
		auto sums = [&](auto h_, int r) {
			constexpr int H = decltype(h_)::value;
			Vec<S, VEC> raw[H][N];
			XVec<S, VEC> xr[H][N];            // realigned storage: the word past a vector comes from the next lane
#pragma unroll
			for(int h = 0; h < H; ++h)
#pragma unroll
				for(int s = 0; s < N; ++s) {
					if constexpr(kRealigned<S>) xr[h][s].load(A + (r0 + r + h) * P.sAo + kc[s], edge[s]);
					else raw[h][s].load(A + (r0 + r + h) * P.sAo + kc[s]);
				}
			__builtin_amdgcn_sched_barrier(0);
			Acc v[H];
#pragma unroll
			for(int h = 0; h < H; ++h) {
				Sum<Acc, KAHAN> acc;
#pragma unroll
				for(int s = 0; s < N; ++s) {
					Acc x[VEC];
					if constexpr(kRealigned<S>) xr[h][s].finish(edge[s], lane, raw[h][s]);
					decode(raw[h][s], x);
					if(!whole)
#pragma unroll
						for(int e = 0; e < VEC; ++e) x[e] = e < head[s] ? Acc(0) : x[e];
#pragma unroll
					for(int e = 0; e < VEC; ++e) acc.fma(x[e], bv[s][e]);
				}
				v[h] = acc.value();
			}
			int base, n;
			bool const store = halving_sum_ct<Acc, H, 64>(v, lane, base, n);     // lane 0: row r, lane 32: row r + 1
			if(store) red[w][r + base] = it == 0 ? v[0] : red[w][r + base] + v[0];
		};
		int r = 0;
		for(; r + 1 < rows; r += 2) sums(std::integral_constant<int, 2>{}, r);
		if(r < rows) sums(std::integral_constant<int, 1>{}, r);
	}
	__syncthreads();
	if(wk != 0) return;
	for(int r = lane; r < rows; r += 64) {
		Acc v = red[w][r];
		for(int q = 1; q < P.KS; ++q) v += red[w + q][r];
		store_out<Acc, kScaled<S>>(C, P, r0 + r, 0, v);
	}
}

} // namespace ttvx
