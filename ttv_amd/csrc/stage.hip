// Launches of the LDS-staged products (stage.hpp) for every storage type.
#include "stage.hpp"

#include "runtime.hpp"

namespace ttvx
{

namespace
{
template<typename S, int PV>
void go(const Config& cfg, const void* a, const void* b, void* c, bool kahan, hipStream_t s)
{
	using Acc = typename Traits<S>::acc;
	dim3 const grid(static_cast<unsigned>(cfg.grid)), block(kBlock);
	if(!std::is_same_v<Acc, double> && kahan)
		hipLaunchKernelGGL((k_stage<S, PV, !std::is_same_v<Acc, double>>), grid, block, cfg.shmem, s, static_cast<const S*>(a),
		                   static_cast<const Acc*>(b), c, cfg.args);
	else
		hipLaunchKernelGGL((k_stage<S, PV, false>), grid, block, cfg.shmem, s, static_cast<const S*>(a),
		                   static_cast<const Acc*>(b), c, cfg.args);
}

template<int PV>
void go_chunks(const Config& cfg, const void* a, const void* b, void* c, hipStream_t s)
{
	hipLaunchKernelGGL((k_stage_chunks<PV>), dim3(static_cast<unsigned>(cfg.grid), static_cast<unsigned>(cfg.ksplit)),
	                   dim3(kBlock), cfg.shmem, s, static_cast<const double*>(a), static_cast<const double*>(b), c, cfg.args);
}

template<typename S, bool SWZ>
void go_rows(const Config& cfg, const void* a, const void* b, void* c, bool kahan, hipStream_t s)
{
	using Acc = typename Traits<S>::acc;
	dim3 const grid(static_cast<unsigned>(cfg.grid)), block(kBlock);
	if(!std::is_same_v<Acc, double> && kahan)
		hipLaunchKernelGGL((k_stage_rows<S, !std::is_same_v<Acc, double>, SWZ>), grid, block, cfg.shmem, s,
		                   static_cast<const S*>(a), static_cast<const Acc*>(b), c, cfg.args);
	else
		hipLaunchKernelGGL((k_stage_rows<S, false, SWZ>), grid, block, cfg.shmem, s, static_cast<const S*>(a),
		                   static_cast<const Acc*>(b), c, cfg.args);
}

template<typename S>
void go_typed(const Config& cfg, const void* a, const void* b, void* c, bool kahan, hipStream_t s)
{
	if(cfg.lean == LEAN_STAGE_ROWS) {
		if constexpr(sizeof(S) != 4) {
			if(cfg.args.swz) go_rows<S, true>(cfg, a, b, c, kahan, s);
			else             go_rows<S, false>(cfg, a, b, c, kahan, s);
		}
	} else if(cfg.lean == LEAN_STAGE_CHUNKS) {
		if constexpr(sizeof(S) == 8) {
			if(cfg.vec == 2) go_chunks<2>(cfg, a, b, c, s);
			else             go_chunks<1>(cfg, a, b, c, s);
		}
	} else if(cfg.vec == 4) {
		if constexpr(sizeof(S) < 8) go<S, 4>(cfg, a, b, c, kahan, s);
	} else if(cfg.vec == 2) {
		go<S, 2>(cfg, a, b, c, kahan, s);
	} else {
		go<S, 1>(cfg, a, b, c, kahan, s);
	}
}
} // namespace

int launch_stage(const Config& cfg, int dtype, const void* a, const void* b, void* c, bool kahan, hipStream_t s)
{
	switch(dtype) {
		case TTVX_F32:  go_typed<float>(cfg, a, b, c, kahan, s); break;
		case TTVX_F64:  go_typed<double>(cfg, a, b, c, kahan, s); break;
		case TTVX_BF16: go_typed<uint16_t>(cfg, a, b, c, kahan, s); break;
		default:        go_typed<uint8_t>(cfg, a, b, c, kahan, s); break;
	}
	hipError_t const e = hipGetLastError();
	return e == hipSuccess ? TTVX_OK : hip_fail(e, "kernel launch");
}

} // namespace ttvx
