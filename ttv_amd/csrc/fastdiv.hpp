// Division of 31-bit indices by a number known on the host, as a multiplication and a shift
// (Granlund and Montgomery, Division by invariant integers using multiplication, 1994).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ttvx
{

struct FastDiv {
	uint32_t mul, sh;
};

// 1 <= n < 2^31
inline FastDiv fast_div(int64_t n)
{
	FastDiv f{0, 0};
	while((int64_t{1} << f.sh) < n) ++f.sh;
	f.mul = static_cast<uint32_t>((((uint64_t{1} << f.sh) - static_cast<uint64_t>(n)) << 32) / static_cast<uint64_t>(n) + 1);
	return f;
}

// x / n for x < 2^31
__device__ __forceinline__ uint32_t div_by(uint32_t x, FastDiv f) { return (__umulhi(f.mul, x) + x) >> f.sh; }

} // namespace ttvx
