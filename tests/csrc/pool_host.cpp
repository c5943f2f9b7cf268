// Test-only host access to the sizing of the path pool and the results ring
// (pool_plan.h).
#include "../../hastyrenderer_amd/csrc/pool_plan.h"

extern "C" {

// Paths and ring entries of a call of n jobs (samples and pixels of each).
void tk_pool_sizes(const uint32_t* samples, const uint64_t* pixels, uint32_t n, uint32_t wanted, uint32_t* out2) {
  hasty::PoolNeed need;
  for (uint32_t i = 0; i < n; ++i) need.add(samples[i], pixels[i]);
  out2[0] = hasty::poolPaths(need, wanted);
  out2[1] = hasty::ringPaths(need);
}

}  // extern "C"
