// Test-only host access to the sizing of the path pool and the results ring
// (pool_plan.h).
#include "../../hastyrenderer_amd/csrc/pool_plan.h"

namespace {
constexpr uint64_t kPathBytes = 300, kRingBytes = 48;
}  // namespace

extern "C" {

// Paths, ring entries and paths with training records of a call of n jobs
// (samples and pixels of each).
void tk_pool_sizes(const uint32_t* samples, const uint64_t* pixels, uint32_t n, uint32_t wanted, uint32_t* out3) {
  hasty::PoolNeed need;
  for (uint32_t i = 0; i < n; ++i) need.add(samples[i], pixels[i]);
  out3[0] = hasty::poolPaths(need, wanted);
  out3[1] = hasty::ringPaths(need);
  out3[2] = hasty::recordPaths(need, wanted);
}

// The pools the autotuner tries; returns how many.
uint32_t tk_tuned_slots(uint32_t* out8) {
  uint32_t n = 0;
  for (uint32_t s : hasty::kTunedSlots) out8[n++] = s;
  return n;
}

// allocHalving on a device with `freeBytes` free, whose allocation number
// `errorAt` (from 1; 0: none) fails with another error.  Returns 0, 1 when out
// of memory, 2 for the other error; out: paths, ring, allocations asked for.
int tk_alloc_halving(uint32_t paths, uint32_t ring, uint64_t film, uint64_t freeBytes, uint32_t errorAt,
                     uint32_t* out3) {
  uint32_t tries = 0;
  int rc = 0;
  out3[0] = out3[1] = 0;
  try {
    const hasty::PoolSize got = hasty::allocHalving({paths, ring}, film, [&](hasty::PoolSize n) {
      if (++tries == errorAt) throw std::runtime_error("unspecified launch failure");
      if (n.paths * kPathBytes + n.ring * kRingBytes > freeBytes) throw hasty::OutOfMemory("out of memory");
    });
    out3[0] = got.paths, out3[1] = got.ring;
  } catch (const hasty::OutOfMemory&) {
    rc = 1;
  } catch (const std::exception&) {
    rc = 2;
  }
  out3[2] = tries;
  return rc;
}

// A scene's pool over n calls on a device of which call k leaves freeBytes[k] to
// the pool: paths and ring held after each, and allocations asked for in it (0
// paths: the call was refused).
void tk_pool_fit(const uint32_t* paths, const uint32_t* ring, const uint64_t* film, const uint64_t* freeBytes,
                 const uint32_t* regrow, uint32_t n, uint32_t* out3) {
  hasty::PoolFit pool;
  auto bytes = [](hasty::PoolSize s) { return hasty::poolBytes(s, false, false); };
  for (uint32_t k = 0; k < n; ++k) {
    uint32_t tries = 0;
    uint64_t held = bytes(pool.have);
    try {
      pool.fit({paths[k], ring[k]}, film[k], regrow[k] != 0, bytes,
               [&] { return freeBytes[k] - std::min(freeBytes[k], held); },
               [&](hasty::PoolSize s) {
                 ++tries;
                 held = 0;
                 if (bytes(s) > freeBytes[k]) throw hasty::OutOfMemory("out of memory");
                 held = bytes(s);
               });
    } catch (const hasty::OutOfMemory&) {
    }
    out3[3 * k] = pool.have.paths, out3[3 * k + 1] = pool.have.ring, out3[3 * k + 2] = tries;
  }
}

}  // extern "C"
