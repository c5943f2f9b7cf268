// Sizes of a render call's path pool and results ring (host only).
#pragma once
#include <stdint.h>

#include <algorithm>
#include <stdexcept>
#include <string>

namespace hasty {

constexpr uint32_t kDefaultSlots = 1u << 24;
// Pools the autotuner tries, up to the default (a larger one is faster still,
// see poolPaths, but a pool is kept once it is allocated, 5 GB at 2^24).
constexpr uint32_t kTunedSlots[] = {1u << 20, 1u << 21, 1u << 22, 1u << 23, kDefaultSlots};

// What the jobs of a call add up to.
struct PoolNeed {
  uint64_t paths = 0;  // of all jobs
  uint64_t film = 0;   // pixels of the largest job
  bool late = false;      // some job has both a sky and emissive triangles
  bool textured = false;  // some job has textured media
  void add(uint32_t samples, uint64_t pixels) {
    paths += samples * pixels;
    film = std::max(film, pixels);
  }
};

// Paths in flight (a path that ends makes room for the next): the wanted pool
// (0: the default), but no more than the call needs (at least 2^16).  Larger
// pools spread a bounce's fixed costs (the tail of its longest rays) over more
// rays: 132 ms at 2^22, 129 at 2^23, 125 at 2^24, 122 at 2^25 for 128 samples of
// the 1024x1024 GGX grid.
inline uint32_t poolPaths(const PoolNeed& need, uint32_t wanted) {
  const uint64_t most = wanted ? wanted : kDefaultSlots;
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(most, std::max<uint64_t>(need.paths, 1ull << 16)));
}

// Results ring: the whole call if it is no more than about 2^27 paths
// (finished paths wait in the ring for the oldest one in flight, so a ring
// much longer than a pool x depth never holds a path's start up), else whole
// samples of the largest film; never less than one, which renderJobs needs.
inline uint32_t ringPaths(const PoolNeed& need) {
  const uint64_t P = std::max<uint64_t>(need.film, 1), most = 1ull << 27;
  if (need.paths <= std::max(P, most))
    return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(need.paths, 1), 0x7FFFFFFFull);
  return (uint32_t)std::min<uint64_t>(std::max(P, most / P * P), 0x7FFFFFFFull / P * P);
}

// Paths with room for the guide's training records (192 B each): those of the
// call, but for a film of more than four pools only that many from the oldest
// in flight on (a call trains on about 2^20 paths, or one sample of the film).
inline uint32_t recordPaths(const PoolNeed& need, uint32_t wanted) {
  const uint64_t most = std::max<uint64_t>(4ull * (wanted ? wanted : kDefaultSlots), 1ull << 20);
  return (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(need.paths, most));
}

struct PoolSize {
  uint32_t paths, ring;
};
// Device memory of a pool (the traversal's overflow slices aside): two sets of
// path records (112 B, and 32 B of media texels), hits, shadow rays (60 B, and
// 104 B where they may be late), and 48 B a ring entry.
inline uint64_t poolBytes(PoolSize n, bool late, bool textured) {
  return (uint64_t)n.paths * (2 * (112 + (textured ? 32 : 0)) + 16 + 60 + (late ? 104 : 0)) + (uint64_t)n.ring * 48;
}

// Thrown by a device allocation that the free memory cannot serve.
struct OutOfMemory : std::runtime_error {
  using std::runtime_error::runtime_error;
};

// The largest of `want`, and of its halvings, that `alloc` can serve: the pool
// down to 2^20 paths, the ring down to 2^20 entries or one sample of the largest
// film.  Errors other than OutOfMemory are the caller's.
template <class Alloc>
PoolSize allocHalving(PoolSize want, uint64_t film, Alloc&& alloc) {
  constexpr uint32_t least = 1u << 20;
  const uint32_t leastRing = (uint32_t)std::max<uint64_t>(film, least);
  for (;;) {
    try {
      alloc(want);
      return want;
    } catch (const OutOfMemory&) {
      if (want.paths <= least && want.ring <= leastRing) throw;
      if (want.paths > least) want.paths /= 2;
      if (want.ring > leastRing) want.ring = std::max(leastRing, want.ring / 2);
    }
  }
}

// The pool a scene holds, kept from call to call and grown when a call needs
// more.  After a shortage the smaller pool stays in use, and the wanted size is
// tried again once the memory for it is there; until then a call that wants more
// than the pool asks for the free memory and allocates nothing.
class PoolFit {
 public:
  PoolSize have{0, 0};
  // Makes `have` at least `want`, or what memory allows.  regrow: the buffers
  // have to be allocated again whatever their size.  bytes(size): memory of a
  // pool; freeBytes(): the device's free memory; alloc as for allocHalving,
  // giving back the former pool first.
  template <class Bytes, class Free, class Alloc>
  void fit(PoolSize want, uint64_t film, bool regrow, Bytes&& bytes, Free&& freeBytes, Alloc&& alloc) {
    if (!regrow && want.paths <= have.paths && want.ring <= have.ring) return;
    want.paths = std::max(want.paths, have.paths), want.ring = std::max(want.ring, have.ring);
    if (!regrow && shortAt_ && have.ring >= std::min<uint64_t>(film, want.ring)) {
      const uint64_t room = freeBytes() + bytes(have);
      if (room < bytes(want) || room <= shortAt_) return;
    }
    have = PoolSize{0, 0};
    shortAt_ = 0;
    const PoolSize got = allocHalving(want, film, alloc);
    if (got.paths < want.paths || got.ring < want.ring) shortAt_ = freeBytes() + bytes(got);
    have = got;
  }

 private:
  uint64_t shortAt_ = 0;  // memory for a pool when one last came out smaller (0: none did)
};

}  // namespace hasty
