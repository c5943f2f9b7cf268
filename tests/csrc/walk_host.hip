// Test-only host run of the BVH walk: the renderer's ray preparation, slab
// test, leaf step and triangle test (pt_device.h) over a tree that its builder
// (bvh.cpp) made, one ray at a time, with every index checked before it is
// used.  A GPU wave steps its lanes at nodes or its lanes at triangles; which
// lanes wait changes nothing for a ray, so the sequence here is a lane's.
#include <algorithm>
#include <vector>

#include "../../hastyrenderer_amd/csrc/bvh.h"
#include "../../hastyrenderer_amd/csrc/pt_device.h"

using namespace hdev;

namespace {

enum Status { kOk = 0, kNodeRange = 1, kTriRange = 2, kStackRange = 3, kCycle = 4 };

void testTri(const RayPre& r, const float* tri12, Hit& best) {
  const float4* p = reinterpret_cast<const float4*>(tri12);
  const int32_t id = __builtin_bit_cast(int32_t, p[0].w);
  float t, u, v;
  if (!intersectTri(r, p[0], p[1], p[2], 1e-6f, &t, &u, &v)) return;
  if (best.tri < 0 || t < best.t || (t == best.t && id < best.tri)) best = Hit{t, u, v, id};
}

Status walkRay(const hasty::Bvh4& b, int width, const DevScene& s, const RayPre& r, Hit* out) {
  struct Entry {
    float e;
    uint32_t ref;
  };
  Walk w;
  walkInit(w, r, __builtin_inff(), 0);
  std::vector<Entry> stack;
  const size_t numTris = b.tris.size() / 12, deepest = (size_t)((width - 1) * b.depth + 1);
  // every node and every triangle is reached once at most
  for (size_t left = (size_t)b.numNodes + numTris + 1;; --left) {
    if (left == 0) return kCycle;
    bool pop = false;
    if (w.ref & kLeafFlag) {
      const uint32_t first = w.ref & 0x00FFFFFFu;
      if (first >= numTris) return kTriRange;
      testTri(w.r, b.tris.data() + (size_t)first * 12, w.best);
      pop = leafNext(w.ref);
    } else {
      if (w.ref >= (uint32_t)b.numNodes) return kNodeRange;
      Entry c[8];
      for (int h = 0; h < width / 4; ++h) {
        float e[4];
        uint32_t ref[4];
        testHalf(s, w.r, width == 4 ? w.ref : 2u * w.ref + (uint32_t)h, w.best.t * kCullSlack, e, ref);
        for (int k = 0; k < 4; ++k) c[4 * h + k] = Entry{e[k], ref[k]};
      }
      std::stable_sort(c, c + width, [](const Entry& x, const Entry& y) { return x.e < y.e; });
      for (int k = width - 1; k > 0; --k)
        if (c[k].e != __builtin_inff()) stack.push_back(c[k]);
      if (stack.size() > deepest) return kStackRange;
      pop = c[0].e == __builtin_inff();
      if (!pop) w.ref = c[0].ref;
    }
    while (pop) {
      if (stack.empty()) {
        *out = w.best;
        return kOk;
      }
      const Entry e = stack.back();
      stack.pop_back();
      if (e.e > w.best.t * kCullSlack) continue;
      w.ref = e.ref;
      pop = false;
    }
  }
}

}  // namespace

extern "C" {

// n rays (6 floats each) against the triangles (9 floats each): tri (-1 =
// miss) and t, u, v per ray by a tree of this node width, or by the triangle
// test over all triangles (width 0).  status: see Status.
int tk_walk_host(const float* triPos, uint32_t numTris, int width, const float* rays, uint32_t n, int32_t* tri,
                 float* tuv, int32_t* status) {
  hasty::Bvh4 b = hasty::buildBvh4(triPos, numTris, hasty::BvhBuildOptions(), width ? width : 4);
  DevScene s{};
  s.nodes = reinterpret_cast<const float4*>(b.nodes.data());
  for (uint32_t q = 0; q < n; ++q) {
    const float* p = rays + (size_t)q * 6;
    const RayPre r = prepareRay(v3(p[0], p[1], p[2]), v3(p[3], p[4], p[5]));
    Hit h{__builtin_inff(), 0.0f, 0.0f, -1};
    status[q] = kOk;
    if (width == 0)
      for (uint32_t t = 0; t < numTris; ++t) testTri(r, b.tris.data() + (size_t)t * 12, h);
    else
      status[q] = walkRay(b, width, s, r, &h);
    tri[q] = h.tri;
    tuv[(size_t)q * 3] = h.t, tuv[(size_t)q * 3 + 1] = h.u, tuv[(size_t)q * 3 + 2] = h.v;
  }
  return 0;
}

}  // extern "C"
