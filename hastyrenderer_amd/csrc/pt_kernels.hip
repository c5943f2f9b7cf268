// Wavefront path tracer for gfx950 with path regeneration:
//   fill, trace, then repeat { shade -> fill -> trace }; accumulate.
// A render call covers n samples of every pixel (n * pixels paths, numbered
// sample-major, pixels in 8x8-tile order).  A pool of path records runs them:
// `shade` takes every path alive one vertex further and packs those that go on
// at the front of the other record set, `fill` appends the next paths of the
// render behind them, and `trace` answers the rays of both kinds: the shadow
// rays `shade` cast and the next extension rays.  A path that ends writes its
// radiance into a results ring.  Every path's random stream is keyed by
// (pixel, sample), so the image does not depend on which record ran which
// path, and `accumulate` adds each pixel's samples in sample order.
//
// The recursion of estimateRadiance (core/src/PathTracing.cpp:21-95) becomes
// one extension ray (BSDF strategy) plus one shadow ray (light strategy) per
// vertex.  `shade` runs a vertex up to both samples and computes the light
// sample's whole term, which is added once its ray is found clear (visibility
// by triangle id, Scene.cpp:558-559 / 572-577); the BSDF strategy's MIS
// weight is applied by the next `shade`, which is where the next hit is
// known.  Radiance is accumulated forward along the path; every decision
// (roulette, lobe choice, rejection, visibility) is made exactly as in the
// recursion.
//
// Records are packed by moving them: a vertex rewrites nearly all of a path's
// state anyway, so writing it to its place in the next bounce's order costs
// nothing extra, and every stage then reads consecutive records with all 64
// lanes live, secondary rays first and the (coherent) camera rays after them.
// Each wave counts its survivors with a ballot, the waves of a block combine
// their counts with a prefix sum in LDS, and the block reserves its ranges of
// paths and shadow rays with one 64-bit atomic.
#include "pt_kernels.h"

#include <algorithm>
#include <stdexcept>
#include <string>
#include <vector>

namespace hasty {
using namespace hdev;

const char* kernelName(int id) {
  switch (id) {
    case kKGenerate: return "pt_generate";
    case kKTrace: return "pt_trace";
    case kKShade: return "pt_shade";
    case kKFinish: return "pt_finish";
    case kKConnect: return "pt_connect_late";
    case kKAccumulate: return "pt_accumulate";
    case kKGraph: return "pt_graph_chunk";
    case kKGuideInfer: return "guide_infer";
    case kKSppmRadii: return "sppm_init_radii";
    case kKSppmCellSize: return "sppm_cell_size";
    case kKSppmPhotons: return "sppm_photons";
    case kKSppmBuild: return "sppm_build";
    case kKSppmCamera: return "sppm_camera";
    case kKSppmGather: return "sppm_gather";
    default: return "pt_misc";
  }
}

namespace {

// Block-wide append of two kinds at once: this lane's index among the paths
// that go on (valid where `go`) and among the shadow rays (where `cast`).
// `counter` holds both counts, paths in the low word.  Must be reached by
// every thread of the block.
__device__ inline void blockAppend2(unsigned long long* counter, bool go, bool cast, uint2* ldsWave,
                                    unsigned long long* ldsBase, uint32_t* idxGo, uint32_t* idxCast) {
  const uint64_t mg = __ballot(go), mc = __ballot(cast);
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint64_t below = (1ull << lane) - 1ull;
  if (lane == 0) ldsWave[wave] = make_uint2((uint32_t)__popcll(mg), (uint32_t)__popcll(mc));
  __syncthreads();
  if (threadIdx.x == 0) {
    uint2 acc = make_uint2(0u, 0u);
    for (uint32_t w = 0; w < (blockDim.x >> 6); ++w) {
      const uint2 c = ldsWave[w];
      ldsWave[w] = acc;
      acc.x += c.x, acc.y += c.y;
    }
    const unsigned long long both = (unsigned long long)acc.x | ((unsigned long long)acc.y << 32);
    *ldsBase = both ? atomicAdd(counter, both) : 0ull;
  }
  __syncthreads();
  const unsigned long long base = *ldsBase;
  const uint2 before = ldsWave[wave];
  *idxGo = (uint32_t)base + before.x + (uint32_t)__popcll(mg & below);
  *idxCast = (uint32_t)(base >> 32) + before.y + (uint32_t)__popcll(mc & below);
  __syncthreads();
}

// Workgroups are dealt round-robin to the 8 XCDs; renumber them so that
// consecutive queue ranges (neighbouring pixels, similar rays) run on the same
// XCD and share its L2.
__device__ inline uint32_t xcdBlock() {
  uint32_t g = gridDim.x, b = blockIdx.x;
  if (g % 8u != 0u) return b;
  return (b % 8u) * (g / 8u) + b / 8u;
}

__device__ inline void waveAddStat(unsigned long long* c, uint32_t v) {
  // lane-sum within the wave, one atomic per wave
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  if ((threadIdx.x & 63u) == 0 && v) atomicAdd(c, (unsigned long long)v);
}

// Entries beyond md.n are never read, so an empty stack is neither loaded
// nor stored.
__device__ inline void loadMedia(const PathSet& ps, uint32_t i, uint32_t flags, const uint32_t* txs, Media& md) {
  md.n = (int)((flags >> 12) & 0xFu);
  md.overflow = (flags >> 16) & 1u;
  md.tx0 = 0u;
  if (md.n == 0) {
#pragma unroll
    for (int k = 0; k < 8; ++k) md.e[k] = 0u;
    return;
  }
  uint4 a = ps.media[(size_t)i * 2], b = ps.media[(size_t)i * 2 + 1];
  md.e[0] = a.x, md.e[1] = a.y, md.e[2] = a.z, md.e[3] = a.w;
  md.e[4] = b.x, md.e[5] = b.y, md.e[6] = b.z, md.e[7] = b.w;
  if (txs) md.tx0 = txs[0];
}
__device__ inline void storeMedia(const PathSet& ps, uint32_t i, const Media& md) {
  ps.media[(size_t)i * 2] = make_uint4(md.e[0], md.e[1], md.e[2], md.e[3]);
  ps.media[(size_t)i * 2 + 1] = make_uint4(md.e[4], md.e[5], md.e[6], md.e[7]);
}
__device__ inline uint32_t packFlags(int depth, int wavelength, const Media& md) {
  return (uint32_t)depth | ((uint32_t)(wavelength + 1) << 8) | ((uint32_t)md.n << 12) |
         (md.overflow ? (1u << 16) : 0u);
}

// ------------------------------------------------------------------ jobs ----
// Job of a global path id: the last job whose pidBase <= pid.
template <bool MULTI>
__device__ inline uint32_t findJob(const JobSet& js, uint32_t pid) {
  if (!MULTI) return 0u;
  uint32_t lo = 0, hi = js.nJobs;
  while (hi - lo > 1u) {
    uint32_t mid = (lo + hi) >> 1;
    if (js.passes[mid].pidBase <= pid) lo = mid;
    else hi = mid;
  }
  return lo;
}
// Batched rendering keeps the job index of a path in flag bits 23-31 (set
// when the path starts) for up to 512 jobs; larger batches search.
constexpr uint32_t kJobShift = 23;
constexpr uint32_t kFlagJobs = 512;
template <bool MULTI>
__device__ inline uint32_t jobOf(const JobSet& js, const uint4& st) {
  if (!MULTI) return 0u;
  return js.nJobs <= kFlagJobs ? st.y >> kJobShift : findJob<true>(js, st.w);
}
__device__ inline uint32_t jobBits(const JobSet& js, uint32_t job) {
  return js.nJobs <= kFlagJobs ? job << kJobShift : 0u;
}
// A copy of *p, which every active lane of the wave passes, read through
// the scalar unit.
template <class T>
__device__ inline T loadUniform(const T* p) {
  static_assert(sizeof(T) % 4 == 0, "word-sized");
  typedef __attribute__((address_space(4))) const uint32_t CWord;
  const CWord* w = (const CWord*)p;
  uint32_t words[sizeof(T) / 4];
#pragma unroll
  for (int i = 0; i < (int)(sizeof(T) / 4); ++i) words[i] = w[i];
  T out;
  __builtin_memcpy(&out, words, sizeof(T));
  return out;
}
// A pointer read from memory is generic to the compiler (flat loads, which
// wait on the LDS counter too); these round trips through the global address
// space give every scene and pass array global loads.
template <class T>
__device__ inline const T* globalPtr(const T* p) {
  return (const T*)(const __attribute__((address_space(1))) T*)p;
}
__device__ inline void makeGlobal(DevScene& s) {
  s.nodes = globalPtr(s.nodes), s.tris = globalPtr(s.tris), s.triPos = globalPtr(s.triPos);
  s.triNrm = globalPtr(s.triNrm), s.triMat = globalPtr(s.triMat), s.triGeom = globalPtr(s.triGeom);
  s.triSmooth = globalPtr(s.triSmooth), s.mats = globalPtr(s.mats), s.lightTris = globalPtr(s.lightTris);
  s.lightCdf = globalPtr(s.lightCdf), s.envRGB = globalPtr(s.envRGB), s.envPdf = globalPtr(s.envPdf);
  s.envCdf = globalPtr(s.envCdf), s.envCdfGuide = globalPtr(s.envCdfGuide);
}
__device__ inline void makeGlobal(PassInfo& pi) {
  pi.tileOrder = globalPtr(pi.tileOrder), pi.rankOf = globalPtr(pi.rankOf), pi.offsets = globalPtr(pi.offsets);
}
// f(scene, pass) of the lane's job.  Batched, the wave's active lanes are
// served one distinct job at a time (normally one: paths are handed out in
// id order), each with its scene and pass in scalar registers.
template <bool MULTI, class F>
__device__ inline void forJob(const JobSet& js, uint32_t job, F&& f) {
  if constexpr (!MULTI) {
    f(js.s, js.pi);
  } else {
    for (;;) {
      const uint32_t j0 = __builtin_amdgcn_readfirstlane(job);
      if (job == j0) {
        DevScene sc = loadUniform(js.scenes + j0);
        PassInfo pi = loadUniform(js.passes + j0);
        makeGlobal(sc);
        makeGlobal(pi);
        f(sc, pi);
        break;
      }
    }
  }
}
// Pixel and sample of a path (global id) of job pi.
__device__ inline void pathPixel(const PassInfo& pi, uint32_t pid, uint32_t* pixel, uint32_t* k) {
  uint32_t local = pid - pi.pidBase;
  uint32_t kk = local / pi.pixels;
  *pixel = pi.tileOrder[local - kk * pi.pixels];
  *k = kk;
}

// ------------------------------------------------------------ path start ----
// Camera ray of path `pid` (Camera.cpp:41-81 with the sample's offset,
// RenderJob.h:53-60) into record i.
__device__ inline void startPath(const DevScene& s, const PathSet& ps, const PassInfo& pi, uint32_t i, uint32_t pid,
                                 uint32_t flags) {
  uint32_t k, pixel;
  pathPixel(pi, pid, &pixel, &k);
  uint32_t x = pixel % s.width, y = pixel / s.width;
  hrng::Stream rng = hrng::make_stream(s.seed, pixel, pi.first + k, hrng::kDomainPath);
  float2 off = pi.offsets[k];
  V3 o, d;
  cameraRay(s, rng, (float)x + off.x, (float)y + off.y, &o, &d);
  // throughput and radiance are not stored here: kShade starts every path
  // from throughput 1 and radiance 0
  ps.rayO[i] = f4(o, 0.0f);
  ps.rayD[i] = f4(d, 0.0f);
  ps.state[i] = make_uint4(rng.counter, flags, 0xFFFFFFFFu, pid);
}

// Occupancy targets (waves per SIMD) of the ray-bound stages: the register
// budget each may use is 512 / waves VGPRs.  0 leaves it to the compiler.
// Shade at 3 waves spills 64 B per lane; at 2 (no spills) the GGX grid takes
// 131 ms, at 4 128 ms, at 3 125 ms.
#ifndef HASTY_TRACE_WAVES
#define HASTY_TRACE_WAVES 8
#endif
#ifndef HASTY_SHADE_WAVES
#define HASTY_SHADE_WAVES 3
#endif
#define HASTY_WAVES_ATTR_(n) __attribute__((amdgpu_waves_per_eu(n)))
#if HASTY_TRACE_WAVES > 0
#define HASTY_TRACE_ATTR HASTY_WAVES_ATTR_(HASTY_TRACE_WAVES)
#else
#define HASTY_TRACE_ATTR
#endif
#if HASTY_SHADE_WAVES > 0
#define HASTY_SHADE_ATTR HASTY_WAVES_ATTR_(HASTY_SHADE_WAVES)
#else
#define HASTY_SHADE_ATTR
#endif

// No path started, nothing alive.
__global__ void kInitRender(uint32_t* c, uint32_t limit) {
  if (threadIdx.x < kNumCounters) c[threadIdx.x] = threadIdx.x == kCntLimit ? limit : 0u;
}
__global__ void kSetLimit(uint32_t* c, uint32_t limit) {
  if (threadIdx.x == 0) c[kCntLimit] = limit;
}

// Paths that start at the end of bounce p: the pool's free places behind the
// paths that went on, up to the ring-space limit.
__device__ inline uint32_t startCount(const PathBuffers& pb, const uint32_t* c) {
  const uint32_t limit = pb.counters[kCntLimit], next = c[kCntNext];
  const uint32_t left = limit > next ? limit - next : 0u;
  return min(pb.capacity - c[kCntA], left);
}
template <bool MULTI>
__global__ void __launch_bounds__(kBlock) kFill(JobSet js, PathBuffers pb, PathSet out, uint32_t p) {
  const uint32_t* c = pb.counters + p * kCntSet;
  const uint32_t n = startCount(pb, c), base = c[kCntA], next = c[kCntNext];
  for (uint32_t r = blockIdx.x * kBlock + threadIdx.x; r < n; r += gridDim.x * kBlock) {
    const uint32_t pid = next + r, j = findJob<MULTI>(js, pid);
    const uint32_t flags = MULTI ? jobBits(js, j) : 0u;
    forJob<MULTI>(js, j, [&](const DevScene& sc, const PassInfo& pi) { startPath(sc, out, pi, base + r, pid, flags); });
  }
}

// ---------------------------------------------------------------- trace ----
// The rays of a bounce in one launch: the shadow rays, then the extension
// rays of the paths alive.  One launch for both kinds because a launch ends
// with a tail of its longest rays (a few hundred dependent node fetches)
// during which the chip is nearly idle; together they have one tail instead
// of two.  Shadow records carry the term to add, so both kinds fit the 64
// registers of 8 waves per SIMD (7 waves: 14% slower on the 1024x1024 GGX
// grid; grids other than the 2048 resident blocks lose 10% and more).
// Bound by the latency of dependent node fetches and by divergence; against
// separate launches over half-filled waves the 128-sample render of that grid
// went from 170 to 125 ms, one sample of a 1283x721 film from 6.1 to 4.1 ms.
// COUNT: add rays, node visits and triangle tests to the statistics (the
// counting is compiled out otherwise).  LATE: some shadow rays look for the
// closest hit (kTargetLate).
// W: node width of the single job's scene (4 or 8), 0 = each job's own.
template <bool MULTI, bool COUNT, int W, bool LATE>
__global__ void __launch_bounds__(kBlock) HASTY_TRACE_ATTR kTrace(JobSet js, PathBuffers pb, PathSet ps, uint32_t p) {
  __shared__ uint2 stack[kStackRows * kBlock];
  const uint32_t gtid = xcdBlock() * blockDim.x + threadIdx.x;
  const uint32_t stride = gridDim.x * blockDim.x;
  uint2* lds = stack + threadIdx.x;
  uint2* ovf = pb.stackOverflow + (size_t)gtid * kStackOvf;
  const uint32_t* c = pb.counters + p * kCntSet;
  const uint32_t nS = c[kCntS];
  uint32_t nodes = 0, tris = 0, rays = 0;
  for (uint32_t k = gtid; k < nS; k += stride) {
    const uint2 ray = pb.sh.q[k];
    const uint32_t i = ray.x, dest = ray.y;
    const float4 o = pb.sh.o[i], d = pb.sh.d[i];
    const int32_t target = __float_as_int(d.w);
    bool clear = false;
    forJob<MULTI>(js, MULTI ? pb.sh.job[i] : 0u, [&](const DevScene& sc, const PassInfo&) {
      if (!LATE || target != kTargetLate) {
        // closest hit == target  <=>  no other triangle is hit before it (or
        // at its t with a smaller index); sky visible  <=>  nothing is hit
        clear = findBlocker<kStackLds, kStackOvf, W>(sc, prepareRay(f4xyz(o), f4xyz(d)), o.w,
                                                     target >= 0 ? target : 0x7FFFFFFF, lds, kBlock, ovf, &nodes,
                                                     &tris) < 0;
      } else {
        const Hit h = traceClosest<kStackLds, kStackOvf, W>(sc, f4xyz(o), f4xyz(d), lds, kBlock, ovf, &nodes, &tris);
        if (h.tri < 0) {
          clear = true;
        } else if (ldg(&sc.mats[ldg(sc.triMat + h.tri)].isLight)) {
          pb.sh.lateHit[i] = make_float4(h.t, h.u, h.v, __int_as_float(h.tri));
          pb.sh.lateQ[atomicAdd(&pb.counters[p * kCntSet + kCntLate], 1u)] = ray;
        }
      }
    });
    if (clear) {
      const float4 t = pb.sh.c[i];
      float4* at = (dest & kDestRing) ? pb.ringL + (dest & ~kDestRing) : ps.L + dest;
      const float4 L = *at;
      *at = f4(f4xyz(L) + f4xyz(t), 0.0f);
    }
    rays++;
  }
  if (COUNT) {
    waveAddStat(&pb.stats[kStatShadowRays], rays);
    waveAddStat(&pb.stats[kStatShadowNodes], nodes);
    waveAddStat(&pb.stats[kStatShadowTris], tris);
    nodes = tris = rays = 0;
  }
  const uint32_t begin = startCount(pb, c), live = c[kCntA] + begin;
  if (gtid == 0) {  // the next bounce's counters (none alive after kFinish)
    uint32_t* d = pb.counters + (p ^ 1u) * kCntSet;
    d[kCntA] = 0u, d[kCntS] = 0u, d[kCntEnded] = 0u, d[kCntLate] = 0u;
    d[kCntLive] = live;
    d[kCntNext] = c[kCntNext] + begin;
  }
  // the threads that got no shadow ray in the last sweep take the first
  // extension rays
  const uint32_t skip = nS % stride;
  for (uint32_t i = gtid >= skip ? gtid - skip : gtid + (stride - skip); i < live; i += stride) {
    const float4 o = ps.rayO[i], d = ps.rayD[i];
    forJob<MULTI>(js, MULTI ? jobOf<MULTI>(js, ps.state[i]) : 0u, [&](const DevScene& sc, const PassInfo&) {
      const Hit h = traceClosest<kStackLds, kStackOvf, W>(sc, f4xyz(o), f4xyz(d), lds, kBlock, ovf, &nodes, &tris);
      pb.hit[i] = make_float4(h.t, h.u, h.v, __int_as_float(h.tri));
    });
    rays++;
  }
  if (COUNT) {
    waveAddStat(&pb.stats[kStatExtRays], rays);
    waveAddStat(&pb.stats[kStatNodes], nodes);
    waveAddStat(&pb.stats[kStatTris], tris);
  }
}

// ---------------------------------------------------------------- shade ----
// Bits 20-21 of the flags: training records of the path (guided rendering).
constexpr uint32_t kRecShift = 20;
// Materials guided by the learned proposal: GGX alpha at least this.
constexpr float kGuideMinAlpha = 0.25f;
// Vertices that sample the guide: rough, non-emitting reflectors.  A
// roughness texture makes the material eligible whatever its texels (the
// one-sample mixture stays unbiased at glossy texels).
__device__ inline bool guideEligible(const DevMaterial& m) {
  return !m.isLight && m.transmission == 0.0f && (m.tex[1] >= 0 || m.alpha >= kGuideMinAlpha);
}
// A path whose throughput has grown past g.maxThroughput samples its BSDF
// alone from then on.  Which technique samples a vertex may depend on the
// path so far without bias; this keeps the guide's 1 / (1 - fraction)
// weights from compounding along long chains of guided vertices.
__device__ inline bool guideThroughputOk(const GuideRun& g, V3 beta) {
  return fmaxf(beta.x, fmaxf(beta.y, beta.z)) <= g.maxThroughput;
}

// A path on its way to a vertex: its ray, what it has gathered, and its media
// stack (txs: the stack's albedo texels, or null).
struct Path {
  V3 o, d;
  float pdf;
  V3 beta, L;
  uint32_t draws, flags;
  int32_t prevTri;
  uint32_t pid;
  Media md;
  uint32_t* txs;
};
__device__ inline Path loadPath(const PathSet& ps, uint32_t i, uint4 st) {
  Path pt;
  const float4 o = ps.rayO[i], d = ps.rayD[i];
  pt.o = f4xyz(o), pt.d = f4xyz(d), pt.pdf = d.w;
  pt.draws = st.x, pt.flags = st.y, pt.prevTri = (int32_t)st.z, pt.pid = st.w;
  // a path's first vertex starts from throughput 1 and radiance 0 (not
  // stored by kFill)
  const bool first = (st.y & 0xFFu) == 0u;
  pt.beta = first ? v3(1.0f, 1.0f, 1.0f) : f4xyz(ps.beta[i]);
  pt.L = first ? v3(0.0f, 0.0f, 0.0f) : f4xyz(ps.L[i]);
  pt.txs = ps.mediaTx ? ps.mediaTx + (size_t)i * kMaxMedia : nullptr;
  loadMedia(ps, i, st.y, pt.txs, pt.md);
  return pt;
}
// What a vertex did: whether the path goes on (with the state left in it),
// and the shadow ray of its light sample with the radiance to add if clear.
struct Vertex {
  bool go, cast;
  V3 so, sd, c;
  float st;  // t of the target triangle (+inf: environment)
  int32_t target;
};

// The term of a light sample that nothing blocks, t2 = thr (fD + fC) cos / pL
// weighted against the BSDF's density pB, times the incident radiance
// (Scene.cpp:560-586, MIS.cpp:32-54); false where it adds nothing.
__device__ inline bool lightTerm(V3 fD, V3 fC, float cosX, V3 thr, float pL, float pB, V3* t2) {
  if (pL == 0.0f) return false;
  const float mm = cosX / pL;
  const V3 tD = fD * mm, tC = fC * mm;
  *t2 = mul(thr, tD + tC);
  if (isZero(*t2)) return false;
  float sum = 0.0f;
  sum += powci<2>(pL);
  sum += powci<2>(pB);
  const float w = powci<2>(pL) / sum;
  *t2 = *t2 * w;
  return true;
}
// Radiance of light triangle `tri` (point hx, normal hn) along -sd, through
// the media of the light ray.
__device__ inline V3 lightRadiance(const DevScene& s, int32_t tri, V3 hx, V3 hn, V3 so, V3 sd, V3 Tc) {
  const DevMaterial lm = ldgStruct(s.mats + ldg(s.triMat + tri));
  const V3 Tb = beersLaw(Tc, norm(hx - so));
  const V3 Le = dot(hn, -sd) <= 0.0f ? v3(0.0f, 0.0f, 0.0f)
                                      : v3(lm.emission[0], lm.emission[1], lm.emission[2]) * (float)kInvPi;
  return mul(Tb, Le);
}

// One vertex of path i, whose ray met h4.
template <bool GUIDED>
__device__ inline void shadeVertex(const DevScene& s, const PassInfo& pi, const GuideRun& g, const PathBuffers& pb,
                                   uint32_t i, Path& pt, float4 h4, Vertex& vx) {
  const bool twoStrategies = s.hasLight && s.useMIS;
  const uint32_t flags = pt.flags;
  int depth = (int)(flags & 0xFFu);
  int wavelength = (int)((flags >> 8) & 0x3u) - 1;
  // per-entry albedo texels of the media stack (albedo-textured scenes)
  uint32_t* txs = s.texturedMedia ? pt.txs : nullptr;
  Media& md = pt.md;
  const V3 ro = pt.o, rd = pt.d;
  const int32_t tri = __float_as_int(h4.w);
  const V3 b0 = pt.beta;
  V3 beta = b0;
  V3& L = pt.L;
  vx.go = vx.cast = false;
  uint32_t nrec = GUIDED ? (flags >> kRecShift) & 3u : 0u;
  if (GUIDED && depth > 0 && nrec > 0 && ((flags >> (kRecShift + 2)) & 1u)) {
    // radiance before the continuation of the last recorded vertex
    g.rec[(size_t)(pt.pid % g.recPaths) * 12 + 6 * (nrec - 1) + 5] = f4(L, 0.0f);
  }
  hrng::Stream rng;
  {
    uint32_t k, pixel;
    pathPixel(pi, pt.pid, &pixel, &k);
    rng = hrng::make_stream(s.seed, pixel, pi.first + k, hrng::kDomainPath);
    rng.counter = pt.draws;
  }
  const EnvUV sky = tri < 0 && s.hasEnv ? envUV(rd) : EnvUV{0.0f, 0.0f, 0.0f};
  const float pSurf = !s.hasEnv ? 1.0f : (s.hasSurfaceLight ? 0.5f : 0.0f);
  // The BSDF sample that produced this ray: self-intersection, then MIS.
  if (depth > 0) {
    if (tri == pt.prevTri) return;
    float pB = pt.pdf;
    float sum = 0.0f;
    if (twoStrategies) {
      float pL;
      if (tri >= 0) {
        V3 hx, hn;
        hitPointNormal(s, tri, h4.y, h4.z, &hx, &hn);
        pL = lightDensity(s, ro, rd, tri, hx, hn);
      } else {
        pL = s.hasEnv ? (1.0f - pSurf) * envPdf(s, sky) : 0.0f;
      }
      sum += powci<2>(pL);
    }
    sum += powci<2>(pB);
    float w = powci<2>(pB) / sum;
    beta = beta * w;
  }
  const uint32_t ri = depth == 0 ? pt.pid % pb.ringPaths : 0u;
  if (tri < 0) {
    V3 T = beersLaw(mediaTransmittance(s, md), 1e6f);
    V3 Lc = mul(T, s.hasEnv ? envLookup(s, sky.u, sky.v) : v3(s.bg[0], s.bg[1], s.bg[2]));
    L = L + mul(beta, Lc);
    if (depth == 0) {
      pb.ringN[ri] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      pb.ringA[ri] = f4(Lc, 0.0f);
    }
    return;
  }
  Interaction it = makeInteraction(s, tri, h4.y, h4.z);
  DevMaterial m = ldgStruct(s.mats + it.mat);
  // guided vertex: rough reflection (no delta lobe, and not so glossy
  // that broad vMF lobes could only waste samples); decided on the
  // material before its textures and on the stored throughput
  // before this vertex's MIS weight, exactly as kGuideInfer decides
  // it, so that every guided vertex has its mixture table
  const bool guided = GUIDED && guideEligible(m) && (uint32_t)depth < g.maxDepth &&
                      (depth == 0 || guideThroughputOk(g, b0));
  if (depth == 0) pb.ringN[ri] = f4(it.ns, 0.0f);  // the default shading normal
  uint32_t texel = 0u;
  if (m.textured) applyTextures(s, m, it, 1.0f - h4.y - h4.z, h4.y, h4.z, &texel);
  if (depth == 0) pb.ringA[ri] = make_float4(m.albedo[0], m.albedo[1], m.albedo[2], 0.0f);
  V3 Tb = beersLaw(mediaTransmittance(s, md), norm(it.x - ro));
  V3 wo = -rd;
  if (m.isLight) {
    V3 Le = dot(it.ng, wo) <= 0.0f ? v3(0.0f, 0.0f, 0.0f)
                                    : v3(m.emission[0], m.emission[1], m.emission[2]) * (float)kInvPi;
    L = L + mul(beta, mul(Tb, Le));
    return;
  }
  float rrQ = depth >= s.rrStart ? s.rrQ : 0.0f;
  if (rng.uniform01f() < rrQ) return;
  V3 thr = Tb / (1.0f - rrQ);
  if (depth + 1 >= s.maxDepth) return;  // every deeper estimate is zero
  // the vertex's mixture table, written by kGuideInfer
  const float4* gm = GUIDED ? g.raw + (size_t)i * 10 : nullptr;
  // kGuideInfer wrote the learned probability of guided vertices
  const float gf = GUIDED ? (g.sel && guided ? g.sel[i] : g.fraction) : 0.0f;
  if (twoStrategies) {
    // ---- light strategy (MIS.cpp:32-54, Scene.cpp:538-586)
    float xi = rng.uniform01f();
    V3 so, sd;
    int32_t target = kTargetSky;
    float tT = __builtin_inff();
    V3 hx = v3(0.0f, 0.0f, 0.0f), hn = v3(0.0f, 0.0f, 0.0f);  // the target's point and normal
    bool lit = true;  // the sampled light point emits toward so and its ray meets it
    if (xi < pSurf) {
      uint32_t li = lightCdfSearch(s, rng.canonical_double());
      target = (int32_t)ldg(s.lightTris + li);
      const float* p = s.triPos + (size_t)target * 9;
      V3 p0 = load3g(p), p1 = load3g(p + 3), p2 = load3g(p + 6);
      float su = rng.uniform01f();
      float tt = hm::fsqrt(rng.uniform01f());
      float b1 = 1.0f - tt;
      float b3 = tt * su;
      float b2 = fmaxf(0.0f, 1.0f - b1 - b3);
      V3 x2 = p0 * b1 + p1 * b2 + p2 * b3;
      V3 diff = x2 - it.x;
      so = offsetOrigin(it, dot(it.ng, diff) >= 0.0f);
      sd = normalize(x2 - so);
      hn = normalize(cross(p1 - p0, p2 - p0));
      lit = !(dot(hn, -sd) <= 0.0f);  // a one-sided light seen from behind gives zero
      if (lit) {
        float uT, vT;
        lit = intersectTri(prepareRay(so, sd), f4(p0, 0.0f), f4(p1, 0.0f), f4(p2, 0.0f), 1e-6f, &tT, &uT, &vT);
        hx = p0 * (1.0f - uT - vT) + p1 * uT + p2 * vT;
      }
    } else {
      float dens;
      sd = envSample(s, rng, &dens);
      so = offsetOrigin(it, dot(it.ng, sd) >= 0.0f);
    }
    BsdfEval ev = bsdfEvaluate(m, it, wo, sd);
    // A light sample the BSDF gives nothing (e.g. below the surface), that
    // sees a light from behind or whose term is zero adds exactly zero
    // whatever its shadow ray meets, so no ray is cast; about a quarter of
    // the samples on the GGX grid.
    if (lit && !isZero(ev.fD + ev.fC)) {
      float pB = bsdfPdf(m, it, wo, sd, mediaOutsideIOR(s, md, it, wo, wavelength));
      if (GUIDED && guided) pB = gf * guide::mixturePdfTable(gm, sd) + (1.0f - gf) * pB;
      const V3 Tc = mediaTransmittanceAfter(s, md, it, wo, sd, texel, txs);
      const float cosX = __builtin_fabsf(dot(sd, it.ng));
      V3 t2, Lt = v3(0.0f, 0.0f, 0.0f);  // the term if nothing is in the way
      if (target >= 0) {
        if (target != tri && lightTerm(ev.fD, ev.fC, cosX, thr, lightDensity(s, so, sd, target, hx, hn), pB, &t2)) {
          Lt = mul(beta, mul(lightRadiance(s, target, hx, hn, so, sd, Tc), t2));
          vx.cast = true;
        }
      } else {
        const EnvUV e = envUV(sd);
        if (lightTerm(ev.fD, ev.fC, cosX, thr, (1.0f - pSurf) * envPdf(s, e), pB, &t2)) {
          Lt = mul(beta, mul(mul(beersLaw(Tc, 1e6f), envLookup(s, e.u, e.v)), t2));
          vx.cast = true;
        }
        if (pSurf > 0.0f) {  // the ray may meet a light instead (kConnectLate)
          vx.cast = true;
          target = kTargetLate;
          pb.sh.lateFD[i] = f4(ev.fD, cosX);
          pb.sh.lateFC[i] = f4(ev.fC, __int_as_float(tri));
          pb.sh.lateThr[i] = f4(thr, pB);
          pb.sh.lateBeta[i] = f4(beta, 0.0f);
          pb.sh.lateT[i] = f4(Tc, 0.0f);
        }
      }
      vx.so = so, vx.sd = sd, vx.c = Lt;
      vx.st = tT, vx.target = target;
    }
  }
  // ---- BSDF strategy (MIS.cpp:6-26, Scene.cpp:328-338)
  float sampleProbability = 1.0f;
  if (wavelength == -1 && m.varyIOR) {
    float p0 = 1.0f / 3.0f;
    float xi = rng.uniform01f();
    if (xi < p0) wavelength = 0;
    else if (xi < p0 + p0) wavelength = 1;
    else wavelength = 2;
    sampleProbability = p0;
  }
  float outsideIOR = mediaOutsideIOR(s, md, it, wo, wavelength);
  BsdfSample bs;
  float pBsdf = 0.0f;  // the BSDF's density of the direction (training records)
  if (GUIDED && guided) {
    // one-sample MIS of guide and BSDF: p = f pG + (1 - f) pB
    if (rng.uniform01f() < gf) {
      float x0 = rng.uniform01f(), x1 = rng.uniform01f(), x2 = rng.uniform01f();
      bs.dir = guide::mixtureSampleTable(gm, x0, x1, x2);
      bs.outside = dot(it.ng, wo) >= 0.0f;
      BsdfEval ev = bsdfEvaluate(m, it, wo, bs.dir);
      float pB = bsdfPdf(m, it, wo, bs.dir, outsideIOR);
      pBsdf = pB;
      bs.pdf = gf * guide::mixturePdfTable(gm, bs.dir) + (1.0f - gf) * pB;
      float mm = bs.pdf > 0.0f ? __builtin_fabsf(dot(bs.dir, it.ng)) / bs.pdf : 0.0f;
      bs.tD = ev.fD * mm;
      bs.tC = ev.fC * mm;
      if (!(bs.pdf > 0.0f)) bs.pdf = 0.0f;
    } else {
      bs = bsdfSample(m, rng, it, wo, wavelength, outsideIOR, false, 3);
      pBsdf = bs.pdf;
      if (bs.pdf != 0.0f) {
        float pMix = gf * guide::mixturePdfTable(gm, bs.dir) + (1.0f - gf) * bs.pdf;
        float sc = bs.pdf / pMix;
        bs.tD = bs.tD * sc;
        bs.tC = bs.tC * sc;
        bs.pdf = pMix;
      }
    }
  } else {
    bs = bsdfSample(m, rng, it, wo, wavelength, outsideIOR, false, 3);
  }
  bs.tD = bs.tD / sampleProbability;
  bs.tC = bs.tC / sampleProbability;
  if (bs.pdf == 0.0f) return;
  V3 t2 = mul(thr, bs.tD + bs.tC);
  if (isZero(t2)) return;
  mediaUpdate(md, it, wo, bs.dir, texel, txs);
  vx.go = true;
  pt.o = offsetOrigin(it, bs.outside);
  pt.d = bs.dir;
  pt.pdf = bs.pdf;
  pt.beta = mul(beta, t2);
  pt.draws = rng.counter;
  pt.prevTri = tri;
  uint32_t recBits = 0u;
  if (GUIDED) {
    if (guided && nrec < 2u && g.sampleCap > 0u) {  // records only when training
      float4* rr = g.rec + (size_t)(pt.pid % g.recPaths) * 12 + 6 * nrec;
      V3 nf = dot(it.ng, wo) >= 0.0f ? it.ng : -it.ng;
      rr[0] = f4(it.x, 0.0f);
      rr[1] = f4(nf, 0.0f);
      rr[2] = f4(wo, bs.pdf);
      rr[3] = f4(bs.dir, pBsdf);
      rr[4] = f4(beta, 0.0f);
      nrec += 1u;
      recBits = (nrec << kRecShift) | (1u << (kRecShift + 2));
    } else {
      recBits = nrec << kRecShift;
    }
  }
  pt.flags = packFlags(depth + 1, wavelength, md) | recBits | (flags & ~((1u << kJobShift) - 1u));
}

// The last paths of a render: when none is left to start and so few are alive
// that launches would only run their longest rays one after another, kFinish
// runs every path to its end by itself (and the bounce kernels, which test the
// same counters, find nothing to do).
__device__ inline bool finishing(const JobSet& js, const uint32_t* c) {
  return js.finishPaths > 0u && c[kCntNext] >= js.paths && c[kCntLive] <= js.finishPaths;
}

// Bounce p: every path alive in `in` one vertex further, those that go on
// packed into `out`, light samples into the shadow rays, and the radiance of
// those that end into the results ring (to which a last light sample is still
// added by kTrace).  With `count`, ended paths whose media stack overflowed
// are counted.
template <bool MULTI, bool GUIDED>
__global__ void __launch_bounds__(kBlock) HASTY_SHADE_ATTR kShade(JobSet js, PathBuffers pb, PathSet in, PathSet out,
                                                                 uint32_t p, uint32_t count) {
  __shared__ uint2 ldsWave[kBlock / 64];
  __shared__ unsigned long long ldsBase;
  uint32_t* c = pb.counters + p * kCntSet;
  if (finishing(js, c)) return;
  const uint32_t n = c[kCntLive];
  uint32_t overflowed = 0;
  for (uint32_t base = blockIdx.x * kBlock; base < n; base += gridDim.x * kBlock) {
    const uint32_t i = base + threadIdx.x;
    Vertex vx;
    vx.go = vx.cast = false;
    Path pt;
    uint32_t stFlags = 0u;
    if (i < n) {
      const uint4 st = in.state[i];
      stFlags = st.y;
      const uint32_t job = jobOf<MULTI>(js, st);
      pt = loadPath(in, i, st);
      const float4 h4 = pb.hit[i];
      forJob<MULTI>(js, job, [&](const DevScene& s, const PassInfo& pi) {
        shadeVertex<GUIDED>(s, pi, js.g, pb, i, pt, h4, vx);
      });
      if (vx.cast) {
        pb.sh.o[i] = f4(vx.so, vx.st);
        pb.sh.d[i] = f4(vx.sd, __int_as_float(vx.target));
        pb.sh.c[i] = f4(vx.c, 0.0f);
        if (MULTI) pb.sh.job[i] = job;
      }
    }
    uint32_t idxN, idxS;
    blockAppend2((unsigned long long*)(c + kCntA), vx.go, vx.cast, ldsWave, &ldsBase, &idxN, &idxS);
    uint32_t dest = idxN;
    if (vx.go) {
      out.rayO[idxN] = f4(pt.o, 0.0f);
      out.rayD[idxN] = f4(pt.d, pt.pdf);
      out.beta[idxN] = f4(pt.beta, 0.0f);
      out.L[idxN] = f4(pt.L, 0.0f);
      out.state[idxN] = make_uint4(pt.draws, pt.flags, (uint32_t)pt.prevTri, pt.pid);
      if (pt.md.n > 0) {
        storeMedia(out, idxN, pt.md);
        if (in.mediaTx)
          for (int k = 0; k < pt.md.n; ++k)
            out.mediaTx[(size_t)idxN * kMaxMedia + k] = in.mediaTx[(size_t)i * kMaxMedia + k];
      }
    } else if (i < n) {  // the path ends here (but for its shadow ray, if any)
      const uint32_t ri = pt.pid % pb.ringPaths;
      dest = ri | kDestRing;
      pb.ringL[ri] = f4(pt.L, 0.0f);
      overflowed += (stFlags >> 16) & 1u;
      const uint32_t nrec = GUIDED ? (stFlags >> kRecShift) & 3u : 0u;
      if (GUIDED && nrec > 0u) pb.ended[atomicAdd(c + kCntEnded, 1u)] = make_uint2(pt.pid, nrec);
    }
    if (vx.cast) pb.sh.q[idxS] = make_uint2(i, dest);
  }
  if (count) waveAddStat(&pb.stats[kStatMediaOverflow], overflowed);
}

// --------------------------------------------------------------- finish ----
// Every path alive at bounce p to its end, one lane per path: the vertices,
// shadow rays and extension rays of kShade and kTrace in the same order (so
// the same bits), with the path in registers.  Few paths are alive, so a wave
// takes as few of them as keeps every wave of the grid busy: its steps then
// wait for the longest ray of 8 to 64 lanes instead of all the paths'.
// Bound by the chain of one path's vertices (instruction and fetch latency).
// One sample of a 1283x721 GGX grid: 12 further bounces of 290 us became one
// launch of 0.9 ms, the render 4.07 -> 2.7 ms; 2^18 paths measured best of
// 2^15 .. 2^19 (2.88, 2.79, 2.76, 2.68, 2.70 ms; caustic box at 720x405: 9.69,
// 9.54, 9.30, 9.31, 9.66).
constexpr uint32_t kFinishBlocks = 768;  // 3 waves per SIMD
#ifndef HASTY_FINISH_PATHS
#define HASTY_FINISH_PATHS (1u << 18)
#endif
constexpr uint32_t kFinishPaths = HASTY_FINISH_PATHS;
template <bool MULTI, bool COUNT, int W>
__global__ void __launch_bounds__(kBlock) HASTY_SHADE_ATTR kFinish(JobSet js, PathBuffers pb, PathSet ps, uint32_t p) {
  __shared__ uint2 stack[kStackRows * kBlock];
  const uint32_t* c = pb.counters + p * kCntSet;
  if (!finishing(js, c)) return;
  const uint32_t n = c[kCntLive];
  const uint32_t lane = threadIdx.x & 63u, wave = (blockIdx.x * kBlock + threadIdx.x) >> 6;
  const uint32_t waves = gridDim.x * (kBlock / 64);
  uint32_t per = 64u;  // paths per wave
  while (per > 8u && n <= waves * (per / 2u)) per /= 2u;
  uint2* lds = stack + threadIdx.x;
  uint2* ovf = pb.stackOverflow + (size_t)(blockIdx.x * kBlock + threadIdx.x) * kStackOvf;
  uint32_t rays = 0, nodes = 0, tris = 0, shRays = 0, shNodes = 0, shTris = 0, overflowed = 0;
  for (uint32_t g = wave; g * per < n; g += waves) {
    const uint32_t i = g * per + lane;
    if (lane >= per || i >= n) continue;
    const uint4 st = ps.state[i];
    const uint32_t job = jobOf<MULTI>(js, st);
    Path pt = loadPath(ps, i, st);
    float4 h4 = pb.hit[i];
    Vertex vx;
    do {
      const uint32_t stFlags = pt.flags;
      forJob<MULTI>(js, job, [&](const DevScene& s, const PassInfo& pi) {
        shadeVertex<false>(s, pi, js.g, pb, i, pt, h4, vx);
        if (vx.cast) {
          const bool clear = findBlocker<kStackLds, kStackOvf, W>(s, prepareRay(vx.so, vx.sd), vx.st,
                                                                  vx.target >= 0 ? vx.target : 0x7FFFFFFF, lds, kBlock,
                                                                  ovf, &shNodes, &shTris) < 0;
          if (clear) pt.L = pt.L + vx.c;
          shRays++;
        }
        if (vx.go) {
          const Hit h = traceClosest<kStackLds, kStackOvf, W>(s, pt.o, pt.d, lds, kBlock, ovf, &nodes, &tris);
          h4 = make_float4(h.t, h.u, h.v, __int_as_float(h.tri));
          rays++;
        }
      });
      if (!vx.go) overflowed += (stFlags >> 16) & 1u;
    } while (vx.go);
    pb.ringL[pt.pid % pb.ringPaths] = f4(pt.L, 0.0f);
  }
  if (COUNT) {
    waveAddStat(&pb.stats[kStatExtRays], rays);
    waveAddStat(&pb.stats[kStatNodes], nodes);
    waveAddStat(&pb.stats[kStatTris], tris);
    waveAddStat(&pb.stats[kStatShadowRays], shRays);
    waveAddStat(&pb.stats[kStatShadowNodes], shNodes);
    waveAddStat(&pb.stats[kStatShadowTris], shTris);
    waveAddStat(&pb.stats[kStatMediaOverflow], overflowed);
  }
}

// -------------------------------------------------------------- connect ----
// Environment samples of bounce p whose ray met a light (scenes with both
// kinds of lights): the light strategy's term for the light (Scene.cpp:560-586).
template <bool MULTI>
__global__ void __launch_bounds__(kBlock) kConnectLate(JobSet js, PathBuffers pb, PathSet ps, uint32_t p) {
  const uint32_t n = pb.counters[p * kCntSet + kCntLate];
  for (uint32_t q = blockIdx.x * kBlock + threadIdx.x; q < n; q += gridDim.x * kBlock) {
    const uint32_t i = pb.sh.lateQ[q].x, dest = pb.sh.lateQ[q].y;
    const uint32_t job = MULTI ? pb.sh.job[i] : 0u;
    forJob<MULTI>(js, job, [&](const DevScene& s, const PassInfo&) {
      const V3 so = f4xyz(pb.sh.o[i]), sd = f4xyz(pb.sh.d[i]);
      const float4 h = pb.sh.lateHit[i];
      const int32_t tri = __float_as_int(h.w);
      V3 hx, hn;
      hitPointNormal(s, tri, h.y, h.z, &hx, &hn);
      const float4 fd = pb.sh.lateFD[i], fc = pb.sh.lateFC[i], thr = pb.sh.lateThr[i];
      V3 t2;
      if (tri == __float_as_int(fc.w) ||
          !lightTerm(f4xyz(fd), f4xyz(fc), fd.w, f4xyz(thr), lightDensity(s, so, sd, tri, hx, hn), thr.w, &t2))
        return;
      const V3 Li = lightRadiance(s, tri, hx, hn, so, sd, f4xyz(pb.sh.lateT[i]));
      float4* L = (dest & kDestRing) ? pb.ringL + (dest & ~kDestRing) : ps.L + dest;
      *L = f4(f4xyz(*L) + mul(f4xyz(pb.sh.lateBeta[i]), mul(Li, t2)), 0.0f);
    });
  }
}

// -------------------------------------------------------------- harvest ----
// Training samples of the paths that ended at bounce p: weight = luminance
// of the radiance the continuation brought, over the throughput before the
// sample.
__global__ void __launch_bounds__(kBlock) kHarvest(GuideRun g, PathBuffers pb, uint32_t p) {
  const uint32_t n = pb.counters[p * kCntSet + kCntEnded];
  for (uint32_t q = blockIdx.x * kBlock + threadIdx.x; q < n; q += gridDim.x * kBlock) {
    const uint2 e = pb.ended[q];
    const float4 Lf = pb.ringL[e.x % pb.ringPaths];
    for (uint32_t r = 0; r < e.y; ++r) {
      const float4* rr = g.rec + (size_t)(e.x % g.recPaths) * 12 + 6 * r;
      float4 b = rr[4], ls = rr[5];
      float cx = b.x > 0.0f ? (Lf.x - ls.x) / b.x : 0.0f;
      float cy = b.y > 0.0f ? (Lf.y - ls.y) / b.y : 0.0f;
      float cz = b.z > 0.0f ? (Lf.z - ls.z) / b.z : 0.0f;
      float F = 0.2126f * cx + 0.7152f * cy + 0.0722f * cz;
      if (F > 0.0f && F < 3.0e38f) {
        uint32_t k = atomicAdd(g.sampleCount, 1u);
        if (k < g.sampleCap) {
          float4 x = rr[0];
          g.samples[4 * (size_t)k] = make_float4(x.x, x.y, x.z, F);
          g.samples[4 * (size_t)k + 1] = rr[1];
          g.samples[4 * (size_t)k + 2] = rr[2];
          g.samples[4 * (size_t)k + 3] = rr[3];
        }
      }
    }
  }
}

// ----------------------------------------------------------- accumulate ----
// Samples [k0, k1) of job pi, from the ring, added pixel by pixel in sample
// order; NaN samples are skipped (PathTracing.cpp:132-135).
__global__ void __launch_bounds__(kBlock) kAccumulate(PathBuffers pb, PassInfo pi, uint32_t k0, uint32_t k1,
                                                      float* color, float* normal, float* albedo) {
  uint32_t P = pi.pixels;
  uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < P; p += stride) {
    float c0 = color[p * 3], c1 = color[p * 3 + 1], c2 = color[p * 3 + 2];
    float n0 = normal[p * 3], n1 = normal[p * 3 + 1], n2 = normal[p * 3 + 2];
    float a0 = albedo[p * 3], a1 = albedo[p * 3 + 1], a2 = albedo[p * 3 + 2];
    uint32_t pid0 = pi.pidBase + pi.rankOf[p];
    for (uint32_t k = k0; k < k1; ++k) {
      uint32_t ri = (pid0 + k * P) % pb.ringPaths;
      float4 L = pb.ringL[ri];
      if (L.x != L.x || L.y != L.y || L.z != L.z) continue;
      float4 an = pb.ringN[ri], aa = pb.ringA[ri];
      c0 += L.x, c1 += L.y, c2 += L.z;
      n0 += an.x, n1 += an.y, n2 += an.z;
      a0 += aa.x, a1 += aa.y, a2 += aa.z;
    }
    color[p * 3] = c0, color[p * 3 + 1] = c1, color[p * 3 + 2] = c2;
    normal[p * 3] = n0, normal[p * 3 + 1] = n1, normal[p * 3 + 2] = n2;
    albedo[p * 3] = a0, albedo[p * 3 + 1] = a1, albedo[p * 3 + 2] = a2;
  }
}

// ------------------------------------------------------------ guide infer ----
// Mixture tables of the paths alive that hit a guided surface: inputs
// are the hit point, the geometric normal facing wo, and wo.  A wave takes 64
// paths, one per lane, for the gathers (hit, material, triangle, ray), then
// runs the network on its four 16-path tiles in turn; the tile's lanes fetch
// their path's inputs from the gathering lane by shuffles.  Blocks of 512
// threads, three per CU (the LDS copy of the network is 41 KiB per block).
#ifndef HASTY_GUIDE_INFER_WAVES
#define HASTY_GUIDE_INFER_WAVES 6
#endif
constexpr uint32_t kGuideInferThreads = 512, kGuideInferBlocks = 256 * 3;
__global__ void __launch_bounds__(kGuideInferThreads) HASTY_WAVES_ATTR_(HASTY_GUIDE_INFER_WAVES)
    kGuideInfer(JobSet js, PathBuffers pb, PathSet ps, uint32_t p) {
  __shared__ guide::LdsNet ldsNet;
  guide::stageNet(js.g.net, &ldsNet, true);
  const DevScene& s = js.s;
  const uint32_t n = pb.counters[p * kCntSet + kCntLive];
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t waves = (gridDim.x * blockDim.x) >> 6;
  for (uint32_t g = wave; g * 64 < n; g += waves) {
    const uint32_t e = g * 64 + lane;
    bool want = false;
    V3 x = v3(0.0f, 0.0f, 0.0f), ng = v3(0.0f, 0.0f, 1.0f), wo = v3(0.0f, 0.0f, 1.0f);
    if (e < n) {
      const float4 h4 = pb.hit[e];
      const int32_t tri = __float_as_int(h4.w);
      if (tri >= 0) {
        // only hits on guided materials read the outputs
        const DevMaterial m = ldgStruct(s.mats + ldg(s.triMat + tri));
        const uint32_t depth = ps.state[e].y & 0xFFu;
        want = guideEligible(m) && depth < js.g.maxDepth;
        if (want && depth > 0) want = guideThroughputOk(js.g, f4xyz(ps.beta[e]));
        if (want) {
          hitPointNormal(s, tri, h4.y, h4.z, &x, &ng);
          wo = -f4xyz(ps.rayD[e]);
          if (dot(ng, wo) < 0.0f) ng = -ng;
          x = guide::normPos(js.g.net, x);
        }
      }
    }
    const unsigned long long wantMask = __ballot(want);
    for (int j = 0; j < 4; ++j) {
      // a tile whose 16 paths have no guided hit skips the network (the test
      // is uniform over the wave)
      if (((wantMask >> (16 * j)) & 0xFFFFull) == 0ull) continue;
      const int src = 16 * j + r;
      const V3 xq = v3(__shfl(x.x, src), __shfl(x.y, src), __shfl(x.z, src));
      const V3 nq = v3(__shfl(ng.x, src), __shfl(ng.y, src), __shfl(ng.z, src));
      const V3 wq = v3(__shfl(wo.x, src), __shfl(wo.y, src), __shfl(wo.z, src));
      const uint32_t sq = g * 64 + src;
      // lane group q holds lobes 2q and 2q + 1 of the path's mixture
      float r10[10], w0, w1, logit;
      guide::tileOutputs(&ldsNet, xq, nq, wq, r10, &w0, &w1, &logit);
      if ((wantMask >> src) & 1ull) {
        float4* out = js.g.raw + (size_t)sq * 10;
        out[2 * q] = guide::lobeEntry(r10, w0);
        out[2 * q + 1] = guide::lobeEntry(r10 + 5, w1);
        reinterpret_cast<float2*>(out + guide::kLobes)[q] = make_float2(w0, w1);
        if (js.g.sel && q == 0) js.g.sel[sq] = guide::selectionOf(js.g.net, logit);
      }
    }
  }
}

// Batched closest-hit queries, grid-stride over the rays.  Bound, as kTrace,
// by dependent node fetches: the time falls with the waves in flight, so the
// registers are held to 8 waves per SIMD and the grid fills the chip (the
// caller's overflow slices allowing).  `slice`: overflow entries per thread.
// 4.2M incoherent rays of the GGX grid: 4.54 ms with 256 blocks (one wave per
// SIMD), 1.14 ms with 2048.
template <int W>
__global__ void __launch_bounds__(kBlock) HASTY_TRACE_ATTR kTraceRays(DevScene s, const float* rays, uint32_t n,
                                                                     int32_t* tri, float* tuv, uint2* overflow,
                                                                     uint32_t slice) {
  __shared__ uint2 stack[kStackRows * kBlock];
  uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t stride = gridDim.x * blockDim.x;
  uint2* ovf = overflow + (size_t)gtid * slice;
  for (uint32_t q = gtid; q < n; q += stride) {
    const float* r = rays + (size_t)q * 6;
    Hit h = traceClosest<kStackLds, kStackOvf, W>(s, v3(r[0], r[1], r[2]), v3(r[3], r[4], r[5]), stack + threadIdx.x,
                                                  kBlock, ovf, nullptr, nullptr);
    tri[q] = h.tri;
    tuv[(size_t)q * 3] = h.t;
    tuv[(size_t)q * 3 + 1] = h.u;
    tuv[(size_t)q * 3 + 2] = h.v;
  }
}

// The same with closest-hit records (HitRecord).
template <int W>
__global__ void __launch_bounds__(kBlock) HASTY_TRACE_ATTR kTraceHits(DevScene s, const float* rays, uint32_t n,
                                                                     HitRecord* hits, uint2* overflow,
                                                                     uint32_t slice) {
  __shared__ uint2 stack[kStackRows * kBlock];
  uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t stride = gridDim.x * blockDim.x;
  uint2* ovf = overflow + (size_t)gtid * slice;
  for (uint32_t q = gtid; q < n; q += stride) {
    const float* r = rays + (size_t)q * 6;
    Hit h = traceClosest<kStackLds, kStackOvf, W>(s, v3(r[0], r[1], r[2]), v3(r[3], r[4], r[5]), stack + threadIdx.x,
                                                  kBlock, ovf, nullptr, nullptr);
    HitRecord rec;
    if (h.tri < 0) {
      rec.geomID = rec.primID = 0xFFFFFFFFu;
      rec.t = __builtin_inff();
      rec.u = rec.v = 0.0f;
      rec.ng[0] = rec.ng[1] = rec.ng[2] = 0.0f;
    } else {
      const uint32_t g = ldg(s.triGeom + h.tri);
      rec.geomID = g;
      rec.primID = (uint32_t)h.tri - ldg(s.shapeTriOffset + g);
      rec.t = h.t;
      rec.u = h.u;
      rec.v = h.v;
      const float* p = s.triPos + (size_t)h.tri * 9;
      const V3 p0 = load3g(p), p1 = load3g(p + 3), p2 = load3g(p + 6);
      const V3 ng = normalize(cross(p1 - p0, p2 - p0));  // Scene.cpp:297, Embree's Ng orientation
      rec.ng[0] = ng.x;
      rec.ng[1] = ng.y;
      rec.ng[2] = ng.z;
    }
    float4* out = reinterpret_cast<float4*>(hits + q);
    out[0] = make_float4(__uint_as_float(rec.geomID), __uint_as_float(rec.primID), rec.t, rec.u);
    out[1] = make_float4(rec.v, rec.ng[0], rec.ng[1], rec.ng[2]);
  }
}

// ------------------------------------------------------ guide photons ----
// Caustic light paths as training samples for the guide, the photon-traced
// training of parametric guiding mixtures (Vorba et al. 2014, "On-line
// learning of parametric mixture models for light transport simulation").
// Light paths leave the surface lights as Scene::sampleLightRay emits them
// (Scene.cpp:527-537) and continue through concentrated lobes only, with the
// roulette of tracePhoton (PhotonMapping.cpp:191-265).  Where one lands on a
// guided receiver with a diffuse lobe after at least one such bounce it adds
// a sample in the camera samples' layout: (x, F = luminance of the flux),
// the normal facing the photon, an outgoing direction drawn around that
// normal (a diffuse receiver's incident light does not depend on it), and
// the direction the photon came from.  Photon t of pass p uses the stream
// (seed, t, p) of its own domain.
__global__ void __launch_bounds__(kBlock) kGuidePhotons(DevScene s, uint32_t pass, uint32_t count, uint2* overflow,
                                                       float4* samples, uint32_t* sampleCount, uint32_t cap) {
  __shared__ uint2 stack[kStackRows * kBlock];
  const uint32_t gtid = blockIdx.x * blockDim.x + threadIdx.x;
  uint2* ovf = overflow + (size_t)gtid * kStackOvf;
  const float minQ = 1.0f - hm::powf_pos(0.1f, 1.0f / (float)s.maxDepth);
  for (uint32_t t = gtid; t < count; t += gridDim.x * blockDim.x) {
    hrng::Stream rng = hrng::make_stream(s.seed, t, pass, hrng::kDomainGuidePhoton);
    const uint32_t li = lightCdfSearch(s, rng.canonical_double());
    const int32_t ltri = (int32_t)ldg(s.lightTris + li);
    const float* pp = s.triPos + (size_t)ltri * 9;
    const V3 p0 = load3g(pp), p1 = load3g(pp + 3), p2 = load3g(pp + 6);
    const V3 ngL = normalize(cross(p1 - p0, p2 - p0));
    const float su = rng.uniform01f();
    const float tt = hm::fsqrt(rng.uniform01f());
    const float b0 = 1.0f - tt, b2 = tt * su, b1 = fmaxf(0.0f, 1.0f - b0 - b2);
    const Interaction itL = makeInteractionB(s, ltri, b0, b1, b2, ngL);
    float pDir;
    V3 rd = sampleCosHemisphere(rng, itL.ng, &pDir);
    const DevMaterial lm = ldgStruct(s.mats + itL.mat);
    const V3 Le = v3(lm.emission[0], lm.emission[1], lm.emission[2]) * (float)kInvPi;
    V3 flux = Le * (__builtin_fabsf(dot(itL.ng, rd)) * s.totalLightArea / pDir);
    V3 ro = offsetOrigin(itL, true);
    Hit h = traceClosest<kStackLds, kStackOvf>(s, ro, rd, stack + threadIdx.x, kBlock, ovf, nullptr, nullptr);
    if (h.tri < 0) continue;
    Media md;
    md.n = 0;
    md.overflow = false;
    md.tx0 = 0u;
    int wavelength = -1;
    for (int depth = 0; depth < s.maxDepth; ++depth) {
      if (!(__builtin_isfinite(flux.x) && __builtin_isfinite(flux.y) && __builtin_isfinite(flux.z))) break;
      Interaction it = makeInteraction(s, h.tri, h.u, h.v);
      DevMaterial m = ldgStruct(s.mats + it.mat);
      if (m.isLight) break;
      uint32_t texel = 0u;
      if (m.textured) applyTextures(s, m, it, 1.0f - h.u - h.v, h.u, h.v, &texel);
      const V3 wo = -rd;
      if (depth > 0 && m.hasDiffuseLobe && guideEligible(m)) {
        const V3 nf = dot(it.ng, wo) >= 0.0f ? it.ng : -it.ng;
        float pd;
        const V3 wos = sampleCosHemisphere(rng, nf, &pd);
        const float F = 0.2126f * flux.x + 0.7152f * flux.y + 0.0722f * flux.z;
        if (F > 0.0f && F < 3.0e38f) {
          const uint32_t k = atomicAdd(sampleCount, 1u);
          if (k < cap) {
            const float pB = bsdfPdf(m, it, wos, wo, mediaOutsideIOR(s, md, it, wos, wavelength));
            samples[4 * (size_t)k] = f4(it.x, F);
            samples[4 * (size_t)k + 1] = f4(nf, 0.0f);
            samples[4 * (size_t)k + 2] = f4(wos, 0.0f);
            samples[4 * (size_t)k + 3] = f4(wo, pB);
          }
        }
      }
      float sp = 1.0f;
      if (wavelength == -1 && m.varyIOR) {
        const float q0 = 1.0f / 3.0f;
        const float xi = rng.uniform01f();
        wavelength = xi < q0 ? 0 : (xi < q0 + q0 ? 1 : 2);
        sp = q0;
      }
      const float outsideIOR = mediaOutsideIOR(s, md, it, wo, wavelength);
      BsdfSample bs = bsdfSample(m, rng, it, wo, wavelength, outsideIOR, true, 2);
      V3 thr = (bs.tD + bs.tC) / sp;
      if (isZero(thr)) break;
      const V3 o2 = offsetOrigin(it, bs.outside);
      const Hit h2 = traceClosest<kStackLds, kStackOvf>(s, o2, bs.dir, stack + threadIdx.x, kBlock, ovf, nullptr,
                                                        nullptr);
      if (h2.tri < 0 || h2.tri == it.tri) break;
      mediaUpdate(md, it, wo, bs.dir, texel, nullptr);
      const Interaction it2 = makeInteraction(s, h2.tri, h2.u, h2.v);
      thr = mul(thr, beersLaw(mediaTransmittance(s, md), norm(it2.x - o2)));
      const float rq = fmaxf(minQ, 1.0f - norm(thr));
      if (rng.uniform01f() <= rq) break;
      flux = mul(flux, thr) / (1.0f - rq);
      h = h2;
      rd = bs.dir;
    }
  }
}

}  // namespace

void tileOrder(uint32_t width, uint32_t height, uint32_t* order, uint32_t* rankOf) {
  uint32_t n = 0;
  for (uint32_t ty = 0; ty < height; ty += 8)
    for (uint32_t tx = 0; tx < width; tx += 8)
      for (uint32_t y = ty; y < ty + 8 && y < height; ++y)
        for (uint32_t x = tx; x < tx + 8 && x < width; ++x) {
          order[n] = y * width + x;
          rankOf[y * width + x] = n;
          ++n;
        }
}

namespace {

void hipOk(hipError_t e, const char* what) {
  if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

// Launches of one render's bounces.  Bounce p (0 or 1, in turn) reads the
// paths of set p and leaves the next bounce's in the other one.
template <bool MULTI, bool GUIDED, int W>
struct Bounces {
  const JobSet& js;
  const PathBuffers& pb;
  const LaunchConfig& cfg;
  hipStream_t stream;
  KernelTimer* timer;
  bool late;  // some job has both an environment and emissive triangles

  template <class F>
  void timed(int id, F&& launch) const {
    if (timer) timer->begin(id, stream);
    launch();
    if (timer) timer->end(id, stream);
  }
  // No more blocks than the pool has work for (an idle block still costs its
  // dispatch); whole rounds of the 8 XCDs.
  uint32_t blocks(uint32_t most, uint64_t items) const {
    const uint64_t need = ((items + kBlock - 1) / kBlock + 7) & ~7ull;
    return (uint32_t)std::min<uint64_t>(most, need);
  }
  void fillTrace(uint32_t p, bool fill) const {
    const PathSet& out = pb.set[p ^ 1u];
    if (fill)
      timed(kKGenerate, [&] {
        kFill<MULTI><<<blocks(8192, pb.capacity), kBlock, 0, stream>>>(js, pb, out, p);
      });
    timed(kKTrace, [&] {
      const uint32_t n = std::min(blocks(cfg.traceBlocks, 2ull * pb.capacity), pb.traceThreads / kBlock);
      if (cfg.countStats && late) kTrace<MULTI, true, W, true><<<n, kBlock, 0, stream>>>(js, pb, out, p);
      else if (cfg.countStats) kTrace<MULTI, true, W, false><<<n, kBlock, 0, stream>>>(js, pb, out, p);
      else if (late) kTrace<MULTI, false, W, true><<<n, kBlock, 0, stream>>>(js, pb, out, p);
      else kTrace<MULTI, false, W, false><<<n, kBlock, 0, stream>>>(js, pb, out, p);
    });
    if (late) timed(kKConnect, [&] { kConnectLate<MULTI><<<blocks(2048, pb.capacity), kBlock, 0, stream>>>(js, pb, out, p); });
    if (GUIDED && js.g.sampleCap > 0u)
      timed(kKMisc, [&] { kHarvest<<<blocks(2048, pb.capacity), kBlock, 0, stream>>>(js.g, pb, p); });
  }
  // The paths of bounce p to their ends, if they are the render's last and
  // few (see finishing).
  void finish(uint32_t p) const {
    timed(kKFinish, [&] {
      const uint32_t n = std::min(blocks(kFinishBlocks, 8ull * pb.capacity), pb.traceThreads / kBlock);
      if (cfg.countStats) kFinish<MULTI, true, W><<<n, kBlock, 0, stream>>>(js, pb, pb.set[p], p);
      else kFinish<MULTI, false, W><<<n, kBlock, 0, stream>>>(js, pb, pb.set[p], p);
    });
  }
  // `n` bounces (even, so every chunk issues identical launches, which is what
  // a captured graph replays).  With `fill` paths may start, and the last ones
  // are left to a later chunk; without, kFinish takes them.
  void chunk(uint32_t n, bool fill) const {
    JobSet shadeJobs = js;
    if (fill) shadeJobs.finishPaths = 0u;  // the test kShade shares with kFinish
    for (uint32_t it = 0; it < n; ++it) {
      const uint32_t p = (it & 1u) ^ 1u;
      if (shadeJobs.finishPaths > 0u) finish(p);
      if (GUIDED)
        timed(kKGuideInfer, [&] {
          kGuideInfer<<<kGuideInferBlocks, kGuideInferThreads, 0, stream>>>(js, pb, pb.set[p], p);
        });
      timed(kKShade, [&] {
        kShade<MULTI, GUIDED><<<blocks(cfg.shadeBlocks, pb.capacity), kBlock, 0, stream>>>(
            shadeJobs, pb, pb.set[p], pb.set[p ^ 1u], p, cfg.countStats ? 1u : 0u);
      });
      fillTrace(p, fill);
    }
  }
};

// f(bounces) with the kernels of a batch or of one job, the jobs' node width
// compiled in (0: a batch of both, each job's width read by the kernels; two
// traversals in one kernel spill at 8 waves per SIMD, 12.4 against 9.0 ms on
// the cuboid batch).
template <class F>
void withBounces(const JobSet& js, const PathBuffers& pb, const LaunchConfig& cfg, hipStream_t stream,
                 KernelTimer* timer, bool late, bool guided, int width, F&& f) {
  if (js.nJobs > 1 && width == 4) f(Bounces<true, false, 4>{js, pb, cfg, stream, timer, late});
  else if (js.nJobs > 1 && width == 8) f(Bounces<true, false, 8>{js, pb, cfg, stream, timer, late});
  else if (js.nJobs > 1) f(Bounces<true, false, 0>{js, pb, cfg, stream, timer, late});
  else if (guided && js.s.bvhWidth == 8) f(Bounces<false, true, 8>{js, pb, cfg, stream, timer, late});
  else if (guided) f(Bounces<false, true, 4>{js, pb, cfg, stream, timer, late});
  else if (js.s.bvhWidth == 8) f(Bounces<false, false, 8>{js, pb, cfg, stream, timer, late});
  else f(Bounces<false, false, 4>{js, pb, cfg, stream, timer, late});
}

}  // namespace

size_t jobTableBytes(uint32_t nJobs) {
  const size_t a = (sizeof(DevScene) * nJobs + 255) & ~(size_t)255;
  return a + sizeof(PassInfo) * nJobs;
}

void renderJobs(const std::vector<RenderJobDesc>& jobs, const PathBuffers& pb, const LaunchConfig& cfg,
                hipStream_t stream, KernelTimer* timer, const GuideRun* guide, void* jobTables) {
  const uint32_t nJobs = (uint32_t)jobs.size();
  if (nJobs == 0) return;
  std::vector<DevScene> scenes(nJobs);
  std::vector<PassInfo> passes(nJobs);
  uint64_t total = 0;
  int maxDepth = 1;
  bool late = false;
  int width = 0;  // the jobs' node width, 0 if they differ
  for (uint32_t j = 0; j < nJobs; ++j) {
    const RenderJobDesc& d = jobs[j];
    scenes[j] = d.scene;
    PassInfo& pi = passes[j];
    pi.first = d.first;
    pi.pixels = d.scene.width * d.scene.height;
    pi.paths = d.n * pi.pixels;
    pi.pidBase = (uint32_t)total;
    pi.tileOrder = d.dTileOrder;
    pi.rankOf = d.dRankOf;
    pi.offsets = d.dOffsets;
    if (pi.pixels > pb.ringPaths) throw std::runtime_error("renderJobs: results ring smaller than one sample");
    total += (uint64_t)d.n * pi.pixels;
    maxDepth = std::max(maxDepth, d.scene.maxDepth);
    late = late || (d.scene.hasEnv && d.scene.hasSurfaceLight);
    width = j == 0 || width == d.scene.bvhWidth ? d.scene.bvhWidth : 0;
  }
  if (total >= (1ull << 31)) throw std::runtime_error("renderJobs: more than 2^31 paths in one call");
  JobSet js{};
  js.s = scenes[0];
  js.pi = passes[0];
  js.nJobs = nJobs;
  js.paths = (uint32_t)total;
  if (guide) {
    if (nJobs != 1) throw std::runtime_error("renderJobs: guided rendering takes one job");
    js.g = *guide;
  }
  if (nJobs > 1) {
    if (!jobTables) throw std::runtime_error("renderJobs: no job table buffer for a batch");
    char* base = (char*)jobTables;
    void* dScenes = base;
    void* dPasses = base + ((sizeof(DevScene) * nJobs + 255) & ~(size_t)255);
    hipOk(hipMemcpyAsync(dScenes, scenes.data(), sizeof(DevScene) * nJobs, hipMemcpyHostToDevice, stream), "copy");
    hipOk(hipMemcpyAsync(dPasses, passes.data(), sizeof(PassInfo) * nJobs, hipMemcpyHostToDevice, stream), "copy");
    js.scenes = (const DevScene*)dScenes;
    js.passes = (const PassInfo*)dPasses;
  }
  if (total == 0) return;
  js.finishPaths = guide || late ? 0u : kFinishPaths;
  if (late && !pb.sh.lateQ) throw std::runtime_error("renderJobs: no buffers for late light samples");
  auto t0 = [&](int k) {
    if (timer) timer->begin(k, stream);
  };
  auto t1 = [&](int k) {
    if (timer) timer->end(k, stream);
  };
  const uint32_t chunk = std::max<uint32_t>(2, (cfg.chunk + 1) & ~1u);
  // Paths started by the end of chunk c have finished `lag` chunks later: a
  // path has at most maxDepth vertices, one per bounce.
  const uint32_t lag = ((uint32_t)maxDepth + chunk - 1) / chunk;
  std::vector<uint32_t> acc(nJobs, 0);  // samples of each job added to its films
  uint32_t front = 0;                    // first job not completely added
  auto accPid = [&]() -> uint64_t {
    return front < nJobs ? (uint64_t)passes[front].pidBase + (uint64_t)acc[front] * passes[front].pixels : total;
  };
  // Paths that may have started when all below `done` have finished: those with
  // a place in the ring, and (training) one for their records.
  auto startLimit = [&](uint64_t done) {
    uint64_t most = std::min<uint64_t>(total, accPid() + pb.ringPaths);
    if (guide && guide->sampleCap > 0u) most = std::min<uint64_t>(most, done + guide->recPaths);
    return (uint32_t)most;
  };
  uint32_t limit = startLimit(0);
  t0(kKMisc);
  kInitRender<<<1, 64, 0, stream>>>(pb.counters, limit);
  t1(kKMisc);
  auto bounces = [&](KernelTimer* t, auto&& f) { withBounces(js, pb, cfg, stream, t, late, guide != nullptr, width, f); };
  bounces(timer, [&](const auto& b) { b.fillTrace(0u, true); });
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  struct GraphFree {
    hipGraph_t& g;
    hipGraphExec_t& e;
    ~GraphFree() {
      if (e) (void)hipGraphExecDestroy(e);
      if (g) (void)hipGraphDestroy(g);
    }
  } graphFree{graph, exec};
  // Per-kernel event timing needs eager launches (HIP gives no elapsed time
  // for events recorded inside a captured graph), so a timed render does not
  // replay graphs.
  if (cfg.useGraph && !timer) {
    hipOk(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
    bounces(nullptr, [&](const auto& b) { b.chunk(chunk, true); });
    hipOk(hipStreamEndCapture(stream, &graph), "hipStreamEndCapture");
    hipOk(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0), "hipGraphInstantiate");
  }
  std::vector<uint32_t> startedBy;
  uint64_t next = std::min<uint64_t>(limit, pb.capacity);  // paths started so far
  for (uint32_t c = 0;; ++c) {
    // a small render is all last paths: no bounce kernels
    const bool finishNow = !exec && total <= js.finishPaths && next >= total;
    if (exec) {
      t0(kKGraph);
      hipOk(hipGraphLaunch(exec, stream), "hipGraphLaunch");
      t1(kKGraph);
    } else {
      bounces(timer, [&](const auto& b) {
        if (finishNow) b.finish(1u);
        else b.chunk(chunk, next < total);
      });
    }
    uint32_t cnt[kNumCounters];
    hipOk(hipMemcpyAsync(cnt, pb.counters, sizeof(cnt), hipMemcpyDeviceToHost, stream), "counter readback");
    hipOk(hipStreamSynchronize(stream), "hipStreamSynchronize");
    // the chunk's last bounce (p = 0) left the next one's counters in set 1
    next = cnt[kCntSet + kCntNext];
    const uint32_t live = finishNow ? 0u : cnt[kCntSet + kCntLive];
    startedBy.push_back((uint32_t)next);
    uint64_t done = live == 0 ? next : (c >= lag ? startedBy[c - lag] : 0u);
    for (uint32_t j = front; j < nJobs && passes[j].pidBase < done; ++j) {
      const PassInfo& pi = passes[j];
      uint32_t n = pi.paths / pi.pixels;
      uint32_t complete = (uint32_t)std::min<uint64_t>(n, (done - pi.pidBase) / pi.pixels);
      if (complete > acc[j]) {
        uint32_t blocks = (pi.pixels + kBlock - 1) / kBlock;
        t0(kKAccumulate);
        kAccumulate<<<blocks, kBlock, 0, stream>>>(pb, pi, acc[j], complete, jobs[j].dColor, jobs[j].dNormal,
                                                   jobs[j].dAlbedo);
        t1(kKAccumulate);
        acc[j] = complete;
      }
    }
    while (front < nJobs && acc[front] * (uint64_t)passes[front].pixels == passes[front].paths) ++front;
    const uint32_t newLimit = startLimit(done);
    if (newLimit != limit) {
      t0(kKMisc);
      kSetLimit<<<1, 64, 0, stream>>>(pb.counters, newLimit);
      t1(kKMisc);
      limit = newLimit;
    }
    if (live == 0 && next >= total) break;
  }
  hipOk(hipStreamSynchronize(stream), "hipStreamSynchronize");
  if (front != nJobs) throw std::runtime_error("renderJobs: not every sample was accumulated");
}

uint32_t queryBlocks(uint32_t n) {
  return std::min<uint32_t>((n + kBlock - 1) / kBlock, kQueryBlocks);
}

namespace {
// Blocks of a query on an overflow array of `entries`, `slice` per thread.
uint32_t queryGrid(uint32_t n, size_t entries, uint32_t slice) {
  // the grid-stride index q + stride stays below 2^32
  if (n >= 0x80000000u) throw std::runtime_error("more than 2^31 - 1 rays in one query");
  if (slice == 0) return queryBlocks(n);
  const size_t most = entries / ((size_t)slice * kBlock);
  if (most == 0) throw std::runtime_error("traversal stack overflow array smaller than one block's");
  return (uint32_t)std::min<size_t>(queryBlocks(n), most);
}
}  // namespace

void launchTraceHits(const DevScene& s, const float* dRays, uint32_t n, HitRecord* dHits, uint2* dOverflow,
                     size_t entries, uint32_t slice, hipStream_t stream) {
  const uint32_t blocks = queryGrid(n, entries, slice);
  if (blocks == 0) return;
  if (s.bvhWidth == 8) kTraceHits<8><<<blocks, kBlock, 0, stream>>>(s, dRays, n, dHits, dOverflow, slice);
  else kTraceHits<4><<<blocks, kBlock, 0, stream>>>(s, dRays, n, dHits, dOverflow, slice);
}

void launchTraceClosest(const DevScene& s, const float* dRays, uint32_t n, int32_t* dTri, float* dTuv, uint2* dOverflow,
                        size_t entries, uint32_t slice, hipStream_t stream) {
  const uint32_t blocks = queryGrid(n, entries, slice);
  if (blocks == 0) return;
  if (s.bvhWidth == 8) kTraceRays<8><<<blocks, kBlock, 0, stream>>>(s, dRays, n, dTri, dTuv, dOverflow, slice);
  else kTraceRays<4><<<blocks, kBlock, 0, stream>>>(s, dRays, n, dTri, dTuv, dOverflow, slice);
}

void launchGuidePhotons(const DevScene& s, uint32_t pass, uint32_t count, uint2* dOverflow, uint32_t overflowThreads,
                        float4* samples, uint32_t* sampleCount, uint32_t cap, hipStream_t stream) {
  if (count == 0 || !s.hasSurfaceLight || s.numLights == 0) return;
  uint32_t blocks = (count + kBlock - 1) / kBlock;
  const uint32_t maxBlocks = overflowThreads / kBlock;
  if (blocks > maxBlocks) blocks = maxBlocks;
  if (blocks == 0) return;
  kGuidePhotons<<<blocks, kBlock, 0, stream>>>(s, pass, count, dOverflow, samples, sampleCount, cap);
}

}  // namespace hasty
