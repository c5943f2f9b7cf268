// Wavefront path-tracing kernels: host-side launch interface.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "guide.h"
#include "pt_device.h"

#include <vector>

namespace hasty {

// Path state, structure of arrays, of the paths alive at one bounce, packed
// at [0, n).  There are two sets: a bounce reads one and writes the paths that
// go on (and then the paths that start) to the other, so every access of
// every stage is to consecutive records whatever ended in between.
struct PathSet {
  float4* rayO;   // origin; w unused
  float4* rayD;   // direction; w = pdf of the BSDF sample that produced it
  float4* beta;   // path throughput (not stored for paths that start)
  float4* L;      // accumulated radiance (not stored for paths that start)
  uint4* state;   // x rng draws, y flags, z previous triangle, w path id
  uint4* media;   // 2 x uint4 per path (8 entries), read when the flags say so
  uint32_t* mediaTx;  // 8 per path: albedo texel of each media entry (or null)
};

// Shadow rays of one bounce: record i belongs to the vertex of path i, and q
// lists the n that were cast.  Every factor of a light sample but its
// visibility is known when it is drawn, so the record carries the radiance to
// add if nothing is in the way, and q says where: to the path's L in the next
// set, or, for a path that ended at the vertex, to the results ring
// (kDestRing).
struct ShadowRays {
  uint2* q;      // record, destination
  float4* o;     // origin; w = t of the target triangle (+inf: environment)
  float4* d;     // direction; w = target triangle, kTargetSky or kTargetLate (bits)
  float4* c;     // radiance to add
  uint32_t* job; // job index (batches)
  // Scenes with both an environment and emissive triangles (else null): an
  // environment sample may meet a light instead of the sky, and its term is
  // then computed from these (see kConnectLate).
  float4* lateFD;   // f_diffuse; w = |cos| at the shading point
  float4* lateFC;   // f_concentrated; w = shading triangle (bits)
  float4* lateThr;  // local throughput (Beer / (1 - q)); w = BSDF pdf of the direction
  float4* lateBeta; // path throughput at the vertex
  float4* lateT;    // transmittance of the light-ray media copy
  float4* lateHit;  // the light that was met: t, u, v, triangle (bits)
  uint2* lateQ;     // entries of q whose ray met a light
};
constexpr int32_t kTargetSky = -1, kTargetLate = -2;
constexpr uint32_t kDestRing = 0x80000000u;

// Memory of a render: the path pool of `capacity` paths in flight (a path
// that ends makes room for the next of the render), its shadow rays, and the
// results ring.
struct PathBuffers {
  PathSet set[2];
  float4* hit;    // closest hits of the paths alive: t, u, v, triangle (bits)
  ShadowRays sh;
  uint2* ended;   // training: path id and record count of the paths that ended
  uint32_t* counters;         // see CounterId
  unsigned long long* stats;  // see StatId
  uint2* stackOverflow;
  float4* ringL;  // finished paths: radiance, normal, albedo at
  float4* ringN;  // ring slot (global path id % ringPaths)
  float4* ringA;
  uint32_t ringPaths;
  uint32_t capacity;
  uint32_t traceThreads;  // threads of the traversal grids (overflow slices)
};

// Counters of a bounce; there are two sets, used in turn, so that the kernel
// that closes a bounce can prepare the next one's while its own are read.
enum CounterId {
  kCntA = 0,     // paths that went on (packed at the front of the next set)
  kCntS = 1,     // shadow rays (A and S are one 64-bit atomic)
  kCntLive = 2,  // paths alive at this bounce
  kCntNext = 3,  // next path id to start
  kCntEnded = 4, // training: paths that ended with records
  kCntLate = 5,  // shadow rays that met a light instead of the sky
  kCntSet = 8,   // words per set
  kCntLimit = 2 * kCntSet,  // path ids below this may start (results ring space)
  kNumCounters = 3 * kCntSet
};

// One job of a render call: samples first .. first + paths / pixels - 1 of
// every pixel of its scene.  Path ids are global over the jobs of a call:
// job j owns [pidBase, pidBase + paths); inside a job, local id =
// (sample - first) * pixels + rank with pixel = tileOrder[rank] (8x8 tiles).
// Finished paths go to ring slot (global id % ringPaths).
struct PassInfo {
  uint32_t first;
  uint32_t pixels;
  uint32_t paths;
  uint32_t pidBase;
  const uint32_t* tileOrder;  // rank -> pixel
  const uint32_t* rankOf;     // pixel -> rank
  const float2* offsets;      // per sample of the call
};

// Guided rendering (single job): guide outputs of the paths alive, training
// records by path id modulo recPaths (2 x {position, normal, wo + the density wi was drawn
// with, wi + the BSDF density of wi, throughput before the sample, radiance
// before the continuation}) and the training samples harvested when paths
// end (4 float4 each: position + weight, normal, wo + drawing density,
// wi + BSDF density).
struct GuideRun {
  guide::Net net;
  float4* raw;      // 10 float4 per path alive
  float4* rec;      // 12 float4 for each of recPaths paths (training)
  uint32_t recPaths;  // paths from the oldest in flight on that may have records
  float4* samples;  // sampleCap x 4 float4
  uint32_t* sampleCount;
  uint32_t sampleCap;
  float fraction;   // probability of drawing the direction from the guide
  float* sel;       // per path alive: that probability as the guide learned it (or null: `fraction`)
  uint32_t maxDepth;  // only vertices of depth below this are guided
  float maxThroughput;  // ... and only while every channel of the path throughput is at most this
};

// The jobs of a render call.  With one job its scene and pass travel in the
// kernel arguments (`s`, `pi`); with several, kernels look them up by path id.
struct JobSet {
  hdev::DevScene s;
  PassInfo pi;
  const hdev::DevScene* scenes;
  const PassInfo* passes;
  uint32_t nJobs;
  uint32_t paths;  // over all jobs
  uint32_t finishPaths;  // the last paths are finished one by one from this many (0: never)
  GuideRun g;      // read by the guided kernels only
};

// Traversal stack entries kept in LDS per lane (the rest spill to a global
// slice); a build knob because it trades LDS for spills.  With the row for
// writes past it, 9 is what 8 blocks of 256 lanes fit in a CU's 160 KB (7, 8,
// 9 entries: 117.2, 116.0, 115.3 ms on the GGX grid).
#ifndef HASTY_STACK_LDS
#define HASTY_STACK_LDS 9
#endif
constexpr int kStackLds = HASTY_STACK_LDS;
constexpr int kStackRows = kStackLds + 1;   // LDS rows (the last for writes past the LDS part)
constexpr int kStackOvf = 80 - kStackLds;  // 80 entries per lane in all
constexpr int kBlock = 256;

// 64-bit device statistics (filled when LaunchConfig::countStats is set).
// kStatNodes / kStatTris count the extension rays' node visits and triangle
// tests, kStatShadowNodes / kStatShadowTris the shadow rays'.
enum StatId {
  kStatExtRays = 0,
  kStatShadowRays,
  kStatNodes,
  kStatTris,
  kStatMediaOverflow,
  kStatShadowNodes,
  kStatShadowTris,
  kNumStats = 8
};

struct LaunchConfig {
  uint32_t traceBlocks = 2048;  // persistent-style grid of the traversal kernels
  uint32_t shadeBlocks = 8192;
  uint32_t chunk = 8;           // bounces between host checks of the live count
  bool useGraph = false;        // replay each chunk of bounces as one captured hipGraph
  bool countStats = false;
};

enum KernelId {
  kKGenerate = 0,
  kKTrace,
  kKShade,
  kKFinish,
  kKConnect,
  kKAccumulate,
  kKMisc,
  kKGraph,
  kKGuideInfer,
  kKSppmRadii,
  kKSppmCellSize,
  kKSppmPhotons,
  kKSppmBuild,
  kKSppmCamera,
  kKSppmGather,
  kNumKernels
};
const char* kernelName(int id);

// Timing hook: called around each launch when profiling is on.
struct KernelTimer {
  virtual void begin(int kernel, hipStream_t s) = 0;
  virtual void end(int kernel, hipStream_t s) = 0;
  virtual ~KernelTimer() {}
};

// One job of renderJobs: scene (seed set), samples [first, first + n), the n
// pixel offsets, the tile order and its inverse, device films (sums, added to
// in sample order).
struct RenderJobDesc {
  hdev::DevScene scene;
  uint32_t first, n;
  const float2* dOffsets;
  const uint32_t* dTileOrder;
  const uint32_t* dRankOf;
  float* dColor;
  float* dNormal;
  float* dAlbedo;
};

// Device bytes of the scene and pass tables of an n-job render call.
size_t jobTableBytes(uint32_t nJobs);

// Renders every job through one shared pool of path slots (paths of all jobs
// in flight together; at most 2^31 paths per call).  Synchronises with the
// stream once per cfg.chunk bounces.  With more than one job the per-job
// tables go to `jobTables` (device memory of jobTableBytes(n) bytes at least).
void renderJobs(const std::vector<RenderJobDesc>& jobs, const PathBuffers& pb, const LaunchConfig& cfg,
                hipStream_t stream, KernelTimer* timer, const GuideRun* guide = nullptr, void* jobTables = nullptr);

// Pixels of a width x height film in 8x8-tile order (row-major inside a
// tile), and the inverse map.
void tileOrder(uint32_t width, uint32_t height, uint32_t* order, uint32_t* rankOf);

// Hit record of a batched closest-hit query: the layout of HastyHit
// (include/hasty_amd.h): geomID, primID (0xFFFFFFFF on a miss), t, u, v,
// unit geometric normal.
struct HitRecord {
  uint32_t geomID, primID;
  float t, u, v;
  float ng[3];
};
static_assert(sizeof(HitRecord) == 32, "HitRecord is 32 bytes");

// Stack entries per lane that a traversal of a BVH of this width and depth
// can need beyond the kStackLds in LDS: at most width - 1 per inner level,
// and the root.
constexpr uint32_t overflowSlice(int width, int depth) {
  const int need = (width - 1) * depth + 1;
  return need > kStackLds ? (uint32_t)(need - kStackLds) : 0u;
}
// Blocks of a query of n rays: the chip's 8 blocks per CU at most.
constexpr uint32_t kQueryBlocks = 2048;
uint32_t queryBlocks(uint32_t n);

// Closest-hit records for n rays (6 floats each).  `overflow` holds `entries`
// stack entries, `slice` (overflowSlice of the scene's BVH) for each thread;
// the grid is cut to what they allow.
void launchTraceHits(const hdev::DevScene& scene, const float* dRays, uint32_t n, HitRecord* dHits, uint2* dOverflow,
                     size_t entries, uint32_t slice, hipStream_t stream);

// Caustic photons as guide training samples (4 float4 each, appended at
// atomicAdd(sampleCount) below cap) from `count` light paths of pass `pass`;
// `overflow`: kStackOvf entries for each of the overflowThreads threads (a
// multiple of kBlock).  Nothing without surface lights.
void launchGuidePhotons(const hdev::DevScene& scene, uint32_t pass, uint32_t count, uint2* dOverflow,
                        uint32_t overflowThreads, float4* samples, uint32_t* sampleCount, uint32_t cap,
                        hipStream_t stream);

// Closest hit for n rays (6 floats each): tri, t, u, v.
void launchTraceClosest(const hdev::DevScene& scene, const float* dRays, uint32_t n, int32_t* dTri, float* dTuv,
                        uint2* dOverflow, size_t entries, uint32_t slice, hipStream_t stream);

}  // namespace hasty
