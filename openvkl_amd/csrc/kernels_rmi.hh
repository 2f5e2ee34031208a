// Interval-driven ray marching with transfer-function compositing, fused
// with the interval iterator and the sampler: the reference's ray-march
// iterator renderer (examples/interactive/renderer/ray_march_iterator/
// RayMarchIterator.ispc:39-137), one ray per work-item. Instantiated by
// kernels_rmi_dense.hip (structuredRegular sources) and
// kernels_rmi_sparse.hip (vdb and temporal sources), which compile in
// parallel.
#pragma once

#include "kernels.h"
#include "kernels_hit.hh"

namespace vklhip {

// TransferFunction_sample (examples/interactive/renderer/
// TransferFunction.ih:17-47): tf holds n (r, g, b, opacity) entries over
// [lo, hi]; floor(v) is kept inside [0, n - 1] so a non-finite range cannot
// index out of the table.
template <typename Table>
VKL_DEV void tfSampleRgba(Table tf, uint32_t n, float lo, float hi, float v, float c[4])
{
  if (__builtin_isnan(v) || n == 0) {
    c[0] = c[1] = c[2] = c[3] = 0.f;
    return;
  }
  if (v <= lo || v >= hi) {
    const auto e = v <= lo ? tf : tf + 4 * (n - 1);
    c[0] = e[0], c[1] = e[1], c[2] = e[2], c[3] = e[3];
    return;
  }
  v        = (v - lo) / (hi - lo) * ((float)n - 1.f);
  float fi = floorf(v);
  if (!(fi >= 0.f)) fi = 0.f;
  if (fi > (float)(n - 1)) fi = (float)(n - 1);
  const int i     = (int)fi;
  const int j     = i + 1 < (int)n - 1 ? i + 1 : (int)n - 1;
  const float rem = v - fi;
#pragma unroll
  for (int k = 0; k < 4; k++) c[k] = (1.f - rem) * tf[4 * i + k] + rem * tf[4 * j + k];
}

VKL_DEV float minf_(float a, float b) { return a < b ? a : b; }

// Samples of an interval that a vdb march takes together (independent loads
// in flight): its samples wait on dependent index and leaf loads. Dense
// marches take one: their coherent rays hit the caches, and they lose more to
// the extra registers than they gain.
constexpr int kSamplesAhead = 4;

// Lanes of a vdb march that wait for an interval, times this, against the
// lanes that have samples to take: below it the interval phase waits. 960 x
// 540 rays in a 512^3 float shell, four samples a voxel: 4.09 ms at 3, 4.50 at
// 1, 4.14 at 2, 4.05 at 6; one sample a voxel 1.53, 1.58, 1.54, 1.55.
constexpr uint32_t kMarchIntervalVote = 3;

// Transfer functions of up to this many entries are read from LDS (4 KB a
// wavefront, so that 5 wavefronts per SIMD still fit): every sample reads two
// entries at its own place of the table, and through the vector L1 these reads
// queued with the voxels'. 1080p frames of a 512^3 float volume, 64 entries,
// 4.40 -> 3.70 ms; 2^18 camera rays in a 1024^3 vdb 3.18 -> 2.98 ms. On both
// sides of the line, 960 x 540 rays in 256 x 240 x 220 floats: 256 entries
// 1.05 ms, 257 1.20 ms; 64 x 48 rays 0.60 and 0.61 ms.
constexpr uint32_t kTableEntries = 256;

// Whether a vdb march takes an interval's samples to its end before the next
// interval, instead of mixing both in one loop (below).
template <int kFilter, int kDepth>
constexpr bool wholeIntervals()
{
  return kDepth <= 1 && kFilter != kFilterCubic;
}

// rgba[4r..4r+3] = composited colour and accumulated opacity of ray r.
//
// vdb sources: bound by dependent loads and by lanes that wait for each
// other, so the wavefront runs one loop in which the lanes whose interval is
// used up visit the next voxel and the others take their next samples. 2^18
// rays through a 1024^3 shell, camera / random: 6.26 / 6.23 -> 3.33 / 4.17 ms
// at depth 2, 14.3 / 19.6 -> 5.3 / 5.9 ms at depth 3, against nested loops
// per interval; 4 waves per SIMD (5 waves: 15-60 % slower; the compiler's 3
// at depth 3: 9.2 ms for random rays). Observed sources (16-24 B of scratch at
// depth 3): 960 x 540 in a 512^3 float shell 4.1 -> 3.1 and 13.0 -> 6.2 ms at
// depths 2 and 3; a temporal vdb (up to 88 B) 6.6 -> 4.7 and 6.9 -> 4.9 ms. At
// depths 0 and 1 an interval is 128 voxels and more, and a lane takes all of
// its samples before the next one, which keeps camera rays in step: 960 x 540
// in a 512^3 float shell at depth 1, 2.60 ms against 3.07 in the one loop
// (depth 0: the same). Tricubic samples keep the one loop there (480 x 270: 8.4
// against 9.7 ms).
//
// structuredRegular sources: bound by instruction issue on coherent rays,
// whose lanes share voxel lines as long as they stay in step, which the
// nested loops keep (one loop as above took twice as long for a 1080p frame of
// a 512^3 volume, with 5 times the L2 requests). 5 waves per SIMD: 91 VGPRs
// without spill at depth 2, the default (4 waves the same, 6 waves 7 % slower).
//
// Tricubic samples keep the compiler's choice. The row loads of x-fastest
// volumes cost float voxels a wavefront per SIMD (3 to 2), which bricks pay: 480
// x 270 rays of 256 x 240 x 220 floats 2.84 -> 1.24 ms x-fastest, 1.43 -> 1.29
// corner-packed, 2.35 -> 2.58 on bricks. Asking for 3 spills: 1.53, 1.57, 2.71.
template <typename Src, int kFilter, int kDepth, int kQuery>
__global__ __launch_bounds__(kIterBlock) __attribute__((
    amdgpu_waves_per_eu(kFilter == kFilterCubic ? 1 : IsDenseSource<Src>::value ? 5 : kDepth <= 1 ? 1 : 4)))
void kRayMarchIntervals(const IteratorContextView *__restrict__ cp,
                                                                  AttrView a, RayMarchIntervalsArgs m)
{
  __shared__ __attribute__((aligned(16))) float table[4 * kTableEntries];
  const uint32_t lane = xcdBandBlock(blockIdx.x, gridDim.x) * kIterBlock + threadIdx.x;
  const uint32_t r    = lane < m.numRays ? lane : m.numRays - 1;
  const IteratorContextView &c = *cp;
  PointSampler<Src, kFilter> smp(c.sampler.grid, a, c.attributeIndex);
  smp.setTime(m.time);
  const F3 o = {m.org[3 * r], m.org[3 * r + 1], m.org[3 * r + 2]};
  const F3 d = {m.dir[3 * r], m.dir[3 * r + 1], m.dir[3 * r + 2]};
  IntervalState st;
  intervalInit<kDepth>(c, st, o, d, rayRange(m.tRanges, r));
  // Wavefronts whose rays all miss the volume leave the table alone: a 1080p
  // frame of such rays took 63 us with 256 entries staged, 45 without.
  const bool staged = m.tfSize <= kTableEntries && __ballot(st.dda.t <= st.tMax) != 0;
  if (staged)
    for (uint32_t i = threadIdx.x; i < 4 * m.tfSize; i += kIterBlock) table[i] = m.tf[i];
  __syncthreads();
  if (lane >= m.numRays) return;
  const float dtNominal = st.nominalDeltaT / m.samplingRate;
  float cr = 0.f, cg = 0.f, cb = 0.f, alpha = 0.f;
  uint32_t taken = 0;
  auto composite = [&](float s, float dt) {
    taken++;
    float rgba[4];
    if (staged)
      tfSampleRgba((const __attribute__((address_space(3))) float *)table, m.tfSize, m.tfLo, m.tfHi, s, rgba);
    else
      tfSampleRgba(m.tf, m.tfSize, m.tfLo, m.tfHi, s, rgba);
    float op = rgba[3] * dt;
    op       = op > 0.f ? op : 0.f;
    op       = op < 1.f ? op : 1.f;
    cr       = cr + (1.f - alpha) * (rgba[0] * op);
    cg       = cg + (1.f - alpha) * (rgba[1] * op);
    cb       = cb + (1.f - alpha) * (rgba[2] * op);
    alpha    = alpha + (1.f - alpha) * op;
  };
  if constexpr (IsDenseSource<Src>::value) {
    IntervalOut iv;
    while (alpha < 0.99f && taken < m.maxSamples && intervalNext<false, kDepth, kQuery>(c, st, iv)) {
      float lo = iv.tLower, hi = minf_(iv.tLower + dtNominal, iv.tUpper);
      while (hi - lo > 0.f && alpha < 0.99f && taken < m.maxSamples) {
        const float t = 0.5f * (lo + hi);
        composite(smp(F3{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z}), hi - lo);
        lo = hi;
        hi = minf_(lo + dtNominal, iv.tUpper);
      }
    }
  } else {
    IntervalWalk walk;
    float lo = 0.f, hi = 0.f, end = 0.f;  // the next sub-interval, the interval's end
    while (alpha < 0.99f && taken < m.maxSamples) {
      IntervalOut iv;
      if constexpr (wholeIntervals<kFilter, kDepth>()) {
        if (!intervalNext<false, kDepth, kQuery>(c, st, iv)) break;
        lo  = iv.tLower;
        end = iv.tUpper;
        hi  = minf_(lo + dtNominal, end);
      } else {
        const uint32_t waiting = (uint32_t)__popcll(__ballot(!(hi - lo > 0.f)));
        const uint32_t others  = (uint32_t)__popcll(__ballot(hi - lo > 0.f));
        if (waiting * kMarchIntervalVote >= others) {
          if (!(hi - lo > 0.f)) {
            const int event = intervalTick<false, kDepth, kQuery>(c, st, walk, iv);
            if (event == 2) break;
            if (event == 1) {
              lo  = iv.tLower;
              end = iv.tUpper;
              hi  = minf_(lo + dtNominal, end);
            }
          }
        }
      }
      if (!(hi - lo > 0.f)) continue;
      // The next kSamplesAhead sub-intervals (the same running sums as one
      // at a time), their samples issued together so that the loads overlap,
      // then composited in order with the same stopping rules; samples past
      // a stop are not counted.
      do {
        float tt[kSamplesAhead], dd[kSamplesAhead], ss[kSamplesAhead];
        uint32_t nk = 0;
#pragma unroll
        for (int k = 0; k < kSamplesAhead; k++) {
          const bool live = hi - lo > 0.f;
          tt[k]           = 0.5f * (lo + hi);
          dd[k]           = hi - lo;
          if (live) {
            nk = k + 1;
            lo = hi;
            hi = minf_(lo + dtNominal, end);
          }
        }
#pragma unroll
        for (int k = 0; k < kSamplesAhead; k++)
          ss[k] = (uint32_t)k < nk ? smp(F3{o.x + tt[k] * d.x, o.y + tt[k] * d.y, o.z + tt[k] * d.z}) : 0.f;
#pragma unroll
        for (int k = 0; k < kSamplesAhead; k++)
          if ((uint32_t)k < nk && alpha < 0.99f && taken < m.maxSamples) composite(ss[k], dd[k]);
      } while (wholeIntervals<kFilter, kDepth>() && hi - lo > 0.f && alpha < 0.99f && taken < m.maxSamples);
    }
  }
  m.rgba[4 * r]     = cr;
  m.rgba[4 * r + 1] = cg;
  m.rgba[4 * r + 2] = cb;
  m.rgba[4 * r + 3] = alpha;
  if (m.count) m.count[r] = taken;
}

// Launches the instantiation for the context's iterator depth on vdb
// sources (the DDA keeps only the levels it walks; on structuredRegular ones
// for the default depth, whose DDA step then needs no re-initialisation: 5.1
// -> 4.9 ms a 1080p frame of the 512^3 volume) and for its query kind
// (denseQueryOf: structuredRegular volumes within one level-1 node use the
// dense node numbering, and their kernels then carry no node-table query).
struct RayMarchIntervalsLaunch
{
  const IteratorContextView *c;
  AttrView a;
  RayMarchIntervalsArgs m;
  uint32_t depth;
  hipStream_t st;
  bool denseQuery;
  template <typename Src, int kFilter, int kDepth, int kQuery>
  hipError_t run() const
  {
    hipLaunchKernelGGL((kRayMarchIntervals<Src, kFilter, kDepth, kQuery>),
                       dim3((m.numRays + kIterBlock - 1) / kIterBlock), dim3(kIterBlock), 0, st, c, a, m);
    return hipGetLastError();
  }
  template <typename Src, int kFilter>
  hipError_t operator()() const
  {
    if constexpr (IsDenseSource<Src>::value) {
      if (denseQuery && depth == 2) return run<Src, kFilter, 2, 1>();
      return denseQuery ? run<Src, kFilter, -1, 1>() : run<Src, kFilter, -1, 0>();
    } else {
      switch (depth) {
      case 0: return run<Src, kFilter, 0, 0>();
      case 1: return run<Src, kFilter, 1, 0>();
      case 2: return run<Src, kFilter, 2, 0>();
      default: return run<Src, kFilter, 3, 0>();
      }
    }
  }
};

}  // namespace vklhip
