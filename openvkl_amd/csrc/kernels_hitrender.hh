// The hit-iterator renderer fused with hit iteration, gradients and shadow
// queries: examples/interactive/renderer/hit_iterator_renderer/
// HitIteratorRenderer.ispc:51-150, one ray per work-item. Instantiated by
// kernels_hitrender_dense.hip (structuredRegular sources) and
// kernels_hitrender_sparse.hip (vdb and temporal sources).
//
// The primary ray's hits are collected first and shaded afterwards, so the
// primary and shadow rays never need two hit-iterator states at once.
#pragma once

#include "kernels.h"
#include "kernels_hit.hh"
#include "kernels_rmi.hh"

namespace vklhip {

// normalize(v) = v (1 / sqrt(v . v)), correctly rounded square root and
// division.
VKL_DEV F3 normalize3(F3 v)
{
  const float inv = 1.f / sqrtf(v.x * v.x + v.y * v.y + v.z * v.z);
  return F3{v.x * inv, v.y * inv, v.z * inv};
}
VKL_DEV float dot3(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// Opacity 0.6 per shaded hit takes the accumulated opacity past 0.99 after
// 6 hits (binary32: 0.6, 0.84, 0.936, 0.9744, 0.98976, 0.995904), so a ray
// shades at most this many hits.
constexpr int kMaxShadedHits = 6;

// Lanes without a running query that let a wavefront stop for its shading.
constexpr uint32_t kShadeVote = 16;

// Two phases per ray, in the reference's order of results: first the
// primary ray's hits that will be shaded (the compositing opacity does not
// depend on the shading, so their number is known in advance), then each hit
// in order: gradient normal, shadow rays, compositing. Primary and shadow
// queries share one search state and one hitTick call site. The hits and the
// shading state wait in LDS while a query runs: they are touched once per
// query, and in registers they displaced the search's own state.
//
// Bound by instruction issue with part of the lanes idle: a 1080p frame of a
// 300 x 260 x 340 float volume with two iso values 33.1 -> 20.2 ms against
// nested loops per query (22 instead of 9 lanes active, 185 k instead of 538 k
// vector instructions a wavefront). 3 waves per SIMD (168 VGPRs): 2 waves took
// 1.4 times as long there, 4 and more spill the search's state and took 2 to 4
// times. The same line on vdb sources (36 bytes of scratch at 3 waves): 960 x
// 540 rays in a 512^3 float shell 17.7 ms, 21.1 at 2 waves; a temporal vdb 24.4
// and 26.9. Shading when 12 to 28 lanes wait measured the same; waiting for all
// 64 took 7 % longer.
template <typename Src, int kFilter, int kQuery>
__global__ __launch_bounds__(kIterBlock) __attribute__((
    amdgpu_waves_per_eu(kFilter == kFilterCubic ? 1 : 3)))
void kHitRender(const IteratorContextView *__restrict__ cp, AttrView a,
                                                          HitRenderArgs m)
{
  __shared__ float hitT[kMaxShadedHits][kIterBlock], hitS[kMaxShadedHits][kIterBlock], hitE[kIterBlock];
  __shared__ float bisect[kBisWords * kHitLanes];
  __shared__ float sN[3][kIterBlock], sCi[kIterBlock], sCo[kIterBlock], sIllum[kIterBlock], sRgba[4][kIterBlock];
  const uint32_t r = xcdBandBlock(blockIdx.x, gridDim.x) * kIterBlock + threadIdx.x;
  if (r >= m.numRays) return;
  const uint32_t lane          = threadIdx.x;
  const IteratorContextView &c = *cp;
  PointSampler<Src, kFilter> smp(c.sampler.grid, a, c.attributeIndex);
  smp.setTime(m.time);
  const uint32_t maxShade = m.maxHits < (uint32_t)kMaxShadedHits ? m.maxHits : (uint32_t)kMaxShadedHits;

  HitSearch st;
  hitInit<hitDepthOf<Src>()>(c, st.h, F3{m.org[3 * r], m.org[3 * r + 1], m.org[3 * r + 2]},
                             F3{m.dir[3 * r], m.dir[3 * r + 1], m.dir[3 * r + 2]}, rayRange(m.tRanges, r), m.time);
  hitBegin(st, bisect + lane);
#pragma unroll
  for (int i = 0; i < 4; i++) sRgba[i][lane] = 0.f;
  bool searching = maxShade > 0, done = false;
  uint32_t hits = 0, k = 0;
  float alphaP = 0.f;  // opacity after the hits collected so far
  int light    = -2;   // next light to test; -1: hit k not started; -2: collecting the hits
  int event    = 0;
  while (!done) {
    if (searching) {
      HitOut h;
      event = hitTick<decltype(smp), kQuery>(c, smp, st, h);
      if (event) {
        searching = false;
        if (light == -2 && event == 1) {
          hitT[hits][lane] = h.t;
          hitS[hits][lane] = h.sample;
          hitE[lane]       = h.epsilon;  // of every hit of a ray
          hits++;
          alphaP    = alphaP + (1.f - alphaP) * 0.6f;
          searching = alphaP < 0.99f && hits < maxShade;
        }
      }
    }
    // Lanes whose query has ended wait until several of them can go on
    // together: the shading below costs more instructions than a tick.
    const uint32_t busy = (uint32_t)__popcll(__ballot(searching));
    const uint32_t idle = (uint32_t)__popcll(__ballot(!searching));
    if (idle < kShadeVote && busy != 0) continue;
    if (searching) continue;
    const F3 light0 = normalize3(F3{1.f, 1.f, 1.f}), light1 = normalize3(F3{1.f, 1.f, -1.f});
    const F3 o = {m.org[3 * r], m.org[3 * r + 1], m.org[3 * r + 2]};
    const F3 d = {m.dir[3 * r], m.dir[3 * r + 1], m.dir[3 * r + 2]};
    F3 p = {0.f, 0.f, 0.f}, N = {sN[0][lane], sN[1][lane], sN[2][lane]};
    float ci = sCi[lane], co = sCo[lane], illum = sIllum[lane];
    if (light == -2) {
      light = -1;
    } else {
      if (event == 2) illum += fabsf(co) * (light == 0 ? 1.f : 0.8f);
      light++;
    }
    // Advance the shading to the next shadow query, compositing every hit
    // whose lights are done.
    bool query = false;
    while (k < hits) {
      const float t = hitT[k][lane];
      p             = F3{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z};
      if (light < 0) {  // start hit k
        const F3 wi = normalize3(F3{-1.f * d.x, -1.f * d.y, -1.f * d.z});
        const F3 q  = xfmPoint(c.sampler.grid.o2i, p);
        F3 gi       = {0.f, 0.f, 0.f};
        if (c.sampler.gradientFilter == kFilterLinear)
          gi = gradientLinear(smp.src, q);
        else if (c.sampler.gradientFilter == kFilterCubic)
          gi = gradientCubicBySlices(smp.src, q);
        N = normalize3(xfmNormal(c.sampler.grid.o2i, gi));
        if (isnan(N.x) || isnan(N.y) || isnan(N.z)) N = F3{0.f, 0.f, 0.f};
        ci = dot3(N, wi);
        if (sqrtf(dot3(N, N)) > 0.f) {
          illum = 0.1f;  // ambient
          light = 0;
        } else {
          illum = 1.f;  // no normal: unshaded
          light = 2;
        }
      }
      // the next light on the viewer's side of the surface
      while (light < 2) {
        co = dot3(N, light == 0 ? light0 : light1);
        if ((co > 0.f) == (ci > 0.f)) break;
        light++;
      }
      if (light < 2) {
        query = true;
        break;
      }
      float albedo[4];
      tfSampleRgba(m.tf, m.tfSize, m.tfLo, m.tfHi, hitS[k][lane], albedo);
      const float alpha = sRgba[3][lane];
      sRgba[0][lane]    = sRgba[0][lane] + (1.f - alpha) * illum * albedo[0];
      sRgba[1][lane]    = sRgba[1][lane] + (1.f - alpha) * illum * albedo[1];
      sRgba[2][lane]    = sRgba[2][lane] + (1.f - alpha) * illum * albedo[2];
      sRgba[3][lane]    = alpha + (1.f - alpha) * 0.6f;
      k++;
      light = -1;
    }
    if (query) {
      sN[0][lane] = N.x, sN[1][lane] = N.y, sN[2][lane] = N.z;
      sCi[lane] = ci, sCo[lane] = co, sIllum[lane] = illum;
      hitInit<hitDepthOf<Src>()>(c, st.h, p, light == 0 ? light0 : light1, Range1f{hitE[lane], vinf()}, m.time);
      hitBegin(st, bisect + lane);
      searching = true;
    } else {
      done = true;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; i++) m.rgba[4 * r + i] = sRgba[i][lane];
  if (m.count) m.count[r] = hits;
}

// The kernel is specialised on the context's query kind (denseQueryOf):
// structuredRegular volumes within one level-1 node carry no node-table
// query.
struct HitRenderLaunch
{
  const IteratorContextView *c;
  AttrView a;
  HitRenderArgs m;
  hipStream_t st;
  bool denseQuery;
  template <typename Src, int kFilter, int kQuery>
  hipError_t run() const
  {
    hipLaunchKernelGGL((kHitRender<Src, kFilter, kQuery>), dim3((m.numRays + kIterBlock - 1) / kIterBlock),
                       dim3(kIterBlock), 0, st, c, a, m);
    return hipGetLastError();
  }
  template <typename Src, int kFilter>
  hipError_t operator()() const
  {
    if constexpr (IsDenseSource<Src>::value)
      return denseQuery ? run<Src, kFilter, 1>() : run<Src, kFilter, 0>();
    else
      return run<Src, kFilter, 0>();
  }
};

}  // namespace vklhip
