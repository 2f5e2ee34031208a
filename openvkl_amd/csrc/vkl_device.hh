// Device functions of the HIP sampling / traversal path (gfx950).
//
// Numerics: compiled with -ffp-contract=off so every binary32 operation is
// rounded on its own, in the operation order of the reference ISPC sources
// cited below (files under openvkl/devices/cpu/). Nearest / linear samples,
// gradients and interval iteration are therefore bit-identical to the
// reference algorithm evaluated without FMA contraction; tricubic uses the
// separable Catmull-Rom form (mathematically equal to the Lekien-Marsden
// matrix on central-difference constraints; agrees to ~1e-6 relative).
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <type_traits>

#include "vkl_views.h"

namespace vklhip {

#define VKL_DEV __device__ __forceinline__

// ---- scalar helpers -----------------------------------------------------------

VKL_DEV float vmin(float a, float b) { return a < b ? a : b; }  // ISPC min
VKL_DEV float vmax(float a, float b) { return a > b ? a : b; }  // ISPC max
VKL_DEV float vinf() { return __int_as_float(0x7f800000); }

// rkcommon lerp: (1 - t) * a + t * b.
VKL_DEV float lerp(float t, float a, float b) { return (1.f - t) * a + t * b; }

// floor then float -> int32 with NaN / out-of-range -> INT32_MIN (the x86
// cvttss2si result the reference CPU device produces). The conversion floors
// and saturates by itself (below -2^31 to INT32_MIN), so only values from
// 2^31 on and NaN are left to a select: 3 instructions instead of 6, on three
// axes of every sample and of every DDA restart (with the 3 instead of 6
// compares of an interior stencil: a 1080p interval rendering of a 512^3
// float volume 4.91 -> 4.56 ms, a hit rendering 21.0 -> 20.6 ms).
VKL_DEV int32_t floorToInt(float f)
{
  int32_t i;
  asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(i) : "v"(f));
  return f < 2147483648.f ? i : INT32_MIN;
}

// Workgroup index remapped so each of the 8 XCDs (which take workgroups
// round-robin, b -> XCD b mod 8, each with its own L2) walks one contiguous
// band of the launch: neighbouring rays, which share voxel cache lines, then
// meet in one L2 instead of eight. A bijection on [0, 8 floor(n / 8)); the
// tail keeps its index.
VKL_DEV uint32_t xcdBandBlock(uint32_t b, uint32_t n)
{
  const uint32_t per = n / 8u;
  return b < per * 8u ? (b % 8u) * per + b / 8u : b;
}

// rkcommon divide_safe: 1 / x with |x| < FLT_MIN clamped to +-FLT_MIN.
VKL_DEV float divideSafe(float x)
{
  const float fltMin = 1.17549435e-38f;
  const float d      = (fabsf(x) < fltMin) ? (x >= 0.f ? fltMin : -fltMin) : x;
  return 1.f / d;
}

template <typename T>
VKL_DEV float toFloat(T v)
{
  return (float)v;
}
template <>
VKL_DEV float toFloat<__half>(__half v)
{
  return __half2float(v);
}

VKL_DEV float fetchAny(const void *p, uint32_t type, uint64_t i)
{
  switch (type) {
  case kTypeUchar: return (float)((const uint8_t *)p)[i];
  case kTypeShort: return (float)((const int16_t *)p)[i];
  case kTypeUshort: return (float)((const uint16_t *)p)[i];
  case kTypeHalf: return __half2float(((const __half *)p)[i]);
  case kTypeDouble: return (float)((const double *)p)[i];
  default: return ((const float *)p)[i];
  }
}

struct F3
{
  float x, y, z;
};
struct I3
{
  int32_t x, y, z;
};

// VdbGrid.h:56-89.
VKL_DEV F3 xfmVector(const float *M, F3 p)
{
  return {M[0] * p.x + M[1] * p.y + M[2] * p.z, M[3] * p.x + M[4] * p.y + M[5] * p.z,
          M[6] * p.x + M[7] * p.y + M[8] * p.z};
}
VKL_DEV F3 xfmPoint(const float *M, F3 p)
{
  const F3 r = xfmVector(M, p);
  return {r.x + M[9], r.y + M[10], r.z + M[11]};
}
VKL_DEV F3 xfmNormal(const float *MI, F3 p)
{
  return {MI[0] * p.x + MI[3] * p.y + MI[6] * p.z, MI[1] * p.x + MI[4] * p.y + MI[7] * p.z,
          MI[2] * p.x + MI[5] * p.y + MI[8] * p.z};
}

// vdb_topology.h.in:96-170: voxel index inside a level-l node, z fastest.
VKL_DEV uint32_t offsetToLinear(uint32_t l, uint32_t x, uint32_t y, uint32_t z)
{
  const uint32_t m = kRes[l] - 1, s = kTotalLogRes[l + 1], L = kLogRes[l];
  return (((x & m) >> s) << (2 * L)) + (((y & m) >> s) << L) + ((z & m) >> s);
}

// Reads through pointers that a kernel itself loads from memory (a context's
// arrays): the compiler knows neither their address space, which costs a
// generic load's bookkeeping, nor that a kernel's own stores leave them
// alone, without which a uniform read is a vector load.
template <typename T>
VKL_DEV T globalLoad(const T *p, uint64_t i)
{
  return reinterpret_cast<const __attribute__((address_space(1))) T *>(reinterpret_cast<uintptr_t>(p))[i];
}
template <typename T>
VKL_DEV T constantLoad(const T *p, int i)
{
  return reinterpret_cast<const __attribute__((address_space(4))) T *>(reinterpret_cast<uintptr_t>(p))[i];
}
VKL_DEV Range1f rangeLoad(const Range1f *p, uint64_t i)
{
  const uint64_t u = globalLoad(reinterpret_cast<const uint64_t *>(p), i);
  return {__uint_as_float((uint32_t)u), __uint_as_float((uint32_t)(u >> 32))};
}

// ---- voxel sources --------------------------------------------------------------

// Dense voxels (structuredRegular), VdbSampler_dense.ih:290-330 and
// VdbSampler_traverseAndSample.ih:314-349: out-of-domain corners read the
// background. Addressing per DenseLayout (x-fastest or brick-swizzled): each
// axis contributes an independent term, so the 8 trilinear corners cost 6
// axis terms and 8 adds.
// Element offset of root-relative voxel (x, y, z) under layout L.
VKL_DEV uint64_t denseOffset(const DenseLayout &L, uint32_t x, uint32_t y, uint32_t z)
{
  const uint32_t S = L.sx + L.sy + L.sz;
  return (((((uint64_t)(x >> L.sx)) << S) + (x & ((1u << L.sx) - 1))) << (L.cornerPacked ? 3 : 0)) +
         (uint64_t)(y >> L.sy) * L.strideY + ((y & ((1u << L.sy) - 1)) << L.sx) +
         (uint64_t)(z >> L.sz) * L.strideZ + ((z & ((1u << L.sz) - 1)) << (L.sx + L.sy));
}

// The 8 elements of a corner-packed cell record, one vector load.
template <typename T>
struct alignas(8 * sizeof(T)) CellRecord
{
  T v[8];
};

// N neighbouring voxels at base + byteOffset, one load.
template <typename T, int N>
struct VoxelRow
{
  T v[N];
};
template <typename T, int N>
VKL_DEV VoxelRow<T, N> loadRow(const T *base, uint32_t byteOffset)
{
  VoxelRow<T, N> r;
  __builtin_memcpy(&r, reinterpret_cast<const char *>(base) + byteOffset, sizeof(r));
  return r;
}

template <typename T, bool kIdx64>
struct DenseSource
{
  using Off = typename std::conditional<kIdx64, uint64_t, uint32_t>::type;
  const T *data;
  uint32_t nx, ny, nz;
  int32_t rx, ry, rz;
  uint32_t sx, sy, sz, S, pk;
  Off strideY, strideZ;
  bool rows;  // x-fastest layout with byte offsets below 2^32
  float bg;

  VKL_DEV DenseSource(const GridView &g, const AttrView &a, uint32_t = 0)
      : data((const T *)a.data),
        nx(g.activeSize[0]),
        ny(g.activeSize[1]),
        nz(g.activeSize[2]),
        rx(g.rootOrigin[0]),
        ry(g.rootOrigin[1]),
        rz(g.rootOrigin[2]),
        sx(g.layout.sx),
        sy(g.layout.sy),
        sz(g.layout.sz),
        S(g.layout.sx + g.layout.sy + g.layout.sz),
        pk(g.layout.cornerPacked ? 3u : 0u),
        strideY((Off)g.layout.strideY),
        strideZ((Off)g.layout.strideZ),
        rows(!(g.layout.sx | g.layout.sy | g.layout.sz | g.layout.cornerPacked) &&
             g.activeSize[2] * g.layout.strideZ <= (1ull << 32) / sizeof(T)),
        bg(a.background)
  {
  }

  VKL_DEV void setTime(float) {}  // temporally constant

  // x-fastest rows: a stencil's rows share one 32-bit byte offset (its first
  // voxel's) and differ in a wavefront-uniform base address, and the
  // neighbouring voxels of a row are one load of their total width (aligned
  // to the element only, which global loads take). It quarters the loads of
  // a tricubic stencil and most of the address arithmetic of both filters:
  // 2.1 M tricubic samples of a half slice 78.9 -> 45.0 us, a 1080p interval
  // rendering of a 512^3 float volume 6.67 -> 5.99 ms, 1080p Woodcock rays in
  // half voxels 3.27 -> 3.08 ms. Random points gain nothing (a point's rows
  // are in different cache lines either way).
  VKL_DEV uint32_t rowOffset(uint32_t x, uint32_t y, uint32_t z) const
  {
    return (x + y * (uint32_t)strideY + z * (uint32_t)strideZ) * (uint32_t)sizeof(T);
  }
  VKL_DEV static void rowPair(const T *base, uint32_t byteOffset, float &a, float &b)
  {
    const VoxelRow<T, 2> r = loadRow<T, 2>(base, byteOffset);
    a                      = toFloat(r.v[0]);
    b                      = toFloat(r.v[1]);
  }

  VKL_DEV Off xTerm(uint32_t x) const { return (((Off)(x >> sx) << S) | (Off)(x & ((1u << sx) - 1))) << pk; }
  VKL_DEV Off yTerm(uint32_t y) const
  {
    return (Off)(y >> sy) * strideY + (Off)((y & ((1u << sy) - 1)) << sx);
  }
  VKL_DEV Off zTerm(uint32_t z) const
  {
    return (Off)(z >> sz) * strideZ + (Off)((z & ((1u << sz) - 1)) << (sx + sy));
  }

  VKL_DEV float at(int32_t x, int32_t y, int32_t z) const
  {
    const uint32_t ox = (uint32_t)(x - rx), oy = (uint32_t)(y - ry), oz = (uint32_t)(z - rz);
    if (!(ox < nx && oy < ny && oz < nz)) return bg;
    return toFloat(data[xTerm(ox) + yTerm(oy) + zTerm(oz)]);
  }

  // Corners s[4x + 2y + z] of the cell at ic (VdbSampler_trilinear.ih:48-108):
  // one bounds test when the whole stencil is inside, else per corner.
  VKL_DEV void corners8(I3 ic, float *s) const
  {
    const uint32_t ox = (uint32_t)(ic.x - rx), oy = (uint32_t)(ic.y - ry), oz = (uint32_t)(ic.z - rz);
    if (ox < nx - 1u && oy < ny - 1u && oz < nz - 1u) {
      if (pk) {  // corner-packed: the cell record holds s[0..7]
        const CellRecord<T> c = *reinterpret_cast<const CellRecord<T> *>(data + xTerm(ox) + yTerm(oy) + zTerm(oz));
#pragma unroll
        for (int i = 0; i < 8; i++) s[i] = toFloat(c.v[i]);
        return;
      }
      if (rows) {  // x-fastest: the two corners of a row in one load
        const uint32_t o = rowOffset(ox, oy, oz);
        rowPair(data, o, s[0], s[4]);
        rowPair(data + strideY, o, s[2], s[6]);
        rowPair(data + strideZ, o, s[1], s[5]);
        rowPair(data + strideY + strideZ, o, s[3], s[7]);
        return;
      }
      const Off x0 = xTerm(ox), x1 = xTerm(ox + 1);
      const Off y0 = yTerm(oy), y1 = yTerm(oy + 1);
      const Off z0 = zTerm(oz), z1 = zTerm(oz + 1);
      const Off a00 = y0 + z0, a01 = y0 + z1, a10 = y1 + z0, a11 = y1 + z1;
      s[0] = toFloat(data[x0 + a00]);
      s[4] = toFloat(data[x1 + a00]);
      s[2] = toFloat(data[x0 + a10]);
      s[6] = toFloat(data[x1 + a10]);
      s[1] = toFloat(data[x0 + a01]);
      s[5] = toFloat(data[x1 + a01]);
      s[3] = toFloat(data[x0 + a11]);
      s[7] = toFloat(data[x1 + a11]);
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) s[i] = at(ic.x + ((i >> 2) & 1), ic.y + ((i >> 1) & 1), ic.z + (i & 1));
  }
};

// Sparse VDB node table (VdbSampler_traverseAndSample.ih:85-202,
// VdbSampleInner.ih.in:33-77). Leaf data is packed: dense leaves of 512
// z-fastest voxels, tiles of one value. kObserve: the sampler has a
// LeafNodeAccess observer; traversals record their leaf and the corner-packed
// cell records (which bypass traversal) are not used. A separate
// instantiation keeps the unobserved kernels free of the marking code, which
// costs the hit iterator about 27 VGPRs.
template <typename T, bool kObserve = false>
struct SparseSource
{
  LevelView lv[3];
  const uint64_t *leafSlot;
  const T *dense;
  const T *tile;
  const float *cells;         // corner-packed cell records (or null)
  const uint32_t *leafIndex;  // leaf cell -> dense-leaf slot (corner-packed)
  // The same leaf-index grid used as a flattened node table: with full-depth
  // sampling (no error voxels) a voxel of a dense leaf is found with one
  // lookup instead of a three-level traversal (null: traverse).
  const uint32_t *flatIndex;
  uint32_t *leafAccess;       // observed samplers: per leaf index, last access stamp
  int32_t root[3];
  uint32_t size[3];
  uint32_t ldim[3];
  uint32_t maxDepth, numAttr, attr, accessStamp;
  float bg;

  VKL_DEV SparseSource(const GridView &g, const AttrView &a, uint32_t attributeIndex)
      : leafSlot(g.leafSlot),
        dense((const T *)a.data),
        tile((const T *)a.tile),
        cells(!kObserve && g.maxSamplingDepth == g.packedDepth ? a.cells : nullptr),
        leafIndex(g.leafIndex),
        flatIndex(!kObserve && g.maxSamplingDepth >= 3u ? g.leafIndex : nullptr),
        leafAccess(g.leafAccess),
        maxDepth(g.maxSamplingDepth),
        numAttr(g.numAttributes),
        attr(attributeIndex),
        accessStamp(g.accessStamp),
        bg(a.background)
  {
#pragma unroll
    for (int i = 0; i < 3; i++) {
      lv[i]   = g.levels[i];
      root[i] = g.rootOrigin[i];
      size[i] = g.activeSize[i];
      ldim[i] = g.leafDims[i];
    }
  }

  // Voxel code for an in-domain root-relative offset; error voxels report
  // their level's value ranges and voxel offset (VdbSampleInner.ih.in:46-54).
  // The three levels are written out: a loop over lv[l] that the compiler
  // does not unroll indexes lv at run time, which places the whole source in
  // scratch memory.
  VKL_DEV uint64_t traverse(uint32_t ox, uint32_t oy, uint32_t oz, const Range1f *&errRanges, uint32_t &errOffset) const
  {
    const uint32_t vo0 = (uint32_t)offsetToLinear(0, ox, oy, oz);
    const uint64_t v0  = globalLoad(lv[0].voxels, vo0);
    if (((uint32_t)v0 & 3u) >= 2u && maxDepth < 1u) return stop(lv[0].valueRange, vo0, errRanges, errOffset);
    if (((uint32_t)v0 & 3u) != 2u) return found(v0);
    const uint32_t vo1 = (uint32_t)((v0 >> 2) * kNumVoxels[1]) + offsetToLinear(1, ox, oy, oz);
    const uint64_t v1  = globalLoad(lv[1].voxels, vo1);
    if (((uint32_t)v1 & 3u) >= 2u && maxDepth < 2u) return stop(lv[1].valueRange, vo1, errRanges, errOffset);
    if (((uint32_t)v1 & 3u) != 2u) return found(v1);
    const uint32_t vo2 = (uint32_t)((v1 >> 2) * kNumVoxels[2]) + offsetToLinear(2, ox, oy, oz);
    const uint64_t v2  = globalLoad(lv[2].voxels, vo2);
    if (((uint32_t)v2 & 3u) >= 2u && maxDepth < 3u) return stop(lv[2].valueRange, vo2, errRanges, errOffset);
    return found(v2);
  }

  // Error voxel: the stopping level's value ranges and the voxel offset.
  VKL_DEV static uint64_t stop(const Range1f *ranges, uint32_t vo, const Range1f *&errRanges, uint32_t &errOffset)
  {
    errRanges = ranges;
    errOffset = vo;
    return 1u;
  }

  // Leaf access observation (VdbSampleInner.ih.in:69-74): every traversal
  // that ends on a leaf pointer records the leaf index. Concurrent lanes
  // store the same stamp, so the races are benign.
  VKL_DEV uint64_t found(uint64_t v) const
  {
    if (kObserve && ((uint32_t)v & 3u) == 3u && leafAccess) leafAccess[v >> 6] = accessStamp;
    return v;
  }

  VKL_DEV void setTime(float) {}  // temporally constant

  VKL_DEV uint64_t slotOf(uint64_t v) const { return leafSlot ? leafSlot[v >> 6] : (v >> 6); }

  VKL_DEV float errorValue(const Range1f *er, uint32_t eo) const
  {
    const Range1f r = er[(uint64_t)eo * numAttr + attr];
    return 0.5f * (r.lower + r.upper);
  }

  VKL_DEV float leafValue(uint64_t v, uint32_t ox, uint32_t oy, uint32_t oz) const
  {
    const uint64_t leaf = slotOf(v);
    if (((v >> 2) & 3u) == 1u) return toFloat(dense[leaf * 512u + (((ox & 7u) << 6) | ((oy & 7u) << 3) | (oz & 7u))]);
    return toFloat(tile[leaf]);
  }

  VKL_DEV bool inDomain(uint32_t ox, uint32_t oy, uint32_t oz) const
  {
    return ox < size[0] && oy < size[1] && oz < size[2];
  }

  // Leaf index grid entry of the 8^3 leaf cell holding root-relative voxel
  // (ox, oy, oz): a dense-leaf slot, kLeafEmpty or kLeafTraverse.
  VKL_DEV uint32_t flatSlot(uint32_t ox, uint32_t oy, uint32_t oz) const
  {
    return globalLoad(flatIndex, ((uint64_t)(oz >> 3) * ldim[1] + (oy >> 3)) * ldim[0] + (ox >> 3));
  }

  // VdbSampler_sample_inner, VdbSampler_traverseAndSample.ih:144-197.
  VKL_DEV float at(int32_t x, int32_t y, int32_t z) const
  {
    const uint32_t ox = (uint32_t)(x - root[0]), oy = (uint32_t)(y - root[1]), oz = (uint32_t)(z - root[2]);
    if (!inDomain(ox, oy, oz)) return bg;
    if (flatIndex) {
      const uint32_t slot = flatSlot(ox, oy, oz);
      if (slot < kLeafTraverse)
        return toFloat(dense[(uint64_t)slot * 512u + (((ox & 7u) << 6) | ((oy & 7u) << 3) | (oz & 7u))]);
      if (slot == kLeafEmpty) return 0.f;  // in the domain, covered by no node
    }
    const Range1f *er  = nullptr;
    uint32_t eo        = 0;
    const uint64_t v   = traverse(ox, oy, oz, er, eo);
    const uint32_t tag = (uint32_t)v & 3u;
    if (tag == 3u) return leafValue(v, ox, oy, oz);
    if (tag == 1u) return errorValue(er, eo);
    return 0.f;
  }

  // Corner-packed volumes: a cell inside a dense leaf reads its record (the
  // 8 values at() returns for its corners, baked at commit). Otherwise, when
  // the 2x2x2 stencil lies in one leaf (7/8 per axis), one traversal serves
  // all corners; the values equal eight separate traversals.
  VKL_DEV void corners8(I3 ic, float *s) const
  {
    const uint32_t ox = (uint32_t)(ic.x - root[0]), oy = (uint32_t)(ic.y - root[1]), oz = (uint32_t)(ic.z - root[2]);
    if (cells && inDomain(ox, oy, oz)) {
      const uint32_t slot = globalLoad(leafIndex, ((uint64_t)(oz >> 3) * ldim[1] + (oy >> 3)) * ldim[0] + (ox >> 3));
      if (slot < kLeafTraverse) {
        const CellRecord<float> c = *reinterpret_cast<const CellRecord<float> *>(
            cells + ((uint64_t)slot * 512u + (((ox & 7u) << 6) | ((oy & 7u) << 3) | (oz & 7u))) * 8u);
#pragma unroll
        for (int i = 0; i < 8; i++) s[i] = c.v[i];
        return;
      }
    }
    if (inDomain(ox, oy, oz) && inDomain(ox + 1, oy + 1, oz + 1) && (ox & 7u) != 7u && (oy & 7u) != 7u &&
        (oz & 7u) != 7u) {
      if (flatIndex) {
        const uint32_t slot = flatSlot(ox, oy, oz);
        if (slot < kLeafTraverse) {
          leafCorners(((uint64_t)slot << 6) | 7u, nullptr, 0, ox, oy, oz, s, true);
          return;
        }
        if (slot == kLeafEmpty) {  // the stencil lies in one empty cell
#pragma unroll
          for (int i = 0; i < 8; i++) s[i] = 0.f;
          return;
        }
      }
      const Range1f *er = nullptr;
      uint32_t eo       = 0;
      const uint64_t v  = traverse(ox, oy, oz, er, eo);
      leafCorners(v, er, eo, ox, oy, oz, s);
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) s[i] = at(ic.x + ((i >> 2) & 1), ic.y + ((i >> 1) & 1), ic.z + (i & 1));
  }

  // The 8 corners of a stencil inside one 8^3 leaf cell, given that cell's
  // traversal result.
  // slotCode: v carries the dense-leaf slot itself (from the flattened
  // index), not a leaf index to map through leafSlot.
  VKL_DEV void leafCorners(uint64_t v, const Range1f *er, uint32_t eo, uint32_t ox, uint32_t oy, uint32_t oz,
                           float *s, bool slotCode = false) const
  {
    const uint32_t tag = (uint32_t)v & 3u;
    if (tag == 3u && ((v >> 2) & 3u) == 1u) {
      const uint64_t slot = slotCode ? (v >> 6) : slotOf(v);
      const T *p = dense + slot * 512u + (((ox & 7u) << 6) | ((oy & 7u) << 3) | (oz & 7u));
      // z-fastest: the two corners of a row in one load.
      constexpr uint32_t kRow[4] = {0, 8, 64, 72};
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const VoxelRow<T, 2> r = loadRow<T, 2>(p, kRow[i] * (uint32_t)sizeof(T));
        s[2 * i]               = toFloat(r.v[0]);
        s[2 * i + 1]           = toFloat(r.v[1]);
      }
      return;
    }
    const float c = (tag == 3u) ? toFloat(tile[slotOf(v)]) : (tag == 1u) ? errorValue(er, eo) : 0.f;
#pragma unroll
    for (int i = 0; i < 8; i++) s[i] = c;
  }
};

// interpolateTemporallyStructured, temporal_data_interpolation.ih:13-45:
// voxel v owns samples [steps * v, steps * v + steps) of data. Time is
// clamped to [0, 1] (NaN to 0), which keeps both reads among the voxel's own
// samples; inside [0, 1] this is the reference's arithmetic.
template <typename T>
VKL_DEV float temporallyStructured(const T *data, uint32_t steps, uint64_t v, float time)
{
  const float tc      = vmin(vmax(time, 0.f), 1.f);
  const float tf      = tc * (float)(steps - 1);
  const uint32_t ts   = (uint32_t)tf;
  const float w       = tf - (float)ts;
  const uint32_t next = (w == 0.f) ? ts : ts + 1;
  const uint64_t base = (uint64_t)steps * v;
  return (1.f - w) * toFloat(data[base + ts]) + w * toFloat(data[base + next]);
}

// interpolateTemporallyUnstructured, temporal_data_interpolation.ih:82-152:
// voxel v owns positions [idx[v], idx[v + 1]) of data and times.
template <typename T, typename I>
VKL_DEV float temporallyUnstructured(const T *data, const I *idx, const float *times, uint64_t v, float time)
{
  const uint64_t i0 = idx[v], i1 = idx[v + 1];
  const float t0    = times[i0];
  if (time <= t0) return toFloat(data[i0]);
  const float t1 = times[i1 - 1];
  if (time >= t1) return toFloat(data[i1 - 1]);
  if (isnan(time)) return time;
  const uint64_t n = i1 - i0;
  if (n == 2) {
    const float w = (time - t0) * (1.f / (t1 - t0));
    return (1.f - w) * toFloat(data[i0]) + w * toFloat(data[i1 - 1]);
  }
  // Binary search for [times[lower], times[upper]] around time. Commit
  // checked that the voxel's times increase strictly, so with
  // t0 < time < t1 every read stays inside the voxel's range and the search
  // ends within log2(n) + 1 rounds; the bound and the clamps only guard it.
  uint64_t lower = 0, upper = n;
  bool found     = false;
  for (int it = 0; it < 66 && lower <= upper; ++it) {
    const uint64_t mid = (lower + upper) / 2;
    const float tm     = times[i0 + mid];
    const uint64_t nx1 = i0 + mid + 1 < i1 ? i0 + mid + 1 : i1 - 1;
    if (time >= tm && time <= times[nx1]) {
      lower = i0 + mid;
      upper = lower + 1 < i1 ? lower + 1 : i1 - 1;
      found = true;
      break;
    } else if (time < tm) {
      upper = mid;
    } else {
      lower = mid;
    }
  }
  if (!found) return __int_as_float(0x7fc00000);
  const float tl = times[lower], th = times[upper];
  const float w  = (time - tl) * (1.f / (th - tl));
  return (1.f - w) * toFloat(data[lower]) + w * toFloat(data[upper]);
}

// structuredRegular with temporal data (temporal_data_interpolation.ih:13-152,
// VdbSampler_dense.ih:360-560): every voxel read interpolates that voxel's
// time samples at the source's current time (setTime; 0 by default, as for
// calls without times). Voxels are x-fastest (temporal volumes have no bricks
// or corner packing).
template <typename T>
struct TemporalDenseSource
{
  const T *data;
  const uint32_t *idx32;
  const uint64_t *idx64;
  const float *times;
  uint32_t nx, ny, nz;
  int32_t rx, ry, rz;
  uint32_t format, numTimesteps;
  float bg, time;

  VKL_DEV TemporalDenseSource(const GridView &g, const AttrView &a, uint32_t = 0)
      : data((const T *)a.data),
        idx32(g.tuIndex64 ? nullptr : (const uint32_t *)g.tuIndices),
        idx64(g.tuIndex64 ? (const uint64_t *)g.tuIndices : nullptr),
        times(g.tuTimes),
        nx(g.activeSize[0]),
        ny(g.activeSize[1]),
        nz(g.activeSize[2]),
        rx(g.rootOrigin[0]),
        ry(g.rootOrigin[1]),
        rz(g.rootOrigin[2]),
        format(g.temporalFormat),
        numTimesteps(g.numTimesteps),
        bg(a.background),
        time(0.f)
  {
  }

  VKL_DEV void setTime(float t) { time = t; }

  // The voxel with linear index v at the current time.
  VKL_DEV float voxel(uint64_t v) const
  {
    if (format == 1u) return temporallyStructured(data, numTimesteps, v, time);
    if (idx64) return temporallyUnstructured(data, idx64, times, v, time);
    return temporallyUnstructured(data, idx32, times, v, time);
  }

  VKL_DEV float at(int32_t x, int32_t y, int32_t z) const
  {
    const uint32_t ox = (uint32_t)(x - rx), oy = (uint32_t)(y - ry), oz = (uint32_t)(z - rz);
    if (!(ox < nx && oy < ny && oz < nz)) return bg;
    return voxel(((uint64_t)oz * ny + oy) * nx + ox);
  }

  // Structured time steps, stencil inside the domain: the step and weight are
  // the same for every voxel, so the 8 corners are 8 independent loads of two
  // neighbouring steps each (temporallyStructured's arithmetic). Otherwise a
  // rolled loop: one inlined copy of the time interpolation per stencil
  // instead of eight. 2^20 random points at random times in 160 x 144 x 131
  // floats of 4 steps: 157 -> 95 us (117 us with the x neighbours four loads
  // apart, when the second one is fetched again).
  VKL_DEV void corners8(I3 ic, float *s) const
  {
    const uint32_t ox = (uint32_t)(ic.x - rx), oy = (uint32_t)(ic.y - ry), oz = (uint32_t)(ic.z - rz);
    if (format == 1u && numTimesteps > 1u && ox < nx - 1u && oy < ny - 1u && oz < nz - 1u) {
      const float tf       = vmin(vmax(time, 0.f), 1.f) * (float)(numTimesteps - 1u);
      const uint32_t ts    = (uint32_t)tf;
      const float w        = tf - (float)ts;
      const uint32_t next  = (w == 0.f) ? ts : ts + 1u;
      const uint32_t first = ts < numTimesteps - 2u ? ts : numTimesteps - 2u;  // both steps are in the pair from here
      const uint64_t v     = ((uint64_t)oz * ny + oy) * nx + ox;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int i       = (k >> 1) | ((k & 1) << 2);  // x neighbours, mostly one cache line, in turn
        const uint64_t vi = v + ((i & 1) ? (uint64_t)nx * ny : 0u) + ((i & 2) ? nx : 0u) + ((i & 4) ? 1u : 0u);
        const VoxelRow<T, 2> r = loadRow<T, 2>(data + (vi * numTimesteps + first), 0);
        const float a = toFloat(r.v[0]), b = toFloat(r.v[1]);
        s[i] = (1.f - w) * (ts == first ? a : b) + w * (next == first ? a : b);
      }
      return;
    }
#pragma unroll 1
    for (int i = 0; i < 8; i++) s[i] = at(ic.x + ((i >> 2) & 1), ic.y + ((i >> 1) & 1), ic.z + (i & 1));
  }
};

// vdb with temporal leaves (VdbSampler_denseZYX.ih / VdbSampler_tile.ih,
// structured and unstructured sampling): the node table is traversed as for
// constant leaves; a leaf pointer's temporal format selects how its voxel is
// read at the source's current time. The traversal records leaf accesses
// when the sampler is observed.
template <typename T>
struct TemporalSparseSource
{
  SparseSource<T, true> nodes;
  const T *data;
  const uint64_t *dataOff, *idxOff, *timesOff, *idx;
  const uint32_t *steps;
  const float *times;
  float time;

  VKL_DEV TemporalSparseSource(const GridView &g, const AttrView &a, uint32_t attributeIndex)
      : nodes(g, a, attributeIndex),
        data((const T *)a.data),
        dataOff(g.leafDataOffset),
        idxOff(g.leafIdxOffset),
        timesOff(g.leafTimesOffset),
        idx((const uint64_t *)g.tuIndices),
        steps(g.leafSteps),
        times(g.tuTimes),
        time(0.f)
  {
    nodes.cells = nullptr;
  }

  VKL_DEV void setTime(float t) { time = t; }

  // Leaf voxel (ox, oy, oz) of the leaf pointer v (tiles: their one voxel).
  VKL_DEV float leafValue(uint64_t v, uint32_t ox, uint32_t oy, uint32_t oz) const
  {
    const uint64_t leaf = v >> 6;
    const uint32_t tf   = (uint32_t)(v >> 4) & 3u;
    const uint64_t vi   = (((v >> 2) & 3u) == 1u) ? (((ox & 7u) << 6) | ((oy & 7u) << 3) | (oz & 7u)) : 0u;
    const T *d          = data + dataOff[leaf];
    if (tf == 1u) return temporallyStructured(d, steps[leaf], vi, time);
    if (tf == 2u) return temporallyUnstructured(d, idx + idxOff[leaf], times + timesOff[leaf], vi, time);
    return toFloat(d[vi]);
  }

  VKL_DEV float at(int32_t x, int32_t y, int32_t z) const
  {
    const uint32_t ox = (uint32_t)(x - nodes.root[0]), oy = (uint32_t)(y - nodes.root[1]),
                   oz = (uint32_t)(z - nodes.root[2]);
    if (!nodes.inDomain(ox, oy, oz)) return nodes.bg;
    const Range1f *er = nullptr;
    uint32_t eo       = 0;
    const uint64_t v  = nodes.traverse(ox, oy, oz, er, eo);
    const uint32_t tag = (uint32_t)v & 3u;
    if (tag == 3u) return leafValue(v, ox, oy, oz);
    if (tag == 1u) return nodes.errorValue(er, eo);
    return 0.f;
  }

  VKL_DEV void corners8(I3 ic, float *s) const
  {
#pragma unroll 1
    for (int i = 0; i < 8; i++) s[i] = at(ic.x + ((i >> 2) & 1), ic.y + ((i >> 1) & 1), ic.z + (i & 1));
  }
};

template <typename T>
VKL_DEV void cubicTaps(const TemporalSparseSource<T> &src, I3 ic, float *S)
{
#pragma unroll 1
  for (int i = 0; i < 64; i++) S[i] = src.at(ic.x + (i >> 4) - 1, ic.y + ((i >> 2) & 3) - 1, ic.z + (i & 3) - 1);
}

// Whether dense offsets (including brick padding) can exceed 32 bits.
VKL_DEV bool denseNeeds64(const GridView &g)
{
  const uint64_t nbz = ((uint64_t)g.activeSize[2] + (1u << g.layout.sz) - 1) >> g.layout.sz;
  return nbz * g.layout.strideZ >= (1ull << 32);
}

// ---- filters ------------------------------------------------------------------

// VdbSampler_nearest.ih:25-57: +0.5 for vertex-centered data.
template <typename Src>
VKL_DEV float sampleNearest(const Src &src, F3 p, float off)
{
  return src.at(floorToInt(p.x + off), floorToInt(p.y + off), floorToInt(p.z + off));
}

// VdbSampler_trilinear.ih:378-399.
template <typename Src>
VKL_DEV float sampleLinear(const Src &src, F3 p)
{
  const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
  const F3 d  = {p.x - (float)ic.x, p.y - (float)ic.y, p.z - (float)ic.z};
  float s[8];
  src.corners8(ic, s);
  return lerp(d.x, lerp(d.y, lerp(d.z, s[0], s[1]), lerp(d.z, s[2], s[3])),
              lerp(d.y, lerp(d.z, s[4], s[5]), lerp(d.z, s[6], s[7])));
}

// VdbSampler_trilinear.ih:751-780 (index-space gradient).
template <typename Src>
VKL_DEV F3 gradientLinear(const Src &src, F3 p)
{
  const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
  const F3 d  = {p.x - (float)ic.x, p.y - (float)ic.y, p.z - (float)ic.z};
  float s[8];
  src.corners8(ic, s);
  F3 r;
  r.x = lerp(d.y, lerp(d.z, s[4] - s[0], s[5] - s[1]), lerp(d.z, s[6] - s[2], s[7] - s[3]));
  r.y = lerp(d.x, lerp(d.z, s[2] - s[0], s[3] - s[1]), lerp(d.z, s[6] - s[4], s[7] - s[5]));
  r.z = lerp(d.x, lerp(d.y, s[1] - s[0], s[3] - s[2]), lerp(d.y, s[5] - s[4], s[7] - s[6]));
  return r;
}

// Catmull-Rom weights for taps -1, 0, 1, 2 at offset t in [0, 1), and their
// derivatives. The tensor product of these equals the tricubic interpolant
// of VdbSampler_tricubic.ih:34-578 (Hermite on central differences).
VKL_DEV void crWeights(float t, float *w)
{
  const float t2 = t * t, t3 = t2 * t;
  w[0] = 0.5f * (-t3 + 2.f * t2 - t);
  w[1] = 0.5f * (3.f * t3 - 5.f * t2 + 2.f);
  w[2] = 0.5f * (-3.f * t3 + 4.f * t2 + t);
  w[3] = 0.5f * (t3 - t2);
}
VKL_DEV void crDerivWeights(float t, float *w)
{
  const float t2 = t * t;
  w[0] = 0.5f * (-3.f * t2 + 4.f * t - 1.f);
  w[1] = 0.5f * (9.f * t2 - 10.f * t);
  w[2] = 0.5f * (-9.f * t2 + 8.f * t + 1.f);
  w[3] = 0.5f * (3.f * t2 - 2.f * t);
}

template <typename Src>
VKL_DEV void cubicTaps(const Src &src, I3 ic, float *S)
{
#pragma unroll
  for (int i = 0; i < 64; i++) S[i] = src.at(ic.x + (i >> 4) - 1, ic.y + ((i >> 2) & 3) - 1, ic.z + (i & 3) - 1);
}

// Corner-packed dense volumes: the 4x4x4 stencil is 8 cell records (cells at
// ic - 1 + 2 (a, b, c)) when it lies inside the domain; same values as 64
// single reads.
template <typename T, bool kIdx64>
VKL_DEV void cubicTaps(const DenseSource<T, kIdx64> &src, I3 ic, float *S)
{
  const uint32_t ox = (uint32_t)(ic.x - src.rx), oy = (uint32_t)(ic.y - src.ry), oz = (uint32_t)(ic.z - src.rz);
  if (src.pk && ox - 1 < src.nx && ox + 2 < src.nx && oy - 1 < src.ny && oy + 2 < src.ny && oz - 1 < src.nz &&
      oz + 2 < src.nz) {
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const uint32_t a = (c >> 2) & 1, b = (c >> 1) & 1, d = c & 1;
      const CellRecord<T> r = *reinterpret_cast<const CellRecord<T> *>(
          src.data + src.xTerm(ox - 1 + 2 * a) + src.yTerm(oy - 1 + 2 * b) + src.zTerm(oz - 1 + 2 * d));
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const uint32_t i = 2 * a + ((k >> 2) & 1), j = 2 * b + ((k >> 1) & 1), l = 2 * d + (k & 1);
        S[16 * i + 4 * j + l] = toFloat(r.v[k]);
      }
    }
    return;
  }
  if (src.rows && ox - 1 < src.nx && ox + 2 < src.nx && oy - 1 < src.ny && oy + 2 < src.ny && oz - 1 < src.nz &&
      oz + 2 < src.nz) {
    // x-fastest: 16 rows of 4 voxels, one load each.
    const uint32_t o = src.rowOffset(ox - 1, oy - 1, oz - 1);
#pragma unroll
    for (int l = 0; l < 4; l++)
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const VoxelRow<T, 4> r = loadRow<T, 4>(src.data + j * src.strideY + l * src.strideZ, o);
#pragma unroll
        for (int i = 0; i < 4; i++) S[16 * i + 4 * j + l] = toFloat(r.v[i]);
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < 64; i++) S[i] = src.at(ic.x + (i >> 4) - 1, ic.y + ((i >> 2) & 3) - 1, ic.z + (i & 3) - 1);
}

// vdb volumes with the flattened leaf index (unobserved, full sampling
// depth): a stencil inside the domain touches at most 2 leaf cells per axis,
// so their 8 index entries are read once and each tap reads its leaf
// directly, instead of one index lookup per tap; the taps equal 64 at()
// calls (dense leaf: its voxel; a cell no node covers: 0). A stencil that
// leaves the domain or meets a tile / error cell takes the 64 at() calls.
template <typename T, bool kObserve>
VKL_DEV void cubicTapsByLeafCells(const SparseSource<T, kObserve> &src, I3 ic, float *S)
{
  const uint32_t ox = (uint32_t)(ic.x - 1 - src.root[0]), oy = (uint32_t)(ic.y - 1 - src.root[1]),
                 oz = (uint32_t)(ic.z - 1 - src.root[2]);
  if (src.flatIndex && src.inDomain(ox, oy, oz) && src.inDomain(ox + 3, oy + 3, oz + 3)) {
    const uint32_t cx0 = ox >> 3, cy0 = oy >> 3, cz0 = oz >> 3;
    const uint32_t cx1 = (ox + 3) >> 3, cy1 = (oy + 3) >> 3, cz1 = (oz + 3) >> 3;
    uint32_t slot[8];
    bool traverse = false;
#pragma unroll
    for (int c = 0; c < 8; c++) {
      const uint32_t cx = (c & 4) ? cx1 : cx0, cy = (c & 2) ? cy1 : cy0, cz = (c & 1) ? cz1 : cz0;
      slot[c]  = src.flatIndex[((uint64_t)cz * src.ldim[1] + cy) * src.ldim[0] + cx];
      traverse = traverse || slot[c] == kLeafTraverse;
    }
    if (!traverse) {
      // The cell of each tap by selects (constant register indices only).
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t x  = ox + i;
        const bool hx     = (x >> 3) != cx0;
        const uint32_t t0 = hx ? slot[4] : slot[0], t1 = hx ? slot[5] : slot[1];
        const uint32_t t2 = hx ? slot[6] : slot[2], t3 = hx ? slot[7] : slot[3];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const uint32_t y  = oy + j;
          const bool hy     = (y >> 3) != cy0;
          const uint32_t u0 = hy ? t2 : t0, u1 = hy ? t3 : t1;
#pragma unroll
          for (int k = 0; k < 4; k++) {
            const uint32_t z  = oz + k;
            const uint32_t sl = (z >> 3) != cz0 ? u1 : u0;
            S[16 * i + 4 * j + k] =
                sl == kLeafEmpty
                    ? 0.f
                    : toFloat(src.dense[(uint64_t)sl * 512u + (((x & 7u) << 6) | ((y & 7u) << 3) | (z & 7u))]);
          }
        }
      }
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < 64; i++) S[i] = src.at(ic.x + (i >> 4) - 1, ic.y + ((i >> 2) & 3) - 1, ic.z + (i & 3) - 1);
}

// Temporal volumes: the 64 reads are a rolled loop. Each read interpolates in
// time (a binary search for unstructured data), and 64 inlined copies of that
// make the kernels that sample them several times larger.
template <typename T>
VKL_DEV void cubicTaps(const TemporalDenseSource<T> &src, I3 ic, float *S)
{
#pragma unroll 1
  for (int i = 0; i < 64; i++) S[i] = src.at(ic.x + (i >> 4) - 1, ic.y + ((i >> 2) & 3) - 1, ic.z + (i & 3) - 1);
}

// The tricubic interpolant at index-space point p from its 64 taps
// S[16 i + 4 j + l] = voxel ic + (i - 1, j - 1, l - 1), ic = floor(p).
VKL_DEV float cubicFromTaps(const float *S, F3 p, I3 ic)
{
  float wx[4], wy[4], wz[4];
  crWeights(p.x - (float)ic.x, wx);
  crWeights(p.y - (float)ic.y, wy);
  crWeights(p.z - (float)ic.z, wz);
  float r = 0.f;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float ry = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float *q = S + 16 * i + 4 * j;
      ry += wy[j] * (wz[0] * q[0] + wz[1] * q[1] + wz[2] * q[2] + wz[3] * q[3]);
    }
    r += wx[i] * ry;
  }
  return r;
}

// Its index-space gradient, from the same taps.
VKL_DEV F3 cubicGradientFromTaps(const float *S, F3 p, I3 ic)
{
  float wx[4], wy[4], wz[4], dx[4], dy[4], dz[4];
  const F3 d = {p.x - (float)ic.x, p.y - (float)ic.y, p.z - (float)ic.z};
  crWeights(d.x, wx);
  crWeights(d.y, wy);
  crWeights(d.z, wz);
  crDerivWeights(d.x, dx);
  crDerivWeights(d.y, dy);
  crDerivWeights(d.z, dz);
  F3 g = {0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    float gy_v = 0.f, gy_dy = 0.f, gy_dz = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float *q = S + 16 * i + 4 * j;
      const float vz = wz[0] * q[0] + wz[1] * q[1] + wz[2] * q[2] + wz[3] * q[3];
      const float dzv = dz[0] * q[0] + dz[1] * q[1] + dz[2] * q[2] + dz[3] * q[3];
      gy_v += wy[j] * vz;
      gy_dy += dy[j] * vz;
      gy_dz += wy[j] * dzv;
    }
    g.x += dx[i] * gy_v;
    g.y += wx[i] * gy_dy;
    g.z += wx[i] * gy_dz;
  }
  return g;
}

template <typename Src>
VKL_DEV float sampleCubic(const Src &src, F3 p)
{
  const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
  float S[64];
  cubicTaps(src, ic, S);
  return cubicFromTaps(S, p, ic);
}

template <typename Src>
VKL_DEV F3 gradientCubic(const Src &src, F3 p)
{
  const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
  float S[64];
  cubicTaps(src, ic, S);
  return cubicGradientFromTaps(S, p, ic);
}

// Whether a source's voxels are plain loads, which a stencil can hold many of;
// a vdb or temporal voxel is a search of its own.
template <typename Src>
struct PlainVoxels : std::false_type
{
};
template <typename T, bool kIdx64>
struct PlainVoxels<DenseSource<T, kIdx64>> : std::true_type
{
};

// gradientCubic with one x slice of the stencil (16 taps) alive at a time, or
// on vdb and temporal sources one tap: the same sums in the same order. For
// kernels that keep much state of their own across the call, where 64 live
// taps would push that state to scratch. 16 unrolled searches of a vdb do that
// as well, whether the call is reached or not (300 bytes a lane of the hit
// renderer, now 36): 1080p hit rendering of a 512^3 float shell with linear
// gradients 145 -> 49 ms. Plain voxels keep the slices: 6.5 ms a 960 x 540
// image with tricubic normals against 8.4 tap by tap.
template <typename Src>
VKL_DEV F3 gradientCubicBySlices(const Src &src, F3 p)
{
  constexpr int kUnroll = PlainVoxels<Src>::value ? 4 : 1;
  const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
  const F3 d  = {p.x - (float)ic.x, p.y - (float)ic.y, p.z - (float)ic.z};
  float wx[4], wy[4], wz[4], dx[4], dy[4], dz[4];
  crWeights(d.x, wx);
  crWeights(d.y, wy);
  crWeights(d.z, wz);
  crDerivWeights(d.x, dx);
  crDerivWeights(d.y, dy);
  crDerivWeights(d.z, dz);
  const auto pick = [](const float *w, int i) { return i == 0 ? w[0] : i == 1 ? w[1] : i == 2 ? w[2] : w[3]; };
  F3 g = {0.f, 0.f, 0.f};
#pragma unroll 1
  for (int i = 0; i < 4; i++) {
    float gy_v = 0.f, gy_dy = 0.f, gy_dz = 0.f;
#pragma unroll kUnroll
    for (int j = 0; j < 4; j++) {
      float vz = 0.f, dzv = 0.f;
#pragma unroll kUnroll
      for (int k = 0; k < 4; k++) {
        const float q = src.at(ic.x + i - 1, ic.y + j - 1, ic.z + k - 1);
        vz            = k ? vz + pick(wz, k) * q : pick(wz, k) * q;
        dzv           = k ? dzv + pick(dz, k) * q : pick(dz, k) * q;
      }
      gy_v += pick(wy, j) * vz;
      gy_dy += pick(dy, j) * vz;
      gy_dz += pick(wy, j) * dzv;
    }
    g.x += pick(dx, i) * gy_v;
    g.y += pick(wx, i) * gy_dy;
    g.z += pick(wx, i) * gy_dz;
  }
  return g;
}

// Tricubic in the stream kernels (kSample, kGradient): vdb sources gather
// their taps by leaf cells (cubicTapsByLeafCells). The fused ray and
// iterator kernels keep the per-tap reads of sampleCubic: inlined at their
// several sampler call sites, the unrolled gather makes those kernels'
// compilation take tens of minutes.
template <typename Src>
struct GathersByLeafCells : std::false_type
{
};
template <typename T, bool kObserve>
struct GathersByLeafCells<SparseSource<T, kObserve>> : std::true_type
{
};

template <typename Src>
VKL_DEV float sampleCubicStream(const Src &src, F3 p)
{
  if constexpr (GathersByLeafCells<Src>::value) {
    const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
    float S[64];
    cubicTapsByLeafCells(src, ic, S);
    return cubicFromTaps(S, p, ic);
  } else {
    return sampleCubic(src, p);
  }
}

template <typename Src>
VKL_DEV F3 gradientCubicStream(const Src &src, F3 p)
{
  if constexpr (GathersByLeafCells<Src>::value) {
    const I3 ic = {floorToInt(p.x), floorToInt(p.y), floorToInt(p.z)};
    float S[64];
    cubicTapsByLeafCells(src, ic, S);
    return cubicGradientFromTaps(S, p, ic);
  } else {
    return gradientCubic(src, p);
  }
}

template <typename Src>
VKL_DEV float sampleFiltered(const Src &src, int filter, F3 p, float nearestOffset)
{
  if (filter == kFilterNearest) return sampleNearest(src, p, nearestOffset);
  if (filter == kFilterCubic) return sampleCubic(src, p);
  return sampleLinear(src, p);
}

// Hit iteration descends to depth 2 on structuredRegular volumes and 3 on vdb
// volumes (HitIteratorContext::commit, IteratorContext.cpp:285-336).
template <typename S>
struct IsDenseSource : std::false_type
{
};
template <typename T, bool B>
struct IsDenseSource<DenseSource<T, B>> : std::true_type
{
};
template <typename T>
struct IsDenseSource<TemporalDenseSource<T>> : std::true_type
{
};
template <typename Src>
constexpr int hitDepthOf()
{
  return IsDenseSource<Src>::value ? 2 : 3;
}

// Object-space sample with one source type and filter per instantiation (the
// sampler entry of VdbSampler_iterator_computeSample_varying,
// VdbSampler.ispc:341-374). Every caller gets its own inlined copy: the
// library has no non-inlined device functions, because branch relaxation in
// a large callee on gfx950 rewrote the return-address register pair s[30:31]
// for its long jumps, which sent the callee's return back into its own body.
template <typename Src, int kFilter>
struct PointSampler
{
  using Source = Src;
  Src src;
  const float *o2i;
  float noff;

  VKL_DEV PointSampler(const GridView &g, const AttrView &a, uint32_t attr)
      : src(g, a, attr), o2i(g.o2i), noff(g.constantCellData ? 0.f : 0.5f)
  {
  }

  VKL_DEV void setTime(float t) { src.setTime(t); }

  VKL_DEV float operator()(F3 oc) const
  {
    const F3 p = xfmPoint(o2i, oc);
    if (kFilter == kFilterNearest) return sampleNearest(src, p, noff);
    if (kFilter == kFilterCubic) return sampleCubic(src, p);
    return sampleLinear(src, p);
  }
};

// ---- interval iteration (VdbIterator.ispc:36-180, Dda.ih, HDDA.ih.in,
//      VdbQueryVoxel.ih.in, VdbQueryVoxelDense.ih) -----------------------------

VKL_DEV int dirSign(float v) { return ((int)(0 < v)) - ((int)(v < 0)); }
VKL_DEV float dirRcp(float v) { return (v == 0) ? vinf() : divideSafe(v); }

// Dda.ih:66-84.
VKL_DEV float planeT(float plane, float org, float inv)
{
  const float t = (plane - org) * inv;
  return (plane == org || isnan(t)) ? vinf() : t;
}

// Dda.ih:127-140.
VKL_DEV int32_t clampCell(float f, int32_t res) { return floorToInt(vmax(f, 0.f)) & ~(res - 1); }

constexpr uint32_t kMaxDdaSteps = 1u << 22;

// Lanes of a wavefront that wait for the interval phase of hitTick, times
// this, against the lanes that have a sample to take. 1080p hit rendering of
// 256 x 240 x 220 floats: 18.4 ms at 3, 19.7 at 1, 18.7 at 2, 18.4 at 6; hit
// batches in dense and vdb volumes 0-10 % slower at 1, the same at 2 and 6.
constexpr uint32_t kHitIntervalVote = 3;

#define DX(l) (l)
#define DY(l) (4 + (l))
#define DZ(l) (8 + (l))

// Every DDA routine below indexes the state arrays with compile-time
// constants (levels are template arguments or fully unrolled loop indices):
// an array indexed at run time is placed in scratch memory, which costs the
// iterators several times their voxel traffic.

// Per-axis step of the level-L cells: tDelta = res * |1 / dir| (Dda.ih:184-186).
template <int L>
VKL_DEV float ddaTDelta(const DdaState &d, int axis)
{
  return (float)kRes[L + 1] * d.absRcp[axis];
}

// The DDA's deepest level: kDepth when the caller knows it at compile time
// (hit iteration: 2 on structuredRegular, 3 on vdb), else d.level.
template <int kDepth>
VKL_DEV uint32_t ddaLevel(const DdaState &d)
{
  return kDepth >= 0 ? (uint32_t)kDepth : d.level;
}

// Dda.ih:145-196.
template <int kDepth = -1>
VKL_DEV void ddaInit(DdaState &d, F3 org, F3 dir, float tMin, uint32_t level)
{
  const F3 oo = {org.x + tMin * dir.x, org.y + tMin * dir.y, org.z + tMin * dir.z};
  const int sx = dirSign(dir.x), sy = dirSign(dir.y), sz = dirSign(dir.z);
  const F3 id = {dirRcp(dir.x), dirRcp(dir.y), dirRcp(dir.z)};
  d.level     = level < 3u ? level : 3u;
  d.t         = tMin;
  d.rayOrg[0] = org.x;
  d.rayOrg[1] = org.y;
  d.rayOrg[2] = org.z;
  d.rayDir[0] = dir.x;
  d.rayDir[1] = dir.y;
  d.rayDir[2] = dir.z;
  d.absRcp[0] = fabsf(id.x);
  d.absRcp[1] = fabsf(id.y);
  d.absRcp[2] = fabsf(id.z);
  // Levels below d.level are never read; they are written as 0 so that no
  // earlier state stays live through a re-initialisation.
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    const bool used   = (uint32_t)l <= ddaLevel<kDepth>(d);
    const int32_t res = (int32_t)kRes[l + 1];
    const int32_t ix = clampCell(oo.x, res), iy = clampCell(oo.y, res), iz = clampCell(oo.z, res);
    d.idx[DX(l)]   = used ? ix : 0;
    d.idx[DY(l)]   = used ? iy : 0;
    d.idx[DZ(l)]   = used ? iz : 0;
    d.tNext[DX(l)] = used ? planeT((float)(ix + res * (sx >= 0)), org.x, id.x) : 0.f;
    d.tNext[DY(l)] = used ? planeT((float)(iy + res * (sy >= 0)), org.y, id.y) : 0.f;
    d.tNext[DZ(l)] = used ? planeT((float)(iz + res * (sz >= 0)), org.z, id.z) : 0.f;
  }
}

// Signed 1 / dir of an axis as dirRcp gives it, from its stored magnitude.
VKL_DEV float ddaRcp(const DdaState &d, int axis)
{
  return d.rayDir[axis] < 0.f ? -d.absRcp[axis] : d.absRcp[axis];
}

// Dda.ih:271-309 (ties: x, then y, then z). Returns the axis along which the
// cell moved (z when it did not).
template <int L>
VKL_DEV int ddaStep(DdaState &d)
{
  // Every field is written on every path (values selected, not addresses),
  // so the state stays in registers.
  const float tx = d.tNext[DX(L)], ty = d.tNext[DY(L)], tz = d.tNext[DZ(L)];
  const float minT  = vmin(vmin(tx, ty), tz);
  const int32_t res = (int32_t)kRes[L + 1];
  const bool sx     = minT == tx;
  const bool sy     = !sx && minT == ty;
  const bool sz     = !sx && !sy;
  d.t               = sx ? tx : (sy ? ty : tz);
  d.tNext[DX(L)]    = sx ? tx + ddaTDelta<L>(d, 0) : tx;
  d.tNext[DY(L)]    = sy ? ty + ddaTDelta<L>(d, 1) : ty;
  d.tNext[DZ(L)]    = sz ? tz + ddaTDelta<L>(d, 2) : tz;
  const int32_t mx  = sx ? dirSign(d.rayDir[0]) * res : 0;
  const int32_t my  = sy ? dirSign(d.rayDir[1]) * res : 0;
  d.idx[DX(L)]      = d.idx[DX(L)] + mx;
  d.idx[DY(L)]      = d.idx[DY(L)] + my;
  d.idx[DZ(L)]      = d.idx[DZ(L)] + (sz ? dirSign(d.rayDir[2]) * res : 0);
  return mx ? 0 : (my ? 1 : 2);
}

// Level l restarts at the position oo (Dda.ih:235-260).
template <int l>
VKL_DEV void ddaReinitLevel(DdaState &d, F3 oo)
{
  const int32_t res = (int32_t)kRes[l + 1];
  d.idx[DX(l)]      = clampCell(oo.x, res);
  d.idx[DY(l)]      = clampCell(oo.y, res);
  d.idx[DZ(l)]      = clampCell(oo.z, res);
  d.tNext[DX(l)]    = planeT((float)(d.idx[DX(l)] + (d.rayDir[0] < 0.f ? 0 : res)), d.rayOrg[0], ddaRcp(d, 0));
  d.tNext[DY(l)]    = planeT((float)(d.idx[DY(l)] + (d.rayDir[1] < 0.f ? 0 : res)), d.rayOrg[1], ddaRcp(d, 1));
  d.tNext[DZ(l)]    = planeT((float)(d.idx[DZ(l)] + (d.rayDir[2] < 0.f ? 0 : res)), d.rayOrg[2], ddaRcp(d, 2));
}

// HDDA.ih.in:52-101, parents of the stepped level L from the nearest one up:
// each one steps only if its child left its cell.
template <int P>
VKL_DEV void hddaParents(DdaState &d, uint32_t L)
{
  if constexpr (P >= 0) {
    bool follow = true;
    if ((uint32_t)P < L) {
      constexpr int C   = P + 1;
      const int32_t res = (int32_t)kRes[P + 1];
      follow = d.idx[DX(C)] < d.idx[DX(P)] || d.idx[DY(C)] < d.idx[DY(P)] || d.idx[DZ(C)] < d.idx[DZ(P)] ||
               d.idx[DX(C)] >= d.idx[DX(P)] + res || d.idx[DY(C)] >= d.idx[DY(P)] + res ||
               d.idx[DZ(C)] >= d.idx[DZ(P)] + res;
      if (follow) (void)ddaStep<P>(d);
    }
    if (follow) hddaParents<P - 1>(d, L);
  }
}

// HDDA.ih.in:24-101: step on level L (the level of the empty voxel, never
// deeper than the DDA's deepest), re-initialise the levels below from the
// current t nudged 1e-2 across the plane the step crossed (Dda.ih:204-266),
// and let parents follow a child that left their cell. Only the step itself
// is a switch over the level; the re-initialisation of a level and the
// parents' steps each have one body that lanes stepping on different levels
// share, because the lanes of a wavefront rarely step on the same level (with
// a body per level, 3 to 9 of 64 lanes were active).
template <int kDepth>
VKL_DEV void hddaStep(DdaState &d, uint32_t L)
{
  constexpr int kMax = kDepth >= 0 ? kDepth : 3;
  int axis;
  if (L == 0)
    axis = ddaStep<0>(d);
  else if (kMax >= 2 && L == 1)
    axis = ddaStep<(kMax < 1 ? kMax : 1)>(d);
  else if (kMax >= 3 && L == 2)
    axis = ddaStep<(kMax < 2 ? kMax : 2)>(d);
  else
    axis = ddaStep<kMax>(d);
  if (L < ddaLevel<kDepth>(d)) {
    F3 oo = {d.rayOrg[0] + d.t * d.rayDir[0], d.rayOrg[1] + d.t * d.rayDir[1], d.rayOrg[2] + d.t * d.rayDir[2]};
    if (axis == 0)
      oo.x = oo.x + (float)dirSign(d.rayDir[0]) * 1e-2f;
    else if (axis == 1)
      oo.y = oo.y + (float)dirSign(d.rayDir[1]) * 1e-2f;
    else
      oo.z = oo.z + (float)dirSign(d.rayDir[2]) * 1e-2f;
    if (kMax >= 1 && L < 1 && 1 <= ddaLevel<kDepth>(d)) ddaReinitLevel<1>(d, oo);
    if (kMax >= 2 && L < 2 && 2 <= ddaLevel<kDepth>(d)) ddaReinitLevel<2>(d, oo);
    if (kMax >= 3 && L < 3 && 3 <= ddaLevel<kDepth>(d)) ddaReinitLevel<3>(d, oo);
  }
  hddaParents<kMax - 1>(d, L);
}

// Pins a value to a register: the optimizer can no longer turn a select
// between array elements into a load from a selected address (a run-time
// array index, which sends the whole array to scratch memory).
VKL_DEV int32_t opaque(int32_t v)
{
  asm volatile("" : "+v"(v));
  return v;
}

// The cell of the DDA's deepest level, selected without a run-time array
// index.
template <int kDepth>
VKL_DEV I3 ddaCell(const DdaState &d)
{
  if constexpr (kDepth >= 0) return I3{d.idx[DX(kDepth)], d.idx[DY(kDepth)], d.idx[DZ(kDepth)]};
  I3 c = {opaque(d.idx[DX(0)]), opaque(d.idx[DY(0)]), opaque(d.idx[DZ(0)])};
#pragma unroll
  for (int l = 1; l < 4; ++l) {
    const I3 cl = {opaque(d.idx[DX(l)]), opaque(d.idx[DY(l)]), opaque(d.idx[DZ(l)])};
    if (d.level == (uint32_t)l) c = cl;
  }
  return c;
}

// ValueRanges.ih:22-52. The reads are uniform. The first two ranges, mostly the
// only ones, are tested without a vote, which costs a short walk 3 to 7 %; the
// loop over more ends with the last lane that is still open: intervals of
// 100 k rays in a 512^3 float shell with 200 ranges at depth 2 / 3, 0.26 /
// 0.40 ms, without an exit 3.57 / 4.76 ms.
VKL_DEV bool rangesOverlap(const IteratorContextView &c, Range1f r)
{
  if (c.numRanges == 0) return true;
  const float *q  = &c.ranges->lower;
  const auto test = [&](int i) { return constantLoad(q, 2 * i + 1) >= r.lower && constantLoad(q, 2 * i) <= r.upper; };
  bool any        = test(0);
  const bool in   = c.rangesMinMax.upper >= r.lower && c.rangesMinMax.lower <= r.upper;
  if (c.numRanges > 1) {
    any = any || test(1);
    for (int i = 2; i < c.numRanges && __ballot(in && !any) != 0; i++) any = any || test(i);
  }
  return any && in;
}

struct VoxelDesc
{
  uint32_t level;
  bool isEmpty;
  Range1f valueRange;
};

// Level L of a node-table query (VdbQueryVoxel.ih.in:42-116): describes the
// voxel of node `node` that holds (x, y, z); true with its child in `node` when
// the query goes on below it.
template <int L>
VKL_DEV bool queryLevel(const IteratorContextView &c, int32_t x, int32_t y, int32_t z, uint32_t depth,
                        VoxelDesc &desc, uint32_t &node)
{
  const GridView &g = c.sampler.grid;
  const uint32_t vo = offsetToLinear(L, (uint32_t)x, (uint32_t)y, (uint32_t)z) + node * (uint32_t)kNumVoxels[L];
  const uint64_t v  = globalLoad(g.levels[L].voxels, vo);
  desc.valueRange   = rangeLoad(g.levels[L].valueRange, (uint64_t)vo * g.numAttributes + c.attributeIndex);
  desc.level        = L;
  desc.isEmpty      = ((v & 3u) == 0u) || !rangesOverlap(c, desc.valueRange);
  if (desc.isEmpty) return false;
  const bool atDepth = (uint32_t)(L + 1) > depth;
  const bool isLeaf  = (v & 3u) == 3u;
  if (isLeaf && !atDepth) desc.level = L + 1;
  node = (uint32_t)(v >> 2);
  return L < 2 && !(atDepth || isLeaf);
}

// VdbQueryVoxel.ih.in:42-116. With kNodeCache, a query in the 128^3 block
// of the previous query's level-2 node starts at level 2 (it.ck / it.cnode):
// the level-0 and level-1 voxels on the way there, and so their outcome, are
// the same. Hit iteration uses it (+7 % on the 4096^3 vdb); plain interval
// iteration does not (its kernel runs 11 % slower with the extra state).
// The levels are written out: as a loop, lanes entering it at different levels
// made the level a per-lane value, and every level's pointers and sizes were
// loaded from memory before its voxel. Together with the typed loads above
// that took 13 % off interval batches in a 1024^3 shell and 6 % off hit batches
// there, and the selector's typed loads 7 and 4 % off the 1080p hit and interval
// renderers.
template <bool kNodeCache>
VKL_DEV void queryVoxel(const IteratorContextView &c, int32_t x, int32_t y, int32_t z, uint32_t depth,
                        VoxelDesc &desc, IntervalState &it)
{
  uint32_t node    = 0;
  const int32_t kx = x >> 7, ky = y >> 7, kz = z >> 7;
  if (kNodeCache && it.ck[0] == kx && it.ck[1] == ky && it.ck[2] == kz) {
    node = it.cnode;
  } else {
    if (!queryLevel<0>(c, x, y, z, depth, desc, node)) return;
    if (!queryLevel<1>(c, x, y, z, depth, desc, node)) return;
    if (kNodeCache) {
      it.ck[0] = kx;
      it.ck[1] = ky;
      it.ck[2] = kz;
      it.cnode = node;
    }
  }
  (void)queryLevel<2>(c, x, y, z, depth, desc, node);
}
// VdbQueryVoxelDense.ih:115-164 (nodes numbered x-fastest, one level-1 node).
VKL_DEV void queryVoxelDense(const IteratorContextView &c, int32_t x, int32_t y, int32_t z, uint32_t depth,
                             VoxelDesc &desc)
{
  const GridView &g = c.sampler.grid;
  desc.level        = depth;
  const uint32_t ox = (uint32_t)x, oy = (uint32_t)y, oz = (uint32_t)z;
  if (!(ox < g.activeSize[0] && oy < g.activeSize[1] && oz < g.activeSize[2])) {
    desc.isEmpty = true;
    return;
  }
  const uint64_t n1x = (g.activeSize[0] + kRes[1] - 1) >> kTotalLogRes[1];
  const uint64_t n1y = (g.activeSize[1] + kRes[1] - 1) >> kTotalLogRes[1];
  const uint64_t l1  = (uint64_t)(oz >> kTotalLogRes[1]) * n1y * n1x + (uint64_t)(oy >> kTotalLogRes[1]) * n1x +
                      (ox >> kTotalLogRes[1]);
  uint64_t vi;
  int lvl;
  if (depth >= 2) {
    const uint64_t n2x = (g.activeSize[0] + kRes[2] - 1) >> kTotalLogRes[2];
    const uint64_t n2y = (g.activeSize[1] + kRes[2] - 1) >> kTotalLogRes[2];
    const uint64_t l2  = (uint64_t)(oz >> kTotalLogRes[2]) * n2y * n2x + (uint64_t)(oy >> kTotalLogRes[2]) * n2x +
                        (ox >> kTotalLogRes[2]);
    vi  = l1 * kNumVoxels[1] + l2 * kNumVoxels[2] + offsetToLinear(2, ox, oy, oz);
    lvl = 2;
  } else if (depth == 1) {
    vi  = l1 * kNumVoxels[1] + offsetToLinear(1, ox, oy, oz);
    lvl = 1;
  } else {
    vi  = offsetToLinear(0, ox, oy, oz);
    lvl = 0;
  }
  desc.valueRange = rangeLoad(g.levels[lvl].valueRange, vi * g.numAttributes + c.attributeIndex);
  desc.isEmpty    = !rangesOverlap(c, desc.valueRange);
}

// box_utility.ih:62-75.
VKL_DEV Range1f intersectBox(F3 org, F3 dir, const float *box, Range1f lim)
{
  const F3 inv  = {divideSafe(dir.x), divideSafe(dir.y), divideSafe(dir.z)};
  const F3 mins = {(box[0] - org.x) * inv.x, (box[1] - org.y) * inv.y, (box[2] - org.z) * inv.z};
  const F3 maxs = {(box[3] - org.x) * inv.x, (box[4] - org.y) * inv.y, (box[5] - org.z) * inv.z};
  Range1f r;
  r.lower = vmax(vmax(vmin(mins.x, maxs.x), vmin(mins.y, maxs.y)), vmax(vmin(mins.z, maxs.z), lim.lower));
  r.upper = vmin(vmin(vmax(mins.x, maxs.x), vmax(mins.y, maxs.y)), vmin(vmax(mins.z, maxs.z), lim.upper));
  return r;
}

// VdbIterator_Initialize, VdbIterator.ispc:36-94.
template <int kDepth = -1>
VKL_DEV void intervalInit(const IteratorContextView &c, IntervalState &it, F3 origin, F3 direction, Range1f tRange)
{
  const GridView &g = c.sampler.grid;
  const F3 o        = xfmPoint(g.o2i, origin);
  const F3 org      = {o.x - (float)g.rootOrigin[0], o.y - (float)g.rootOrigin[1], o.z - (float)g.rootOrigin[2]};
  const F3 dir      = xfmVector(g.o2i, direction);
  it.nominalDeltaT  = vmin(vmin(1.f * divideSafe(fabsf(dir.x)), 1.f * divideSafe(fabsf(dir.y))),
                          1.f * divideSafe(fabsf(dir.z)));
  it.ck[0] = it.ck[1] = it.ck[2] = INT32_MIN;
  it.cnode = 0;
  const Range1f ti = intersectBox(org, dir, g.domainBox, tRange);
  // A ray that misses the box gets tMax = -inf (and t = 0), which ends its
  // iteration; the DDA is initialised either way so that every field of the
  // state is written on both paths.
  const bool miss = ti.upper <= ti.lower;
  it.tMax         = miss ? -vinf() : ti.upper;
  ddaInit<kDepth>(it.dda, org, dir, miss ? 0.f : ti.lower, c.maxIteratorDepth);
}

// Whether a context's queries use the dense node numbering: dense node
// indices assume one level-1 node (VdbQueryVoxelDense.ih:48-57); larger
// volumes use the general query, which stays inside the node table.
VKL_DEV bool denseQuery(const GridView &g)
{
  return g.dense != 0 && g.activeSize[0] <= kRes[1] && g.activeSize[1] <= kRes[1] && g.activeSize[2] <= kRes[1];
}

// What an interval walk keeps beside the state of the caller.
struct IntervalWalk
{
  uint32_t steps;    // voxels visited since the last interval
  bool inLeaf;       // depth 3: the next cell lies in the leaf of the last query,
  Range1f leafRange;  // whose value range this is

  VKL_DEV IntervalWalk() : steps(0), inLeaf(false), leafRange{0.f, 0.f} {}
};

// One voxel of VdbIterator_iterateIntervalInternal (VdbIterator.ispc:96-159):
// 0 the voxel was empty, 1 `out` holds its interval, 2 the ray has ended.
// The lanes of a wavefront take one voxel each per call, and there is one
// query and one DDA step for empty and occupied voxels alike, so lanes with
// an interval do not wait for the ones still crossing empty space. kQuery: 0
// the general query, 1 the dense one, -1 chosen per context at run time.
template <bool kNodeCache, int kDepth, int kQuery>
VKL_DEV int intervalTick(const IteratorContextView &c, IntervalState &it, IntervalWalk &w, IntervalOut &out)
{
  DdaState &dda = it.dda;
  // Every step advances t by a positive tDelta; a ray whose steps make no
  // progress (infinite direction components) is ended after kMaxDdaSteps.
  if (!(dda.t <= it.tMax) || ++w.steps > kMaxDdaSteps) return 2;
  const I3 cell = ddaCell<kDepth>(dda);
  VoxelDesc v{3u, false, w.leafRange};
  if (kDepth != 3 || !w.inLeaf) {
    const uint32_t l = ddaLevel<kDepth>(dda);
    if (kQuery >= 0 ? kQuery == 1 : denseQuery(c.sampler.grid))
      queryVoxelDense(c, cell.x, cell.y, cell.z, l, v);
    else
      queryVoxel<kNodeCache>(c, cell.x, cell.y, cell.z, l, v, it);
  }
  const float tLower = dda.t;
  hddaStep<kDepth>(dda, v.level);
  if (kDepth == 3) {
    // The voxels of a leaf share one query result (its majorant). The dense
    // query calls cells outside the volume empty, and a volume's upper faces
    // may cut a leaf: there the next cell has to lie inside, too.
    const I3 to = ddaCell<kDepth>(dda);
    w.inLeaf    = !v.isEmpty && v.level == 3u &&
               (uint32_t)((cell.x ^ to.x) | (cell.y ^ to.y) | (cell.z ^ to.z)) < kRes[3];
    if (kQuery >= 0 ? kQuery == 1 : denseQuery(c.sampler.grid)) {
      const uint32_t *n = c.sampler.grid.activeSize;
      w.inLeaf          = w.inLeaf && (uint32_t)to.x < n[0] && (uint32_t)to.y < n[1] && (uint32_t)to.z < n[2];
    }
    w.leafRange = v.valueRange;
  }
  if (v.isEmpty) return 0;
  if (!(tLower < it.tMax)) return 2;
  w.steps           = 0;
  out.vLower        = v.valueRange.lower;
  out.vUpper        = v.valueRange.upper;
  out.tLower        = tLower;
  out.tUpper        = vmin(dda.t, it.tMax);
  out.nominalDeltaT = it.nominalDeltaT;
  return 1;
}

// The next interval of one ray.
template <bool kNodeCache = false, int kDepth = -1, int kQuery = -1>
VKL_DEV bool intervalNext(const IteratorContextView &c, IntervalState &it, IntervalOut &out)
{
  IntervalWalk w;
  int event;
  do
    event = intervalTick<kNodeCache, kDepth, kQuery>(c, it, w, out);
  while (event == 0);
  if (event == 2) it.tMax = -vinf();
  return event == 1;
}

// ---- hit iteration (DefaultIterator.ispc:141-258, Iterator.ih:17-200) --------

template <typename S>
VKL_DEV float sampleAlong(const S &smp, F3 o, F3 d, float t)
{
  return smp(F3{o.x + t * d.x, o.y + t * d.y, o.z + t * d.z});
}

template <int kDepth = -1>
VKL_DEV void hitInit(const IteratorContextView &c, HitState &h, F3 origin, F3 direction, Range1f tRange, float time)
{
  intervalInit<kDepth>(c, h.iv, origin, direction, tRange);
  h.origin[0] = origin.x;
  h.origin[1] = origin.y;
  h.origin[2] = origin.z;
  h.direction[0] = direction.x;
  h.direction[1] = direction.y;
  h.direction[2] = direction.z;
  h.time             = time;
  h.curLower         = 1.f;  // resetInterval, Interval.ih:15-22
  h.curUpper         = -1.f;
  h.curNominalDeltaT = 0.f;
  h.lastHitOffsetT   = -vinf();
}

// A ray's hit iteration as a state machine that advances one voxel query or
// one sample at a time (hitTick). The lanes of a wavefront are in different
// phases of the reference's nested loops (intervals, the march through one,
// bisection) most of the time; run as nested loops, every lane waits for the
// longest inner loop of its wavefront (3.3 of 64 lanes active on a 1024^3
// vdb, 8.7 in the hit renderer). Here every lane advances at each tick, all
// samples (start, march, bisection) share one sampler call, and the kernels
// hold one copy of the query, the DDA step and the sampler.
struct HitSearch
{
  HitState h;
  uint32_t mode;      // what the ray waits for
  uint32_t tries;     // NaN retries or bisection probes done
  IntervalWalk walk;
  float tp;           // position of the pending sample
  float t0, s0;       // start of the march step and its sample
  float tKnown;       // position s0 was taken at
  float t;            // end of the march step
  // What only a bisection keeps from tick to tick, one LDS word each at
  // bisect[word * kHitLanes] (in registers these 10 words cost the kernels an
  // occupancy step or as much scratch).
  float *bisect;
};

constexpr uint32_t kHitLanes = 64;  // lanes of a block that searches
enum : uint32_t
{
  kBisT0    = 0,  // the bracket and its samples
  kBisS0    = 1,
  kBisT1    = 2,
  kBisS1    = 3,
  kBisTol   = 4,
  kBisTs    = 5,  // position and value of the march sample
  kBisS     = 6,
  kBisHit   = 7,  // nearest hit of the step so far and its iso value
  kBisValue = 8,
  kBisIso   = 9,  // index of the iso value being bisected
  kBisWords = 10
};

enum : uint32_t
{
  kHitInterval = 0,  // the next interval
  kHitStart    = 1,  // the sample at the start of a range
  kHitMarch    = 2,  // the sample at the end of a march step
  kHitBisect   = 3,  // a bisection probe
  kHitDone     = 4,
};

// Start or resume the search of h (DefaultIterator.ispc:186-200).
VKL_DEV void hitResume(HitSearch &q)
{
  q.tries = 0;
  q.t0 = q.tp = q.h.curLower;
  q.mode      = q.h.curLower == vinf() ? kHitDone : (q.h.curUpper <= q.h.curLower ? kHitInterval : kHitStart);
}

// `bisect`: the lane's first word of kBisWords * kHitLanes floats of LDS.
VKL_DEV void hitBegin(HitSearch &q, float *bisect)
{
  q.walk   = IntervalWalk();
  q.bisect = bisect;
  q.tKnown = __builtin_nanf("");
  q.s0     = 0.f;
  hitResume(q);
}

// The next march step from (t0, s0), Iterator.ih:113-125; past the range's
// end, or without float progress, the next interval.
VKL_DEV void hitMarch(HitSearch &q)
{
  q.t     = q.t0 + vmin(q.h.iv.nominalDeltaT, q.h.curUpper - q.t0);
  q.tp    = q.t;
  q.tries = 0;
  q.mode  = kHitMarch;
  if (!(q.t0 < q.h.curUpper && q.t > q.t0)) {
    q.h.curLower = vinf();
    q.mode       = kHitInterval;
  }
}

// One tick; every lane of the wavefront that still searches calls it
// together. 0: still searching, 1: `hit` holds the next hit, 2: no more hits.
template <typename S, int kQuery = -1>
VKL_DEV int hitTick(const IteratorContextView &c, const S &smp, HitSearch &q, HitOut &hit)
{
  constexpr int kDepth = hitDepthOf<typename S::Source>();
  HitState &h          = q.h;
  int event            = 0;
  if (q.mode == kHitDone || c.numValues == 0) return 2;

  // The interval phase runs for a wavefront once a quarter of its searching
  // lanes wait for it (or none has a sample to take): running it for one or
  // two lanes costs as many instructions as for all.
  const uint32_t waiting = (uint32_t)__popcll(__ballot(q.mode == kHitInterval));
  const uint32_t others  = (uint32_t)__popcll(__ballot(q.mode != kHitInterval));
  if (waiting * kHitIntervalVote >= others) {
    if (q.mode == kHitInterval) {
      IntervalOut iv;
      const int found = intervalTick<true, kDepth, kQuery>(c, h.iv, q.walk, iv);
      if (found == 2) event = 2;
      if (found == 1) {
        h.curLower         = vmax(iv.tLower, h.lastHitOffsetT);
        h.curUpper         = iv.tUpper;
        h.curNominalDeltaT = iv.nominalDeltaT;  // the caller's state; the search reads iv's
        if (!(h.curUpper <= h.curLower)) {
          // Adjoining ranges share their end sample.
          q.t0    = h.curLower;
          q.tp    = h.curLower;
          q.tries = 0;
          q.mode  = kHitStart;
          if (q.t0 == q.tKnown && !isnan(q.s0)) hitMarch(q);
        }
      }
    }
  }

  // The sample phase: the sample each lane waits for, and what follows
  // from it (bisect and intersectSurfacesBisection, Iterator.ih:23-197).
  if (event == 0 && q.mode != kHitInterval) {
    const F3 o      = {h.origin[0], h.origin[1], h.origin[2]};
    const F3 d      = {h.direction[0], h.direction[1], h.direction[2]};
    const float sm  = sampleAlong(smp, o, d, q.tp);
    const float tHi = h.curUpper, step = h.iv.nominalDeltaT;
    float *bis      = q.bisect;
    bool compare = false, resumed = false, go = false;
    // The march sample under comparison, the nearest hit so far.
    float ts = q.tp, s = sm, tHit = vinf(), value = vinf();
    int iso = 0;
    if (q.mode == kHitBisect) {
      float b0 = bis[kBisT0 * kHitLanes], c0 = bis[kBisS0 * kHitLanes];
      float b1 = bis[kBisT1 * kHitLanes], c1 = bis[kBisS1 * kHitLanes];
      iso         = __float_as_int(bis[kBisIso * kHitLanes]);
      const float v = c.values[iso];
      float tIso    = vinf();
      bool more     = false;
      if (isnan(sm)) {
        tIso = (fabsf(v - c0) < fabsf(v - c1)) ? b0 : b1;
      } else if (sm == v || (v - c0) * (v - sm) < 0.f) {
        b1   = q.tp;
        c1   = sm;
        more = true;
      } else if (c1 == v || (v - c1) * (v - sm) < 0.f) {
        b0   = q.tp;
        c0   = sm;
        more = true;
      }
      if (more) {
        tIso = q.tp;
        more = ++q.tries < 10u;
        if (more) {
          q.tp = 0.5f * (b0 + b1);
          if (0.5f * (b1 - b0) < bis[kBisTol * kHitLanes]) {
            tIso = q.tp;
            more = false;
          }
        }
      }
      if (more) {
        bis[kBisT0 * kHitLanes] = b0;
        bis[kBisS0 * kHitLanes] = c0;
        bis[kBisT1 * kHitLanes] = b1;
        bis[kBisS1 * kHitLanes] = c1;
      } else {
        ts    = bis[kBisTs * kHitLanes];
        s     = bis[kBisS * kHitLanes];
        tHit  = bis[kBisHit * kHitLanes];
        value = bis[kBisValue * kHitLanes];
        if (tIso < tHit && tIso <= tHi) {
          tHit  = tIso;
          value = v;
        }
        compare = resumed = true;
      }
    } else if (isnan(sm) && q.tries < 10u && (q.mode == kHitStart ? q.t0 < tHi : ts > q.t0)) {
      const float nudge = vmax(1e-5f, 1e-5f * step);
      q.tries++;
      q.tp = q.mode == kHitStart ? q.t0 + nudge : ts - nudge;
      if (q.mode == kHitStart) q.t0 = q.tp;
    } else if (q.mode == kHitStart) {
      q.s0     = sm;
      q.tKnown = q.t0;
      go       = true;
    } else {
      compare = true;
    }
    if (compare) {
      for (int i = 0; i < c.numValues; i++) {
        const float v = constantLoad(c.values, i);
        if (!compare || i < iso) continue;
        if (!(resumed && i == iso)) {
          if (fabsf(q.s0 - v) < 1e-6f) {
            if (q.t0 < tHit && q.t0 <= tHi) {
              tHit  = q.t0;
              value = v;
            }
          } else if (!isnan(q.s0 + s) && (v - q.s0) * (v - s) < 0.f) {
            const float tol = vmin(1e-6f, 0.01f * vmin(step, tHi - q.t0));
            q.tp            = 0.5f * (q.t0 + ts);
            if (0.5f * (ts - q.t0) < tol) {
              if (q.tp < tHit && q.tp <= tHi) {
                tHit  = q.tp;
                value = v;
              }
            } else {
              bis[kBisT0 * kHitLanes]    = q.t0;
              bis[kBisS0 * kHitLanes]    = q.s0;
              bis[kBisT1 * kHitLanes]    = ts;
              bis[kBisS1 * kHitLanes]    = s;
              bis[kBisTol * kHitLanes]   = tol;
              bis[kBisTs * kHitLanes]    = ts;
              bis[kBisS * kHitLanes]     = s;
              bis[kBisHit * kHitLanes]   = tHit;
              bis[kBisValue * kHitLanes] = value;
              bis[kBisIso * kHitLanes]   = __int_as_float(i);
              q.tries = 0;
              q.mode  = kHitBisect;
              compare = false;
              continue;
            }
          }
        }
        if (q.t == tHi && fabsf(s - v) < 1e-6f) {
          if (ts < tHit && ts <= tHi) {
            tHit  = ts;
            value = v;
          }
        }
      }
    }
    if (compare) {
      if (tHit < vinf()) {
        hit.t            = tHit;
        hit.sample       = value;
        hit.epsilon      = 0.125f * step * sqrtf(d.x * d.x + d.y * d.y + d.z * d.z);
        h.curLower       = hit.t + hit.epsilon;
        h.lastHitOffsetT = hit.t + hit.epsilon;
        hitResume(q);
        event = 1;
      } else {
        q.t0     = q.t;
        q.s0     = s;
        q.tKnown = ts;
        go       = true;
      }
    }
    if (go) hitMarch(q);
  }
  return event;
}

// DefaultHitIterator_iterateHit, DefaultIterator.ispc:168-258, for one ray.
template <typename S, int kQuery = -1>
VKL_DEV bool hitNext(const IteratorContextView &c, const S &smp, HitState &h, HitOut &hit)
{
  float bisect[kBisWords * kHitLanes];  // registers: every index is constant
  HitSearch q;
  q.h = h;
  hitBegin(q, bisect);
  int event;
  do
    event = hitTick<S, kQuery>(c, smp, q, hit);
  while (event == 0);
  if (event == 2) q.h.curLower = vinf();
  h = q.h;
  return event == 1;
}

}  // namespace vklhip
