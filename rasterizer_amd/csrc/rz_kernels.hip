// gfx950 kernels of the occlusion-culling rasterizer.
//
// Pipeline of one draw (a frame of items, or a single rasterize call):
//   rz_prep_kernel   one thread per item: rasterize prologue (matrix, c0, c1)
//                    and the depth-independent half of queryVisibility.
//   rz_setup_kernel  one thread per quad: transform, cull, bounding rectangle,
//                    depth plane, edge normalization (Rasterizer.cpp:657-1081).
//   rz_frame_kernel  one work-group per screen tile, all tiles co-resident:
//                    the tile's depth and hiZ live in LDS; items are walked in
//                    draw order; a query2D is reduced across the tiles that
//                    overlap its rectangle with device atomics, so each item
//                    is drawn exactly when the reference would draw it.  A wave64
//                    takes 64 (quad, block) pairs at a time, a lane each, for
//                    their coverage, then one 8x8 block at a time with lane =
//                    pixel (Rasterizer.cpp:1095-1292).
#include "rz_kernels.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>

#include "rz_x86.h"

extern "C" __device__ uint32_t __ockl_wfred_min_u32(uint32_t);
extern "C" __device__ uint32_t __ockl_wfred_max_u32(uint32_t);
extern "C" __device__ uint32_t __ockl_wfred_add_u32(uint32_t);
extern "C" __device__ uint32_t __ockl_wfred_or_u32(uint32_t);
extern "C" __device__ uint32_t __ockl_wfscan_add_u32(uint32_t, bool);

namespace rzd {

constexpr uint32_t kModeTriangle0 = 1, kModeTriangle1 = 2, kModeConcaveRight = 3, kModeConcaveLeft = 4,
                   kModeConcaveCenter = 5, kModeConvex = 6;

// modeTable of Rasterizer.cpp:30-64: primitive mode for each 8-bit
// configuration (bits 0-3: triangle area <= 0, bits 4-7: w < 0).
__constant__ uint8_t c_modeTable[256] = {
    6, 2, 4, 2, 1, 0, 1, 0, 3, 2, 0, 2, 1, 0, 1, 0, 6, 2, 4, 2, 1, 0, 1, 0, 0, 2, 5, 2, 1, 0, 1, 0,
    6, 0, 4, 2, 1, 0, 1, 0, 3, 2, 5, 2, 1, 0, 0, 0, 6, 2, 4, 0, 1, 0, 1, 0, 3, 2, 5, 2, 0, 0, 1, 0,
    6, 2, 0, 2, 1, 0, 1, 0, 3, 2, 5, 2, 1, 0, 1, 0, 0, 2, 5, 2, 1, 0, 1, 0, 5, 2, 5, 2, 1, 0, 1, 0,
    6, 2, 4, 2, 1, 0, 0, 0, 3, 0, 5, 2, 1, 0, 1, 0, 2, 2, 2, 2, 0, 0, 0, 0, 2, 2, 2, 0, 0, 0, 0, 0,
    6, 2, 4, 2, 0, 0, 1, 0, 3, 2, 5, 0, 1, 0, 1, 0, 6, 2, 4, 2, 1, 0, 0, 0, 3, 0, 5, 2, 1, 0, 1, 0,
    0, 2, 4, 2, 1, 0, 1, 0, 3, 2, 5, 2, 1, 0, 1, 0, 3, 2, 0, 2, 1, 0, 1, 0, 3, 2, 5, 2, 1, 0, 1, 0,
    6, 2, 4, 0, 1, 0, 1, 0, 3, 2, 5, 2, 0, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 1, 0, 0, 0,
    4, 2, 4, 2, 1, 0, 1, 0, 0, 2, 5, 2, 1, 0, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0,
};

constexpr uint64_t kEmptyBox = 0x000000000000FFFFull;  // min column 0xFFFF > max column 0

// ---------------------------------------------------------------------------
// Depth-independent half of queryVisibility (Rasterizer.cpp:125-273).
// ---------------------------------------------------------------------------
struct QueryPre {
  uint32_t kind;  // 0 frustum-culled, 1 near the camera plane, 2 empty rectangle, 3 rectangle test
  uint32_t minX, maxX, minY, maxY, maxZ;
};

__device__ QueryPre query_pre(const Mvp& M, const float* bmin, const float* bmax, uint32_t width, uint32_t height,
                              const uint32_t* __restrict__ rcpTab) {
  QueryPre out = {0, 0, 0, 0, 0, 0};
  float ext[4], cen[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ext[j] = bmax[j] - bmin[j];
    cen[j] = bmax[j] + bmin[j];
  }
  // Six frustum planes from the raw rows; the box corner is chosen by the
  // plane's sign bits (:135-167).  A set sign bit on any distance culls.
  const float* R = M.raw;
  uint32_t signs = 0;
#pragma unroll
  for (int pl = 0; pl < 6; ++pl) {
    const int rr = pl >> 1;
    float plane[4], off[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      plane[j] = (pl & 1) ? (R[12 + j] - R[4 * rr + j]) : (R[12 + j] + R[4 * rr + j]);
      off[j] = cen[j] + xor_sign(ext[j], fbits(plane[j]) & 0x80000000u);
    }
    signs |= fbits(dp4_x86(plane[0], plane[1], plane[2], plane[3], off[0], off[1], off[2], off[3]));
  }
  if (signs & 0x80000000u) return out;

  // Eight corners with the prebaked columns (:169-198).
  const float* C = M.prebaked;
  float c[8][4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float e0 = C[0 + j] * ext[0];
    const float e1 = C[4 + j] * ext[1];
    const float e2 = C[8 + j] * ext[2];
    c[0][j] = fmaf(C[0 + j], bmin[0], fmaf(C[4 + j], bmin[1], fmaf(C[8 + j], bmin[2], C[12 + j])));
    c[1][j] = c[0][j] + e0;
    c[2][j] = c[0][j] + e1;
    c[4][j] = c[0][j] + e2;
    c[3][j] = c[1][j] + e1;
    c[5][j] = c[4][j] + e0;
    c[6][j] = c[2][j] + e2;
    c[7][j] = c[6][j] + e0;
  }
  // Per-lane near-plane epsilon (:204-213): lane j compares corners j and j+4.
  float me1[4], me2[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) me1[j] = max_x86(ext[j], ext[j ^ 2]);
#pragma unroll
  for (int j = 0; j < 4; ++j) me2[j] = max_x86(me1[j], me1[j ^ 1]);
  bool close = false;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float eps = me2[j] * 0.001f;
    close |= (c[j][3] < eps) || (c[4 + j][3] < eps);
  }
  if (close) {
    out.kind = 1;
    return out;
  }
  // Projection, screen rectangle (:217-264).
  float px[8], py[8], pz[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float rw = rcp_x86(c[k][3], rcpTab);
    px[k] = c[k][0] * rw;
    py[k] = c[k][1] * rw;
    pz[k] = c[k][2] * rw;
  }
  float minsX[4], maxsX[4], minsY[4], maxsY[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    minsX[j] = min_x86(px[j], px[4 + j]);
    maxsX[j] = max_x86(px[j], px[4 + j]);
    minsY[j] = min_x86(py[j], py[4 + j]);
    maxsY[j] = max_x86(py[j], py[4 + j]);
  }
  float mXY[4] = {min_x86(minsX[0], minsX[2]), min_x86(minsY[0], minsY[2]), min_x86(minsX[1], minsX[3]),
                  min_x86(minsY[1], minsY[3])};
  float MXY[4] = {max_x86(maxsX[0], maxsX[2]), max_x86(maxsY[0], maxsY[2]), max_x86(maxsX[1], maxsX[3]),
                  max_x86(maxsY[1], maxsY[3])};
  const float lim[4] = {float(width - 1), float(height - 1), float(width - 1), float(height - 1)};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    mXY[j] = max_x86(mXY[j], 0.0f);
    MXY[j] = -min_x86(MXY[j], lim[j]);
  }
  const float bf[4] = {min_x86(mXY[0], mXY[2]), min_x86(MXY[0], MXY[2]), min_x86(mXY[1], mXY[3]),
                       min_x86(MXY[1], MXY[3])};
  int32_t bi[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) bi[j] = cvtt_x86(floorf(bf[j]));
  bi[1] = int32_t(0u - uint32_t(bi[1]));
  bi[3] = int32_t(0u - uint32_t(bi[3]));
  if (bi[0] >= bi[1] || bi[2] >= bi[3]) {
    out.kind = 2;
    return out;
  }
  uint32_t maxZ = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) maxZ = max(maxZ, pack_depth(pz[k]));
  out.kind = 3;
  out.minX = uint32_t(bi[0]);
  out.maxX = uint32_t(bi[1]);
  out.minY = uint32_t(bi[2]);
  out.maxY = uint32_t(bi[3]);
  out.maxZ = maxZ;
  return out;
}

// One buffer's depth as the query kernels read it from device memory.
struct QueryBufs {
  const uint16_t* __restrict__ depth;
  const uint16_t* __restrict__ hiz;
  const uint16_t* __restrict__ tileMin;
  uint32_t bX, pyrX;
};

// Whether block (bx, by) has a pixel of the rectangle nearer than maxZ.  Pixels
// outside it are set to the largest depth, so the test is one packed minimum
// over the rows; four rows' loads are issued before their use.
typedef unsigned short U16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ bool block_pixels_hit(const QueryBufs& B, uint32_t bx, uint32_t by, uint32_t minX,
                                                 uint32_t maxX, uint32_t minY, uint32_t maxY, uint32_t maxZ) {
  const int32_t sy = int32_t(minY - 8 * by), ey = int32_t(maxY - 8 * by);
  const int32_t sx = int32_t(minX - 8 * bx), ex = int32_t(maxX - 8 * bx);
  const uint32_t startY = uint32_t(sy > 0 ? sy : 0), endY = uint32_t(ey < 7 ? ey : 7);
  const uint32_t startX = uint32_t(sx > 0 ? sx : 0), endX = uint32_t(ex < 7 ? ex : 7);
  const uint32_t in = (0xFFu << startX) & (0xFFu >> (7u - endX));
  uint32_t outside[4];
#pragma unroll
  for (uint32_t x = 0; x < 4; ++x)
    outside[x] = ((in >> (2 * x)) & 1u ? 0u : 0xFFFFu) | ((in >> (2 * x + 1)) & 1u ? 0u : 0xFFFF0000u);
  const uint4* rows = reinterpret_cast<const uint4*>(B.depth + (size_t(by) * B.bX + bx) * 64);
  U16x2 least = {0xFFFF, 0xFFFF};
  for (uint32_t h = startY & ~3u; h <= endY; h += 4) {
    uint4 r[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      r[j] = make_uint4(0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu);
      if (h + j >= startY && h + j <= endY) r[j] = rows[h + j];
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      const uint32_t w[4] = {r[j].x, r[j].y, r[j].z, r[j].w};
#pragma unroll
      for (uint32_t x = 0; x < 4; ++x)
        least = __builtin_elementwise_min(least, __builtin_bit_cast(U16x2, w[x] | outside[x]));
    }
  }
  return uint32_t(least.x < least.y ? least.x : least.y) < maxZ;
}

// query2D (Rasterizer.cpp:283-349) by one wave on the buffers in device
// memory.  The result is the OR over the rectangle's blocks of "maxZ > hiZ
// and (block interior to the rectangle, or a pixel in range nearer than
// maxZ)", so blocks may be visited in any order: lanes take 8x8-block tiles
// whose minimum hiZ is below maxZ (other tiles hold no candidate block), then
// one block per lane inside each candidate tile.
__device__ bool query2d_wave(uint32_t minX, uint32_t maxX, uint32_t minY, uint32_t maxY, uint32_t maxZ,
                             const QueryBufs& B, uint32_t lane) {
  const uint32_t bx0 = minX >> 3, bx1 = maxX >> 3, by0 = minY >> 3, by1 = maxY >> 3;
  const uint32_t tx0 = bx0 >> 3, tx1 = bx1 >> 3, ty0 = by0 >> 3, ty1 = by1 >> 3;
  const uint32_t ntx = tx1 - tx0 + 1, nt = ntx * (ty1 - ty0 + 1);
  for (uint32_t tb = 0; tb < nt; tb += 64) {
    const uint32_t t = tb + lane;
    const bool cand = t < nt && uint32_t(B.tileMin[(ty0 + t / ntx) * B.pyrX + tx0 + t % ntx]) < maxZ;
    uint64_t cm = __ballot(cand);
    while (cm) {
      const uint32_t k = uint32_t(__builtin_ctzll(cm));
      cm &= cm - 1;
      const uint32_t tt = tb + k;
      const uint32_t bx = (tx0 + tt % ntx) * 8 + (lane & 7u), by = (ty0 + tt / ntx) * 8 + (lane >> 3);
      bool v = false;
      if (bx >= bx0 && bx <= bx1 && by >= by0 && by <= by1) {
        if (maxZ > uint32_t(B.hiz[by * B.bX + bx])) {
          v = (minX <= 8 * bx && maxX >= 8 * bx + 7 && minY <= 8 * by && maxY >= 8 * by + 7) ||
              block_pixels_hit(B, bx, by, minX, maxX, minY, maxY, maxZ);
        }
      }
      if (__ballot(v) != 0ull) return true;
    }
  }
  return false;
}

// query2D of the wave's boxes, one rectangle per lane with `test` set; returns
// the lane's answer.
//   - A rectangle of at most 4x4 tiles first takes its tiles' minima alone, one
//     lane per box: what they cover is answered here, for 64 boxes at once.
//   - The rest go eight at a time, eight lanes each, a lane to a column of
//     blocks: a candidate tile's 64 hiZ values are one load per row and lane,
//     all in flight together, and only where no interior block is open do the
//     blocks at the rectangle's border read their pixels.
//   - Wider rectangles take the whole wave, one after another; so do all with
//     WHOLE.
// Bound by latency (box, reciprocal table, tile minima, hiZ, pixels in turn)
// and instructions: a city query's rectangle has some tens of blocks, so a
// whole wave for each box in turn left most lanes idle.  A batch of 1,000,003
// city boxes, together with launch_query's rule: 157 to 180 us before, 18 to 24 us
// now, by where the camera stands (the table in launch_query is of one of them).
template <bool WHOLE>
__device__ bool query2d_boxes(const QueryPre& Q, bool test, const QueryBufs& B, uint32_t lane) {
  const uint32_t tx0 = Q.minX >> 6, ty0 = Q.minY >> 6;
  const uint32_t ntx = (Q.maxX >> 6) - tx0 + 1, nty = (Q.maxY >> 6) - ty0 + 1;
  const bool narrow = !WHOLE && test && ntx <= 4u && nty <= 4u;
  bool vis = false;
  uint32_t cand = 0;  // bit 4 y + x: tile (tx0 + x, ty0 + y) may hold an open block
  if (narrow) {
    const uint16_t* row = B.tileMin + ty0 * B.pyrX + tx0;
    for (uint32_t y = 0; y < nty; ++y, row += B.pyrX) {
      uint32_t z[4];
#pragma unroll
      for (uint32_t x = 0; x < 4; ++x) z[x] = x < ntx ? uint32_t(row[x]) : 0xFFFFu;
#pragma unroll
      for (uint32_t x = 0; x < 4; ++x) cand |= z[x] < Q.maxZ ? 1u << (4 * y + x) : 0u;
    }
  }
  uint64_t m = __ballot(cand != 0u);
  const uint32_t group = lane >> 3, shift = lane & ~7u;
  while (m) {
    uint32_t from[8], src = 64;
#pragma unroll
    for (uint32_t g = 0; g < 8; ++g) {
      from[g] = m ? uint32_t(__builtin_ctzll(m)) : 64u;
      m &= m - 1ull;
      src = group == g ? from[g] : src;
    }
    const int j = int(src & 63u);
    const uint32_t minX = __shfl(Q.minX, j), maxX = __shfl(Q.maxX, j);
    const uint32_t minY = __shfl(Q.minY, j), maxY = __shfl(Q.maxY, j);
    const uint32_t maxZ = __shfl(Q.maxZ, j);
    uint32_t c = __shfl(cand, j);
    if (src == 64u) c = 0;
    bool hit = false;
    while (c) {
      const uint32_t t = uint32_t(__builtin_ctz(c));
      c &= c - 1u;
      const uint32_t bx = ((minX >> 6) + (t & 3u)) * 8 + (lane & 7u), y0 = ((minY >> 6) + (t >> 2)) * 8;
      const bool inX = bx >= minX >> 3 && bx <= maxX >> 3;
      uint32_t z[8];
#pragma unroll
      for (uint32_t r = 0; r < 8; ++r) {
        z[r] = 0xFFFFu;
        if (inX && y0 + r >= minY >> 3 && y0 + r <= maxY >> 3) z[r] = B.hiz[(y0 + r) * B.bX + bx];
      }
      const bool wholeX = minX <= 8 * bx && maxX >= 8 * bx + 7;
      uint32_t border = 0;
      bool v = false;
#pragma unroll
      for (uint32_t r = 0; r < 8; ++r) {
        const bool whole = wholeX && minY <= 8 * (y0 + r) && maxY >= 8 * (y0 + r) + 7;
        if (z[r] < maxZ) {
          if (whole) v = true;
          else border |= 1u << r;
        }
      }
      hit = ((__ballot(v) >> shift) & 0xFFull) != 0ull;
      while (!hit && ((__ballot(border != 0u) >> shift) & 0xFFull) != 0ull) {
        if (border) {
          const uint32_t by = y0 + uint32_t(__builtin_ctz(border));
          border &= border - 1u;
          v = block_pixels_hit(B, bx, by, minX, maxX, minY, maxY, maxZ);
        }
        hit = ((__ballot(v) >> shift) & 0xFFull) != 0ull;
      }
      if (hit) c = 0;
    }
    const uint64_t hits = __ballot(hit);
#pragma unroll
    for (uint32_t g = 0; g < 8; ++g)
      if (lane == from[g]) vis = ((hits >> (8 * g)) & 1ull) != 0ull;
  }
  m = __ballot(test && !narrow);
  while (m) {
    const int j = int(__builtin_ctzll(m));
    m &= m - 1ull;
    const uint32_t minX = uint32_t(__builtin_amdgcn_readlane(int(Q.minX), j));
    const uint32_t maxX = uint32_t(__builtin_amdgcn_readlane(int(Q.maxX), j));
    const uint32_t minY = uint32_t(__builtin_amdgcn_readlane(int(Q.minY), j));
    const uint32_t maxY = uint32_t(__builtin_amdgcn_readlane(int(Q.maxY), j));
    const uint32_t maxZ = uint32_t(__builtin_amdgcn_readlane(int(Q.maxZ), j));
    const bool v = query2d_wave(minX, maxX, minY, maxY, maxZ, B, lane);
    if (int(lane) == j) vis = v;
  }
  return vis;
}

// ---------------------------------------------------------------------------
// Prep: rasterize prologue per item (Rasterizer.cpp:616-655) and the item's
// status for the draw loop.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) rz_prep_kernel(PrepParams p) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.nItems) return;
  ItemDesc D;
  if (p.hostItems) {
    D = p.hostItems[i];
    p.itemsOut[i] = D;
  } else {
    D = p.items[i];
  }
  if (p.groupItem && D.quadCount != 0u) {
    // Items cover the quads 0..nQuads-1 in order, so each group's first
    // quad lies in exactly one non-empty item.
    const uint32_t last = (D.quadBase + D.quadCount - 1u) >> 6;
    for (uint32_t k = (D.quadBase + 63u) >> 6; k <= last; ++k) p.groupItem[k] = i;
  }
  ItemState& S = p.state[i];
  const Mvp* M = &p.mvp;
  uint32_t width = p.width, height = p.height, tileW = p.tileW, tileH = p.tileH;
  if (p.views) {
    const ViewDesc& V = p.views[D.view];
    M = &V.mvp;
    width = V.width;
    height = V.height;
    tileW = tileH = V.tileB;
  }
  if (i == 0 && p.queue) *p.queue = 0u;
  const float* P = M->prebaked;
  float ext[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) ext[j] = D.refMax[j] - D.refMin[j];
  const float k0 = 1.0f / float(2047ull << 21);
  const float k1 = 1.0f / float(2047 << 10);
  const float k2 = 1.0f / float(1023);
  float m0[4], m1[4], m2[4], m3[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    m3[j] = fmaf(P[0 + j], D.refMin[0], fmaf(P[4 + j], D.refMin[1], fmaf(P[8 + j], D.refMin[2], P[12 + j])));
    m0[j] = P[0 + j] * (ext[0] * k0);
    m1[j] = P[4 + j] * (ext[1] * k1);
    m2[j] = P[8 + j] * (ext[2] * k2);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    m3[j] = fmaf(m0[j], 2147483648.0f, m3[j]);
    m1[j] = m1[j] - m0[j];
    m2[j] = m2[j] - m0[j];
  }
#pragma unroll
  for (int o = 0; o < 4; ++o) {
    S.T[o][0] = m0[o];
    S.T[o][1] = m1[o];
    S.T[o][2] = m2[o];
    S.T[o][3] = m3[o];
  }
  const float Za = m3[2], Zb = dp4_x86(m0[2], m1[2], m2[2], m3[2], 2097152.0f, 1024.0f, 1.0f, 1.0f);
  const float Wa = m3[3], Wb = dp4_x86(m0[3], m1[3], m2[3], m3[3], 2097152.0f, 1024.0f, 1.0f, 1.0f);
  // x86 NaN rules: a tiny reference box can make both differences 0.
  const float q = div_x86(Za - Zb, Wa - Wb);
  S.c0 = q;
  S.c1 = fnmadd_x86(q, Wa, Za);

  S.fp[0] = 0xFFFFFFFFu;
  S.fp[1] = 0u;
  S.fp[2] = 0xFFFFFFFFu;
  S.fp[3] = 0u;
  S.expected = 0;
  S.qMinX = S.qMaxX = S.qMinY = S.qMaxY = S.qMaxZ = 0;
  p.done[i] = 0;
  p.visible[i] = 0;
  uint32_t status;
  if (D.kind == kItemForceNoClip) {
    status = kStatusNoClip;
  } else if (D.kind == kItemForceClip) {
    status = kStatusClip;
  } else if (D.kind == kItemClassify) {
    // Frustum cull, near-plane test and empty rectangle only; no query2D.
    const QueryPre Q = query_pre(*M, D.boundsMin, D.boundsMax, width, height, p.rcp);
    status = Q.kind == 1 ? kStatusClip : (Q.kind == 3 ? kStatusNoClip : kStatusSkip);
  } else {
    const QueryPre Q = query_pre(*M, D.boundsMin, D.boundsMax, width, height, p.rcp);
    if (Q.kind == 1) {
      status = kStatusClip;
    } else if (Q.kind == 3) {
      status = kStatusTest;
      S.qMinX = Q.minX;
      S.qMaxX = Q.maxX;
      S.qMinY = Q.minY;
      S.qMaxY = Q.maxY;
      S.qMaxZ = Q.maxZ;
      const uint32_t tx0 = (Q.minX >> 3) / tileW, tx1 = (Q.maxX >> 3) / tileW;
      const uint32_t ty0 = (Q.minY >> 3) / tileH, ty1 = (Q.maxY >> 3) / tileH;
      S.expected = (tx1 - tx0 + 1) * (ty1 - ty0 + 1);
    } else {
      status = kStatusSkip;
    }
  }
  S.status = status;
}

// ---------------------------------------------------------------------------
// Setup: one quad per thread (Rasterizer.cpp:660-1063).
// ---------------------------------------------------------------------------
struct SetupOut {
  bool valid;
  QuadRec rec;
};

__device__ void setup_quad(const ItemState& S, const uint32_t I[4], bool clip, uint32_t bX, uint32_t bY,
                           const uint32_t* __restrict__ rcpTab, SetupOut& out) {
  const float maxInvW = 1.84467430e+19f;  // sqrt(FLT_MAX) rounded to float (Rasterizer.cpp:11)
  float x[4], y[4], invW[4];
  uint32_t ws[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float Xf = float(int32_t(I[k]));
    const float Yf = float(int32_t(I[k] & (2047u << 10)));
    const float Zf = float(int32_t(I[k] & 1023u));
    const float X = fmaf(Xf, S.T[0][0], fmaf(Yf, S.T[0][1], fmaf(Zf, S.T[0][2], S.T[0][3])));
    const float Y = fmaf(Xf, S.T[1][0], fmaf(Yf, S.T[1][1], fmaf(Zf, S.T[1][2], S.T[1][3])));
    const float W = fmaf(Xf, S.T[3][0], fmaf(Yf, S.T[3][1], fmaf(Zf, S.T[3][2], S.T[3][3])));
    const float r = rcp_x86(W, rcpTab);
    invW[k] = clip ? min_x86(maxInvW, max_x86(-maxInvW, r)) : r;
    x[k] = rintf(X * invW[k]) * 0.125f;
    y[k] = rintf(Y * invW[k]) * 0.125f;
    ws[k] = clip ? (fbits(invW[k]) & 0x80000000u) : 0u;
  }
  float eX[5], eY[5];
  eX[0] = y[1] - y[0];
  eX[1] = y[2] - y[1];
  eX[2] = y[3] - y[2];
  eX[3] = y[0] - y[3];
  eY[0] = x[0] - x[1];
  eY[1] = x[1] - x[2];
  eY[2] = x[2] - x[3];
  eY[3] = x[3] - x[0];
  const float area0 = fmaf(eX[0], eY[1], -(eX[1] * eY[0]));
  const float area1 = fmaf(eX[1], eY[2], -(eX[2] * eY[1]));
  const float area2 = fmaf(eX[2], eY[3], -(eX[3] * eY[2]));
  const float area3 = (area0 + area2) - area1;
  // Area signs with zero counted as negative; flipped per w < 0 vertex when
  // clipping (:775-803).
  const uint32_t s0 = xor_sign(xor_sign(area0, ws[0]), ws[1] ^ ws[2]) <= 0.0f;
  const uint32_t s1 = xor_sign(xor_sign(area1, ws[1]), ws[2] ^ ws[3]) <= 0.0f;
  const uint32_t s2 = xor_sign(xor_sign(area2, ws[0]), ws[2] ^ ws[3]) <= 0.0f;
  const uint32_t s3 = xor_sign(xor_sign(area3, ws[1]), ws[0] ^ ws[3]) <= 0.0f;
  const uint32_t config = s0 | (s1 << 1) | (s2 << 2) | (s3 << 3) | (ws[0] >> 27) | (ws[1] >> 26) | (ws[2] >> 25) |
                          (ws[3] >> 24);
  const uint32_t mode = c_modeTable[config];
  out.valid = false;
  if (mode == 0) return;

  float minFx, minFy, maxFx, maxFy;
  if (clip) {
    // Clipless bounding box from the intervals of w > 0 and w < 0 vertices
    // (:820-909).
    const float infP = 10000.0f, infN = -10000.0f;
    float minPx[4], minPy[4], maxPx[4], maxPy[4], minNx[4], minNy[4], maxNx[4], maxNy[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool neg = ws[k] != 0u;
      minPx[k] = neg ? infP : x[k];
      minPy[k] = neg ? infP : y[k];
      maxPx[k] = xor_sign(minPx[k], ws[k]);
      maxPy[k] = xor_sign(minPy[k], ws[k]);
      minNx[k] = neg ? x[k] : infP;
      minNy[k] = neg ? y[k] : infP;
      maxNx[k] = neg ? x[k] : infN;
      maxNy[k] = neg ? y[k] : infN;
    }
    // Reductions in the reference's pairing: op(op(v0, v1), op(v2, v3)).
    const float mPx = min_x86(min_x86(minPx[0], minPx[1]), min_x86(minPx[2], minPx[3]));
    const float mPy = min_x86(min_x86(minPy[0], minPy[1]), min_x86(minPy[2], minPy[3]));
    const float MPx = max_x86(max_x86(maxPx[0], maxPx[1]), max_x86(maxPx[2], maxPx[3]));
    const float MPy = max_x86(max_x86(maxPy[0], maxPy[1]), max_x86(maxPy[2], maxPy[3]));
    const float mNx = min_x86(min_x86(minNx[0], minNx[1]), min_x86(minNx[2], minNx[3]));
    const float mNy = min_x86(min_x86(minNy[0], minNy[1]), min_x86(minNy[2], minNy[3]));
    const float MNx = max_x86(max_x86(maxNx[0], maxNx[1]), max_x86(maxNx[2], maxNx[3]));
    const float MNy = max_x86(max_x86(maxNy[0], maxNy[1]), max_x86(maxNy[2], maxNy[3]));
    const float incAx = (MNx > mPx) ? infN : mPx;
    const float incAy = (MNy > mPy) ? infN : mPy;
    const float incBx = (MPx > mNx) ? infP : MPx;
    const float incBy = (MPy > mNy) ? infP : MPy;
    minFx = min_x86(incAx, incBx);
    minFy = min_x86(incAy, incBy);
    maxFx = max_x86(incAx, incBx);
    maxFy = max_x86(incAy, incBy);
  } else {
    minFx = min_x86(min_x86(x[0], x[1]), min_x86(x[2], x[3]));
    minFy = min_x86(min_x86(y[0], y[1]), min_x86(y[2], y[3]));
    maxFx = max_x86(max_x86(x[0], x[1]), max_x86(x[2], x[3]));
    maxFy = max_x86(max_x86(y[0], y[1]), max_x86(y[2], y[3]));
  }
  int32_t minX = cvtt_x86(minFx + 0.6249875f);
  int32_t minY = cvtt_x86(minFy + 0.6249875f);
  int32_t maxX = cvtt_x86(maxFx + 1.375f);
  int32_t maxY = cvtt_x86(maxFy + 1.375f);
  minX = max(minX, 0);
  minY = max(minY, 0);
  maxX = min(maxX, int32_t(bX));
  maxY = min(maxY, int32_t(bY));
  if (!(maxX > minX && maxY > minY)) return;

  float z[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) z[k] = fmadd_x86(invW[k], S.c1, S.c0);
  float maxZ = max_x86(max_x86(z[0], z[1]), max_x86(z[2], z[3]));
  if ((ws[0] | ws[1] | ws[2] | ws[3]) != 0u) maxZ = 1.0f;

  // Depth plane from the larger triangle (:963-999).
  const bool tri0 = mode == kModeTriangle0, tri1 = mode == kModeTriangle1;
  const bool greater = !tri0 && (tri1 || (__builtin_fabsf(area0) < __builtin_fabsf(area2)));
  const float selArea = greater ? area2 : area0;
  const float invArea = clip ? 1.0f / selArea : rcp_x86(selArea, rcpTab);
  const float z12 = z[1] - z[2], z20 = z[2] - z[0], z30 = z[3] - z[0];
  eX[4] = y[0] - y[2];
  eY[4] = x[2] - x[0];
  const float dpx = greater ? fmaf(-z20, eX[3], z30 * eX[4]) : fmaf(z20, eX[1], -(z12 * eX[4]));
  const float dpy = greater ? fmaf(-z20, eY[3], z30 * eY[4]) : fmaf(z20, eY[1], -(z12 * eY[4]));
  const float dp1 = invArea * dpx;
  const float dp2 = invArea * dpy;
  const float x0 = x[0] - float(minX);
  const float y0 = y[0] - float(minY);
  const float dp0 = fmaf(-x0, dp1, fmaf(-y0, dp2, z[0]));

  // Triangle modes swap in the diagonal edge (:1001-1005); edges facing w < 0
  // are flipped (:1007-1022); normalization to 70 / (|nx| + |ny|) (:452-468).
  if (tri0) {
    eX[2] = eX[4];
    eY[2] = eY[4];
  }
  if (tri1) {
    eX[0] = -eX[4];
    eY[0] = -eY[4];
  }
  uint32_t flip[4] = {0u, 0u, 0u, 0u};
  if (clip) {
    flip[0] = ws[0] ^ (tri1 ? ws[2] : ws[1]);
    flip[1] = ws[1] ^ ws[2];
    flip[2] = ws[2] ^ (tri0 ? ws[0] : ws[3]);
    flip[3] = ws[0] ^ ws[3];
  }
  const float edgeScale = 63.0f / (0.45f - -0.45f);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float invLen = rcp_x86(__builtin_fabsf(eX[e]) + __builtin_fabsf(eY[e]), rcpTab);
    const float mul = clip ? xor_sign(edgeScale, flip[e]) : edgeScale;
    invLen = mul * invLen;
    eX[e] = eX[e] * invLen;
    eY[e] = eY[e] * invLen;
  }
  // Edge offsets at the rectangle origin (:1030-1045).
  const float add = 0.5f - -0.45f * 63.0f / (0.45f - -0.45f);
  const float fMinX = float(minX), fMinY = float(minY);
  float off0 = fmaf(-x0, eX[0], fmaf(-y0, eY[0], add));
  float off1 = fmaf(-x[1], eX[1], fmaf(-y[1], eY[1], add));
  float off2 = fmaf(-x[2], eX[2], fmaf(-y[2], eY[2], add));
  float off3 = fmaf(-x[3], eX[3], fmaf(-y[3], eY[3], add));
  off1 = fmaf(fMinX, eX[1], off1);
  off2 = fmaf(fMinX, eX[2], off2);
  off3 = fmaf(fMinX, eX[3], off3);
  off1 = fmaf(fMinY, eY[1], off1);
  off2 = fmaf(fMinY, eY[2], off2);
  off3 = fmaf(fMinY, eY[3], off3);
  // Slope buckets with ny <= 0 selecting the odd bucket (:482-493).
  const float slopeMul = 15.5f / edgeScale;
  uint32_t slope[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int32_t q = cvtt_x86(fmaf(eX[e], slopeMul, 16.0f));
    slope[e] = ((uint32_t(q) << 1) + (eY[e] <= 0.0f ? 1u : 0u)) << 6;
  }

  QuadRec& R = out.rec;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    R.nx[e] = eX[e];
    R.ny[e] = eY[e];
  }
  R.off[0] = off0;
  R.off[1] = off1;
  R.off[2] = off2;
  R.off[3] = off3;
  R.dp0 = dp0;
  R.dDx = dp1;
  R.dDy = dp2;
  // 16-bit lane multiply of the first block index (:1054).
  R.fb = ((uint32_t(minY) * bX) & 0xFFFFu) + uint32_t(minX);
  R.range = uint32_t(maxX - minX) | (uint32_t(maxY - minY) << 16);
  R.modeZ = mode | (pack_depth(maxZ) << 16);
  R.slope01 = (slope[0] & 0xFFFFu) | (slope[1] << 16);
  R.slope23 = (slope[2] & 0xFFFFu) | (slope[3] << 16);
  out.valid = true;
}

// Conservative screen-block box of a quad's blocks fb + r*bX + c,
// 0 <= r < rangeY, 0 <= c < rangeX (exact unless the 16-bit multiply
// wrapped the row index, when it spans whole rows).
__device__ uint64_t quad_box(uint32_t fb, uint32_t rangeX, uint32_t rangeY, uint32_t bX, uint32_t bY) {
  const uint32_t col = fb % bX, row = fb / bX;
  uint32_t c0, c1, r0 = row, r1;
  if (col + rangeX <= bX) {
    c0 = col;
    c1 = col + rangeX - 1;
    r1 = row + rangeY - 1;
  } else {
    c0 = 0;
    c1 = bX - 1;
    r1 = row + rangeY;
  }
  r1 = min(r1, bY - 1);
  return uint64_t(c0) | (uint64_t(c1) << 16) | (uint64_t(r0) << 32) | (uint64_t(r1) << 48);
}

// The item that holds quad g: the last item whose quadBase <= g (items are
// in quad order; empty items share their successor's quadBase).  With a
// group table (groupItem[k] = the item of quad 64k) the search starts there
// and steps forward over the items that begin inside the 64-quad group.
__device__ __forceinline__ uint32_t item_of_quad(const ItemDesc* __restrict__ items, uint32_t nItems, uint32_t g,
                                                 const uint32_t* __restrict__ groupItem = nullptr) {
  if (groupItem) {
    uint32_t i = min(groupItem[g >> 6], nItems - 1u);
    while (i + 1 < nItems && items[i + 1].quadBase <= g) ++i;
    return i;
  }
  uint32_t lo = 0, hi = nItems - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if (items[mid].quadBase <= g) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__global__ void __launch_bounds__(256) rz_setup_kernel(SetupParams p) {
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  const bool inRange = g < p.nQuads;
  uint32_t item = 0;
  bool valid = false;
  uint64_t box = kEmptyBox;
  uint32_t fz = 0u;
  if (inRange) {
    item = item_of_quad(p.items, p.nItems, g, p.groupItem);
    const ItemDesc& D = p.items[item];
    const ItemState& S = p.state[item];
    const uint32_t st = S.status;
    if (st != kStatusSkip) {
      uint32_t bX = p.bX, bY = p.bY;
      if (p.views) {
        bX = p.views[D.view].bX;
        bY = p.views[D.view].bY;
      }
      const uint32_t q = g - D.quadBase;
      const uint32_t* pk = D.packets + (q >> 3) * 32 + (q & 7);
      const uint32_t I[4] = {pk[0], pk[8], pk[16], pk[24]};
      SetupOut o;
      setup_quad(S, I, st == kStatusClip, bX, bY, p.rcp, o);
      if (o.valid) {
        valid = true;
        p.recs[g] = o.rec;
        box = quad_box(o.rec.fb, o.rec.range & 0xFFFFu, o.rec.range >> 16, bX, bY);
        if ((o.rec.range & 0xFFFFu) != 0u && (o.rec.range >> 16) != 0u) fz = o.rec.modeZ | kFeatValid;
      }
    }
    // Records and boxes of items that are not drawn are never read (tiles,
    // binning and features test the item's status first), so only drawn
    // items write them; an empty rectangle marks a quad as not drawn.
    if (st != kStatusSkip) {
      if (!valid) p.recs[g].range = 0u;
      p.bbox[g] = box;
      if (p.featZ) p.featZ[g] = fz;
    }
  }
  // Footprint of each item's valid quads: one atomic per wave when the whole
  // wave works on one item, else one per valid lane.
  const uint32_t c0 = valid ? uint32_t(box & 0xFFFF) : 0xFFFFFFFFu;
  const uint32_t c1 = valid ? uint32_t((box >> 16) & 0xFFFF) : 0u;
  const uint32_t r0 = valid ? uint32_t((box >> 32) & 0xFFFF) : 0xFFFFFFFFu;
  const uint32_t r1 = valid ? uint32_t(box >> 48) : 0u;
  const uint32_t firstItem = __builtin_amdgcn_readfirstlane(item);
  const bool sameItem = __ballot(inRange && item != firstItem) == 0ull;
  const uint32_t a = __ockl_wfred_min_u32(c0), b = __ockl_wfred_max_u32(c1);
  const uint32_t c = __ockl_wfred_min_u32(r0), d = __ockl_wfred_max_u32(r1);
  // Box of this aligned group of 64 quads (the wave's), for the frame
  // kernel's coarse overlap test.
  if ((threadIdx.x & 63u) == 0u && inRange)
    p.groupBox[g >> 6] = a != 0xFFFFFFFFu
                             ? uint64_t(a) | (uint64_t(b) << 16) | (uint64_t(c) << 32) | (uint64_t(d) << 48)
                             : kEmptyBox;
  if (sameItem) {
    if ((threadIdx.x & 63u) == 0u && a != 0xFFFFFFFFu) {
      uint32_t* fp = p.state[firstItem].fp;
      atomicMin(&fp[0], a);
      atomicMax(&fp[1], b);
      atomicMin(&fp[2], c);
      atomicMax(&fp[3], d);
    }
  } else if (valid) {
    uint32_t* fp = p.state[item].fp;
    atomicMin(&fp[0], c0);
    atomicMax(&fp[1], c1);
    atomicMin(&fp[2], r0);
    atomicMax(&fp[3], r1);
  }
}

// ---------------------------------------------------------------------------
// Frame kernel.
// ---------------------------------------------------------------------------
__device__ __forceinline__ float readlane_f(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// A value that is the same in every lane, as a scalar.
__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t uniform(uint64_t v) {
  return uniform(uint32_t(v)) | uint64_t(uniform(uint32_t(v >> 32))) << 32;
}
template <typename T>
__device__ __forceinline__ T* uniform(T* p) {
  return reinterpret_cast<T*>(uniform(reinterpret_cast<uint64_t>(p)));
}

__device__ __forceinline__ uint32_t readlane_u(uint32_t v, uint32_t l) { return __builtin_amdgcn_readlane(v, l); }

__device__ __forceinline__ uint64_t readlane_u64(uint64_t v, uint32_t l) {
  return uint64_t(readlane_u(uint32_t(v), l)) | uint64_t(readlane_u(uint32_t(v >> 32), l)) << 32;
}

__device__ __forceinline__ int div_bx(int d, int bX, float invBX) {
  int q = int(float(d) * invBX);
  if (q * bX > d) --q;
  else if ((q + 1) * bX <= d) ++q;
  return q;
}

// What a tile needs of one item, gathered once per item window.
struct ItemLocal {
  uint32_t index;
  uint32_t flags;  // bit 0: query rectangle overlaps the tile, bit 1: footprint does, bits 2-3: status, 16-31: tiles
                   // of the rectangle
  uint32_t qMinX, qMaxX, qMinY, qMaxY, qMaxZ;
  uint32_t quadBase, quadCount;
  uint32_t nGroups;  // its groups that may touch the tile (all when they exceed 64)
  uint64_t groups;   // bit k: aligned 64-quad group (quadBase >> 6) + k may touch the tile
};

constexpr uint32_t kQuadChunk = 64;   // records staged in LDS at a time
constexpr uint32_t kNoWinner = 0xFFFFFFFFu;  // pixel winner of labelled draws: none
// A scan pass tests one quad per thread: 64 * NW quads.

template <int TBX, int TBY>
struct TileSmem {
  // Sizes that let two work-groups share a CU's 160 KB: a 16x16-block tile's
  // depth leaves less room than an 8x8-block tile's.  A chunk of 64 small
  // quads has about two rows a quad in a tile; one that needs more rows than
  // the fold table holds is drawn in several passes.
  static constexpr uint32_t kItemWindow = TBX * TBY > 64 ? 64 : 128;  // items gathered at a time
  static constexpr int kEntryRows = TBX * TBY > 64 ? 112 : 256;
  // Coverage table (Rasterizer.cpp:547-604), each word's bits in lane order:
  // bit L is pixel (L & 7, L >> 3) of the block.
  uint64_t cov[4096];
  uint16_t depth[TBX * TBY * 64];  // the tile's depth, block-linear
  uint16_t hiz[TBX * TBY];
  ItemLocal items[kItemWindow];    // this window's items that touch the tile
  QuadRec recs[kQuadChunk];        // setup records of the quads being drawn
  uint32_t qid[TBX * TBY > 64 ? 1 : kQuadChunk];  // their frame quad numbers (labelled draws, 8x8-block tiles)
  // Per tile row of each staged quad's rectangle, the folded edge offsets and
  // depth samples at the rectangle's first column in the tile.
  float entry[kEntryRows * 12];
  uint16_t pairs[8][64];  // per wave: the (block, quad) pairs being drawn
  uint32_t wcnt[2][8];
  // Where a round's run of items ends, and the mask of its visible query items.
  uint4 run[2];
  uint32_t wnext;          // candidate position where the next item window starts
  uint32_t blockStats[4];  // observability builds: visited, rejected, written, fold steps
};

// Wave that owns tile-local block (lbx, lby) while a chunk of quads is drawn:
// diagonals, so that any horizontal or vertical run of blocks is shared by
// all waves.
template <int NW>
__device__ __forceinline__ uint32_t block_owner(int lbx, int lby) { return uint32_t(lbx + lby) & uint32_t(NW - 1); }

// Adds `step` to `s` n times, each add rounded: the reference's per-row and
// per-block folds (Rasterizer.cpp:1130-1131, 1145-1146).  IEEE addition
// commutes, so step + s and s + step are the same operation.
__device__ __forceinline__ float fold_n(float s, float step, int n) {
  for (; n >= 8; n -= 8) {
    s = s + step; s = s + step; s = s + step; s = s + step;
    s = s + step; s = s + step; s = s + step; s = s + step;
  }
  for (; n > 0; --n) s = s + step;
  return s;
}

// Per-wave counters of the block loop (observability builds only): (quad,
// block) pairs visited, rejected by hiZ or by the edge tests, and written.
struct BlockCounters {
  uint32_t visited = 0, rejected = 0, written = 0, foldSteps = 0;
};

// Component e of a quad's fold at its rectangle origin and its row and column
// steps: e < 4 edge offset e, else depth sample e - 4 (rows 0/1 of a block).
__device__ __forceinline__ void quad_component(const QuadRec& R, uint32_t e, float& base, float& stepY,
                                               float& stepX) {
  const bool edge = e < 4u;
  const float* at = edge ? &R.off[e] : &R.dp0;
  stepY = *(edge ? &R.ny[e] : &R.dDy);
  stepX = *(edge ? &R.nx[e] : &R.dDx);
  base = *at;
  if (!edge) {
    const uint32_t k = e - 4u;
    base = fmaf(stepX, -0.4375f + 0.125f * float(k & 3u), fmaf(stepY, -0.4375f + 0.125f * float(k >> 2), base));
  }
}

// x in the lanes whose bit of the wave-uniform mask is set, 0 in the others.
__device__ __forceinline__ uint32_t lane_select(uint64_t mask, uint32_t x) {
  return __builtin_amdgcn_inverse_ballot_w64(mask) ? x : 0u;
}

// Orders this wave's LDS writes before its later reads of other lanes' words.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Draws a staged chunk of n quads (Rasterizer.cpp:1095-1292), in passes of as
// many quads as the fold table holds rows for.
//
// Phase A: for each row of each quad's rectangle in the tile, the twelve
// folded components (edge offsets and the eight depth samples of block rows
// 0/1) at the rectangle's first column, twelve lanes a row and five rows a
// wave at a time, each folded from the quad's origin: row steps, then column
// steps, each add rounded.
//
// Phase B: each wave lists the (quad, block) pairs of the blocks it owns, up
// to 64 at a time in submission order: lane q turns quad q's rectangle into
// one bit per owned block and writes its pairs behind those of the quads
// before it.  Then one lane per pair tests the block's hiZ, finishes the
// pair's four edge folds with the column steps left, looks up the four
// coverage words and forms the 64-pixel mask by the quad's mode (Convex: any
// offset >= 63 rejects; other modes: an empty mask does).  None of that
// depends on what earlier pairs write (a block that is not fast-cleared only
// grows), so 64 pairs cost one pass of about 150 instructions where a wave
// per pair took about that much for each.  What is left runs block by block
// and within a block pair by pair in submission order, lane = pixel, with the
// block's depth in registers: the hiZ reject, the depth rows 0/1 and 8/9 from
// the plane with rows 2-7 as rounding-up averages, and the max-merge
// (replacing while the block is fast-cleared, hiZ == 1).
//
// A block's state: until its first write, the hiZ it was opened with; after
// it, hiZ is the minimum of the depth in registers, so the reject test is a
// ballot over the depth (hiZ >= maxZ exactly when no pixel is below maxZ) and
// the fast-clear test (hiZ == 1) two ballots.  The minimum itself is taken
// once, when the block is closed.
//
// A quad whose first block index wrapped in the reference's 16-bit multiply
// (Rasterizer.cpp:1054) covers blocks fb + r * bX + c that form no screen
// rectangle: each block finds its (r, c) and folds from the quad's origin.
//
// LABELS: each block's pixel winners (`winner`, the view's block-linear
// array) are loaded with its depth unless the block is cleared (its first
// write sets them all) and stored with it; quad q's batch is qid[q] / 8.
//
// What bounds it: instruction issue and LDS latency of the waves that own a
// busy tile's blocks, not bandwidth.  Before, 16x16-block tiles drew quad by
// quad (every wave folding every quad) and 8x8-block tiles formed each pair's
// mask with a whole wave.  Measured, before and after: a 3840x2160 frame of
// 12,000 icospheres (16x16-block tiles) 8.40 and 1.35 ms; the raster launch
// of 128 city frames in flight (the same tiles) 11.0 and 5.0 ms; one 1080p
// city frame (8x8-block tiles) 0.32 and 0.26 ms.
//
// Returns (observability builds) the s_memrealtime stamp at which the last
// phase B started.
template <int TBX, int TBY, int NW, bool STATS, bool LABELS>
__device__ uint64_t draw_chunk(TileSmem<TBX, TBY>& sm, uint32_t n, int tbx0, int tbx1, int tby0, int tby1, int bX,
                               float invBX, uint32_t wave, uint32_t lane, BlockCounters& bc,
                               uint32_t* __restrict__ winner) {
  static_assert(TBX % NW == 0, "diagonal block ownership");
  constexpr int kPerRow = TBX / NW;  // the wave's blocks in a row
  constexpr int kGroupRows = kPerRow * TBY <= 32 ? TBY : 32 / kPerRow;
  constexpr int kRows = TileSmem<TBX, TBY>::kEntryRows;
  // The wave index as a scalar, so that block indices derived from it are
  // wave-uniform.
  wave = __builtin_amdgcn_readfirstlane(wave);
  uint64_t tB = 0;

  // Lane q: staged quad q's rectangle in the tile and its constants.
  const bool have = lane < n;
  const QuadRec& RL = sm.recs[have ? lane : 0u];
  const int rangeX = int(RL.range & 0xFFFFu), rangeY = int(RL.range >> 16);
  const int minY = div_bx(int(RL.fb), bX, invBX), minX = int(RL.fb) - minY * bX;
  const bool wrap = have && minX + rangeX > bX;
  const int x0 = wrap ? 0 : max(tbx0, minX) - tbx0, x1 = wrap ? TBX - 1 : min(tbx1, minX + rangeX - 1) - tbx0;
  const int y0 = wrap ? 0 : max(tby0, minY) - tby0, y1 = wrap ? TBY - 1 : min(tby1, minY + rangeY - 1) - tby0;
  const bool drawn = have && x0 <= x1 && y0 <= y1;
  const uint32_t rows = drawn && !wrap ? uint32_t(y1 - y0 + 1) : 0u;
  const uint32_t incl = __ockl_wfscan_add_u32(rows, true);  // fold table rows of quads 0..lane
  const uint32_t maxZq = RL.modeZ >> 16;
  // Row and column steps from the quad's origin to the rectangle's.
  const uint32_t steps = uint32_t(y0 + tby0 - minY) | uint32_t(x0 + tbx0 - minX) << 16;

  // The lane's pixel: its depth sample of the eight, and how its row comes
  // from rows 0/1 and 8/9.
  const int kLane = int((lane & 3u) + 4u * ((lane >> 3) & 1u));
  const bool right = (lane & 4u) != 0u, low = (lane & 32u) != 0u, odd = (lane & 16u) != 0u;

  for (uint32_t q0 = 0; q0 < n;) {
    // Quads q0..q1-1 fit the table (a quad has at most TBY rows).
    const int before = q0 ? int(readlane_u(incl, q0 - 1u)) : 0;
    const bool inPass = have && lane >= q0 && int(incl) - before <= kRows;
    const uint32_t q1 = q0 + uint32_t(__popcll(__ballot(inPass)));
    const int nRows = int(readlane_u(incl, q1 - 1u)) - before;
    const int rowBase = int(incl - rows) - before;  // table row of the rectangle's first row

    const uint32_t g = lane / 12u, e = lane - 12u * g;
    for (int j0 = int(wave) * 5; j0 < nRows; j0 += 5 * NW) {
      // The quad of table row j: the number of quads that end at or before it.
      uint32_t q = 0;
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const uint32_t qk = uint32_t(__popcll(__ballot(int(incl) - before <= j0 + k)));
        q = g == uint32_t(k) ? qk : q;
      }
      const int j = j0 + int(g);
      const bool ok = g < 5u && j < nRows;
      q = ok ? q : q0;
      const uint32_t st = uint32_t(__shfl(int(steps), int(q)));
      const int first = __shfl(rowBase, int(q));
      const int r = ok ? int(st & 0xFFFFu) + (j - first) : 0, c = ok ? int(st >> 16) : 0;
      float base, stepY, stepX;
      quad_component(sm.recs[q], e, base, stepY, stepX);
      const float s = fold_n(fold_n(base, stepY, r), stepX, c);
      if (ok) sm.entry[j * 12 + int(e)] = s;
      if (STATS) bc.foldSteps += __ockl_wfred_max_u32(uint32_t(r + c));
    }
    __syncthreads();
    if (STATS) tB = __builtin_amdgcn_s_memrealtime();

    const bool valid = drawn && inPass;
    const bool anyWrap = __ballot(valid && wrap) != 0ull;
    // What a pair's lane needs of its quad: first column, wrap flag and table
    // row of tile row 0 (biased: it can be negative).
    const uint32_t pairInfo = uint32_t(x0) | (wrap ? 0x100u : 0u) | uint32_t(rowBase - y0 + 1024) << 16;
    const uint32_t colBits = valid ? (2u << (uint32_t(x1) & 31u)) - (1u << (uint32_t(x0) & 31u)) : 0u;
    const uint32_t rowBits = valid ? (2u << (uint32_t(y1) & 31u)) - (1u << (uint32_t(y0) & 31u)) : 0u;

    // The wave's blocks, at most 32 at a time: block k of a group is in row
    // yg + k % kGroupRows, in the (k / kGroupRows)-th of the row's columns.
    for (int yg = 0; yg < TBY; yg += kGroupRows) {
      auto block_of = [&](uint32_t k) -> uint32_t {
        const uint32_t y = uint32_t(yg) + k % uint32_t(kGroupRows);
        return y * TBX + ((wave - y) & uint32_t(NW - 1)) + NW * (k / uint32_t(kGroupRows));
      };
      // Lane q: which of them quad q's rectangle holds.  Row y's columns are
      // (wave - y) mod NW and every NW-th after it: the column bits, repeated,
      // reversed and rotated, give one bit a row.
      uint32_t own = 0;
#pragma unroll
      for (int kx = 0; kx < kPerRow; ++kx) {
        const uint32_t field = (colBits >> (NW * kx)) & uint32_t((1 << NW) - 1);
        const uint32_t byRow = __builtin_bitreverse32(field * (NW == 8 ? 0x01010101u : NW == 4 ? 0x11111111u : 0x55555555u));
        const uint32_t turn = (31u - wave + uint32_t(yg)) & 31u;
        own |= (__builtin_amdgcn_alignbit(byRow, byRow, turn) & (rowBits >> yg) & uint32_t((1 << kGroupRows) - 1))
               << (kx * kGroupRows);
      }
      if (anyWrap) {
        uint32_t w = 0;
        for (uint32_t k = 0; k < uint32_t(kPerRow * kGroupRows); ++k) {
          const int b = int(block_of(k));
          const int dd = (tby0 + b / TBX) * bX + tbx0 + b % TBX - int(RL.fb);
          const int r = div_bx(max(dd, 0), bX, invBX);
          if (dd >= 0 && r < rangeY && dd - r * bX < rangeX && tbx0 + b % TBX <= tbx1 && tby0 + b / TBX <= tby1)
            w |= 1u << k;
        }
        if (valid && wrap) own = w;
      }
      uint32_t count = uint32_t(__popc(own));
      uint32_t upTo = __ockl_wfscan_add_u32(count, true);  // pairs of quads 0..lane
      uint32_t total = readlane_u(upTo, 63u);
      if (total > 64u) {
        // More than one round of pairs: drop those below their block's hiZ
        // first (one block at a time; a block that is not fast-cleared only
        // grows).
        const uint32_t hz = lane < uint32_t(kPerRow * kGroupRows) ? uint32_t(sm.hiz[block_of(lane)]) : 0u;
        for (uint32_t left = __ockl_wfred_or_u32(own); left; left &= left - 1u) {
          const uint32_t k = uint32_t(__builtin_ctz(left)), bhz = readlane_u(hz, k);
          if (bhz != 1u) own &= maxZq <= bhz ? ~(1u << k) : ~0u;
        }
        if (STATS) {
          const uint32_t dropped = __ockl_wfred_add_u32(count - uint32_t(__popc(own)));
          bc.visited += dropped;
          bc.rejected += dropped;
        }
        count = uint32_t(__popc(own));
        upTo = __ockl_wfscan_add_u32(count, true);
        total = readlane_u(upTo, 63u);
      }

      for (uint32_t taken = 0; taken < total;) {
        // The next quads' pairs, 64 or fewer (a quad has at most 32), as
        // block << 6 | quad in submission order.
        const bool inRound = upTo > taken && upTo - taken <= 64u;
        const uint32_t last = 63u - uint32_t(__builtin_clzll(__ballot(inRound)));
        const uint32_t fill = readlane_u(upTo, last) - taken;
        uint32_t pos = upTo - count - taken;
        for (uint32_t mine = inRound ? own : 0u; mine; mine &= mine - 1u)
          sm.pairs[wave][pos++] = uint16_t(block_of(uint32_t(__builtin_ctz(mine))) << 6 | lane);
        taken += fill;
        wave_lds_fence();

        // One lane per pair: coverage.
        const bool active = lane < fill;
        const uint32_t pr = active ? uint32_t(sm.pairs[wave][lane]) : uint32_t(sm.pairs[wave][0]);
        const uint32_t pq = pr & 63u, pb = pr >> 6;
        const QuadRec& R = sm.recs[pq];
        const uint32_t info = uint32_t(__shfl(int(pairInfo), int(pq)));
        const int plx = int(pb % TBX), ply = int(pb / TBX);
        const uint32_t phz = sm.hiz[pb];
        const bool pwrap = info & 0x100u;
        const int pc = plx - int(info & 0xFFu);
        const int row = int(info >> 16) - 1024 + ply;
        float o[4], nx[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) nx[i] = R.nx[i];
        if (!pwrap) {
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = sm.entry[row * 12 + i];
          for (int t = 0; t < pc; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = o[i] + nx[i];
        } else {
          const int dd = (tby0 + ply) * bX + tbx0 + plx - int(R.fb);
          const int r = div_bx(dd, bX, invBX);
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = fold_n(fold_n(R.off[i], R.ny[i], r), nx[i], dd - r * bX);
        }
        const uint32_t modeZ = R.modeZ, mode = modeZ & 0xFFu, s01 = R.slope01, s23 = R.slope23;
        float pdDx = R.dDx, pdDy = R.dDy;
        const bool convex = mode == kModeConvex;
        uint64_t word[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t tc = uint32_t(max(cvtt_x86(o[i]), 0));
          const uint32_t sl = i == 0 ? s01 & 0xFFFFu : i == 1 ? s01 >> 16 : i == 2 ? s23 & 0xFFFFu : s23 >> 16;
          word[i] = sm.cov[(sl | (convex ? tc : min(tc, 63u))) & 4095u];
        }
        const uint64_t A = word[0], B = word[1], C = word[2], D = word[3];
        // Convex, or one triangle (which leaves an edge out); concave quads are
        // rare enough for a branch of their own.
        uint64_t mask = (A & C) & ((B | (mode == kModeTriangle1 ? ~0ull : 0ull)) & (D | (mode == kModeTriangle0 ? ~0ull : 0ull)));
        const bool concave = mode >= kModeConcaveRight && mode <= kModeConcaveCenter;
        if (__ballot(concave) != 0ull && concave)
          mask = mode == kModeConcaveRight    ? (A | D) & (B & C)
                 : mode == kModeConcaveCenter ? (A & B) | (C & D)
                                              : (A & D) & (B | C);
        // Any offset >= 63 (a NaN is not): fmaxf leaves NaNs out.
        const bool outside = fmaxf(fmaxf(o[0], o[1]), fmaxf(o[2], o[3])) >= 63.0f;
        const uint64_t cm = __ballot(convex);
        uint64_t live = __ballot(active && !(phz != 1u && phz >= (modeZ >> 16))) &
                        ((cm & ~__ballot(outside)) | (~cm & __ballot(mask != 0ull)));
        if (STATS) {
          bc.visited += fill;
          bc.rejected += fill - uint32_t(__popcll(live));
        }
        // What the pair's turn needs, as scalars by readlane: column steps to
        // its samples, wrap flag and maximum depth; its depth gradients, its
        // mask (one bit a lane) and where its samples are (any address when
        // wrapped).
        const uint32_t desc = uint32_t(pwrap ? 0 : pc) | (pwrap ? 0x10u : 0u) | (modeZ & 0xFFFF0000u);
        const uint32_t maskLo = uint32_t(mask), maskHi = uint32_t(mask >> 32);
        const uint32_t sampleAt = pwrap ? 0u : uint32_t(row * 12 + 4);
        // Loaded before the loop, whose waits would otherwise cover its prefetches.
        asm volatile("" : "+v"(pdDx), "+v"(pdDy));

        // The pairs that cover pixels, block by block, a block's in submission
        // order; the next block's depth and the next pair's depth sample are
        // loaded while a pair is merged.
        uint32_t head = 0, b = 0, dNext = 0;
        auto fetch_block = [&]() {
          head = uint32_t(__builtin_ctzll(live));
          b = readlane_u(pb, head);
          dNext = sm.depth[b * 64u + lane];
        };
        if (live) fetch_block();
        while (live) {
          const uint32_t block = b, hz = readlane_u(phz, head);
          uint64_t same = live & __ballot(pb == block);
          live &= ~same;
          // `test` is what the hiZ reject compares with a quad's maximum depth
          // in every lane: the block's hiZ until its first write here, then its
          // depth.  `floor` is what a write is merged with: 0 while the block
          // reads as fast-cleared, else its depth.
          bool dirty = false, cleared = hz == 1u;
          uint32_t test = hz, floor = cleared ? 0u : dNext, win = kNoWinner;
          uint32_t* const winners =
              LABELS ? winner + ((size_t(tby0) + block / TBX) * size_t(bX) + size_t(tbx0) + block % TBX) * 64u + lane
                     : nullptr;
          if (LABELS && !cleared) win = *winners;
          uint32_t at = uint32_t(__builtin_ctzll(same));
          float vNext = sm.entry[readlane_u(sampleAt, at) + uint32_t(kLane)];
          if (live) fetch_block();
          do {
            const uint32_t turn = at, dsc = readlane_u(desc, turn);
            float v = vNext;
            same &= same - 1ull;
            if (same) {
              at = uint32_t(__builtin_ctzll(same));
              vNext = sm.entry[readlane_u(sampleAt, at) + uint32_t(kLane)];
            }
            if (__ballot(test < (dsc >> 16)) == 0ull) {
              if (STATS) bc.rejected++;
              continue;
            }
            if (STATS) bc.written++;
            const float dDx = readlane_f(pdDx, int(turn)), dDy = readlane_f(pdDy, int(turn));
            if (__builtin_expect(!(dsc & 0x10u), 1)) {
              if (TBX > 8 && (dsc & 8u)) {
                v = v + dDx; v = v + dDx; v = v + dDx; v = v + dDx;
                v = v + dDx; v = v + dDx; v = v + dDx; v = v + dDx;
              }
              if (dsc & 4u) {
                v = v + dDx; v = v + dDx; v = v + dDx; v = v + dDx;
              }
              if (dsc & 2u) {
                v = v + dDx; v = v + dDx;
              }
              if (dsc & 1u) v = v + dDx;
            } else {
              const QuadRec& W = sm.recs[readlane_u(pq, turn)];
              const int dd = (tby0 + int(block) / TBX) * bX + tbx0 + int(block) % TBX - int(W.fb);
              const int r = div_bx(dd, bX, invBX);
              float base, stepY, stepX;
              quad_component(W, 4u + uint32_t(kLane), base, stepY, stepX);
              v = fold_n(fold_n(base, stepY, r), stepX, dd - r * bX);
            }
            // Rows 0/1 and 8/9 from the plane, rows 2-7 as PAVGW of them.
            if (right) v = fmaf(dDx, 0.5f, v);
            const uint32_t top = pack_depth(v), bottom = pack_depth(dDy + v);
            const uint32_t mid = avg_u16(top, bottom), mean = avg_u16(low ? bottom : top, mid);
            const uint64_t pm = uint64_t(readlane_u(maskLo, turn)) | uint64_t(readlane_u(maskHi, turn)) << 32;
            const uint32_t d = lane_select(pm, odd ? mean : (low ? mid : top));
            if (LABELS) {
              // The first write of a cleared block sets every pixel's winner
              // (none where the written depth is 0), later ones only where they
              // raise the depth.
              const uint32_t batch = sm.qid[readlane_u(pq, turn)] >> 3;
              win = cleared ? (d != 0u ? batch : kNoWinner) : (d > floor ? batch : win);
            }
            test = floor = max(d, floor);
            dirty = true;
            cleared = false;
            // hiZ == 1 after this write (no pixel at 0 and one at 1) reads as
            // fast-cleared to the next one.
            if (__ballot(test == 0u) == 0ull && __ballot(test == 1u) != 0ull) {
              cleared = true;
              floor = 0u;
            }
          } while (same);
          if (dirty) {
            sm.depth[block * 64u + lane] = uint16_t(test);
            const uint32_t mn = __ockl_wfred_min_u32(test);
            if (lane == 0) sm.hiz[block] = uint16_t(mn);
            if (LABELS) *winners = win;
          }
        }
        wave_lds_fence();  // the pair list is reused
      }
    }
    q0 = q1;
    if (q0 < n) __syncthreads();  // the fold table is reused
  }
  return tB;
}

// query2D restricted to the tile (Rasterizer.cpp:283-349), by one wave: 1 if a
// pixel of the rectangle in the tile is visible, and with EARLY 2 if a block
// of the rectangle in it has hiZ 0 or 1; 0 otherwise.  One lane per block for
// the hiZ tests, then, where no interior block is visible, one lane per pixel
// for each block at the rectangle's border that passed, four at a time.  Any
// order of the blocks gives the same answer.
//
// EARLY: query2D evaluated ahead of the item's turn.  A block with hiZ >= 2
// can never read as cleared (hiZ == 1) again, since its minimum only grows:
// every later write max-merges, so its depth and hiZ only grow, and every test
// of query2D (the hiZ skip and the row test) can only move from visible to not
// visible.  So a result of 0 is the answer the tile gives at the item's turn.
// A cleared block's next write replaces its stale depth, and a block at hiZ 0
// could reach exactly 1, so neither proves anything.
template <int TBX, int TBY, bool EARLY>
__device__ __forceinline__ uint32_t query_tile(const ItemLocal& S, const TileSmem<TBX, TBY>& sm, int tbx0, int tbx1,
                                               int tby0, int tby1, uint32_t lane) {
  constexpr int kSteps = TBX * TBY / 64;  // 64 blocks a step
  const int x0 = int(uniform(S.qMinX)), x1 = int(uniform(S.qMaxX));
  const int y0 = int(uniform(S.qMinY)), y1 = int(uniform(S.qMaxY));
  const uint32_t maxZ = uniform(S.qMaxZ);
  uint64_t border[kSteps];
#pragma unroll
  for (int t = 0; t < kSteps; ++t) {
    const int lb = 64 * t + int(lane), bx = tbx0 + lb % TBX, by = tby0 + lb / TBX;
    const bool in = bx >= x0 >> 3 && bx <= x1 >> 3 && by >= y0 >> 3 && by <= y1 >> 3 && bx <= tbx1 && by <= tby1;
    const uint32_t hz = sm.hiz[lb];
    if (EARLY && __ballot(in && hz <= 1u) != 0ull) return 2u;
    const bool open = in && maxZ > hz;
    const bool whole = x0 <= 8 * bx && x1 >= 8 * bx + 7 && y0 <= 8 * by && y1 >= 8 * by + 7;
    if (__ballot(open && whole) != 0ull) return 1u;
    border[t] = __ballot(open);
  }
  const int px = int(lane & 7u), py = int(lane >> 3);
#pragma unroll
  for (int t = 0; t < kSteps; ++t) {
    for (uint64_t m = border[t]; m;) {
      bool hit = false;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int lb = 64 * t + (m ? __builtin_ctzll(m) : 0);
        const bool some = m != 0ull;
        m &= m - 1ull;
        const int x = 8 * (tbx0 + lb % TBX) + px, y = 8 * (tby0 + lb / TBX) + py;
        hit |= some && x >= x0 && x <= x1 && y >= y0 && y <= y1 && uint32_t(sm.depth[lb * 64 + int(lane)]) < maxZ;
      }
      if (__ballot(hit) != 0ull) return 1u;
    }
  }
  return 0u;
}

__device__ __forceinline__ bool box_touches(uint64_t bb, int tbx0, int tbx1, int tby0, int tby1) {
  const int c0 = int(bb & 0xFFFF), c1 = int((bb >> 16) & 0xFFFF), r0 = int((bb >> 32) & 0xFFFF), r1 = int(bb >> 48);
  return c0 <= c1 && c0 <= tbx1 && c1 >= tbx0 && r0 <= tby1 && r1 >= tby0;
}

// A setup record as five 16-byte words, each loaded whole and all before any
// is used (taken field by field, the compiler loads some only once a test on
// the others has passed).
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;
struct RecWords {
  u32x4 w[5];
};
static_assert(sizeof(QuadRec) == sizeof(RecWords) && offsetof(QuadRec, ny) == 16 && offsetof(QuadRec, off) == 32 &&
                  offsetof(QuadRec, fb) == 60 && offsetof(QuadRec, range) == 64 && offsetof(QuadRec, modeZ) == 68,
              "QuadRec layout");
__device__ __forceinline__ RecWords load_rec(const QuadRec* __restrict__ at) {
  const u32x4* p = reinterpret_cast<const u32x4*>(at);
  RecWords r = {{p[0], p[1], p[2], p[3], p[4]}};
  asm volatile("" : "+v"(r.w[0]), "+v"(r.w[1]), "+v"(r.w[2]), "+v"(r.w[3]), "+v"(r.w[4]));
  return r;
}

// Whether a quad may cover a pixel of the tile: its blocks touch the tile,
// and no edge is outside for every block they share.  The block loop folds
// each edge offset as off + nY + ... + nY (row steps) + nX + ... + nX (column
// steps) in float; after k steps the fold differs from the exact off + r*nY +
// c*nX by at most k * max|partial sum| * 2^-24 (each rounding is within half
// an ulp), and the corner values below by a few roundings more, so a minimum
// over the corners of at least 63 + that bound (taken more than twice over)
// proves the offset test (Rasterizer.cpp:1158) or the clamped lookup of
// bucket 63, whose table entry is empty (:599), rejects every block.  For the
// non-convex modes the offset must also stay below 2^31, where the truncation
// would wrap to bucket 0.  Infinities and NaNs make the bound infinite or NaN,
// which proves nothing.  Quads whose block index wrapped in the 16-bit
// multiply span whole rows and are never rejected by an edge.  A pass is bound
// by its loads' latency and then by these instructions: with double arithmetic
// and integer divisions the scans of 128 city frames in flight took 185 ms of
// work-group time, with these 145 ms.
__device__ __forceinline__ bool quad_touches_tile(const RecWords& R, int tbx0, int tbx1, int tby0, int tby1, int bX,
                                                  float invBX) {
  const int fb = int(R.w[3].w), rangeX = int(R.w[4].x & 0xFFFFu), rangeY = int(R.w[4].x >> 16);
  if (rangeX == 0) return false;  // not drawn
  const int minY = div_bx(fb, bX, invBX), minX = fb - minY * bX;
  if (minX + rangeX > bX) return minY <= tby1 && minY + rangeY >= tby0;
  const int c0 = max(tbx0 - minX, 0), c1 = min(tbx1 - minX, rangeX - 1);
  const int r0 = max(tby0 - minY, 0), r1 = min(tby1 - minY, rangeY - 1);
  if (c0 > c1 || r0 > r1) return false;
  const uint32_t mode = R.w[4].y & 0xFFu;
  const float fr0 = float(r0), fr1 = float(r1), fc0 = float(c0), fc1 = float(c1);
  const float steps = fr1 + fc1 + 8.0f;
  bool out[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float o = bitsf(R.w[2][e]), nx = bitsf(R.w[0][e]), ny = bitsf(R.w[1][e]);
    const float a = fmaf(fr0, ny, o), b = fmaf(fr1, ny, o);
    const float loX = fminf(fc0 * nx, fc1 * nx), hiX = fmaxf(fc0 * nx, fc1 * nx);
    const float bound = fmaf(fr1, __builtin_fabsf(ny), fmaf(fc1, __builtin_fabsf(nx), __builtin_fabsf(o)));
    const float err = steps * fmaf(bound, 0x1p-22f, 0x1p-120f);
    out[e] = (fminf(a, b) + loX) - err >= 63.0f &&
             (mode == kModeConvex || (fmaxf(a, b) + hiX) + err < 2147483648.0f);
  }
  bool misses = false;
  switch (mode) {
    case kModeConvex: misses = out[0] || out[1] || out[2] || out[3]; break;
    case kModeTriangle0: misses = out[0] || out[1] || out[2]; break;
    case kModeTriangle1: misses = out[0] || out[2] || out[3]; break;
    case kModeConcaveRight: misses = out[1] || out[2] || (out[0] && out[3]); break;
    case kModeConcaveLeft: misses = out[0] || out[3] || (out[1] && out[2]); break;
    case kModeConcaveCenter: misses = (out[0] || out[1]) && (out[2] || out[3]); break;
  }
  return !misses;
}

// The blocks that a quad whose block index did not wrap shares with the tile.
__device__ __forceinline__ uint32_t quad_blocks(const RecWords& R, int tbx0, int tbx1, int tby0, int tby1, int bX,
                                                float invBX) {
  const int fb = int(R.w[3].w), minY = div_bx(fb, bX, invBX), minX = fb - minY * bX;
  const int columns = min(tbx1, minX + int(R.w[4].x & 0xFFFFu) - 1) - max(tbx0, minX) + 1;
  const int rows = min(tby1, minY + int(R.w[4].x >> 16) - 1) - max(tby0, minY) + 1;
  return uint32_t(columns * rows);
}

// Whether every block that a quad may write in the tile already rejects it (hiZ
// at or above its largest depth), for a quad of at most kHiddenBlocks blocks in
// the tile.  Only blocks with hiZ >= 2 count: their minimum only grows, so they
// still reject it at its turn (a block at hiZ 0 could come to read as cleared).
// Where most quads are hidden this spares them the staging and the draw's two
// phases: a 4K frame of 12,000 icospheres 0.71 ms without, 0.47 ms with it.
constexpr int kHiddenBlocks = 64;
template <int TBX, int TBY>
__device__ __forceinline__ bool quad_hidden(const RecWords& R, const TileSmem<TBX, TBY>& sm, int tbx0, int tbx1,
                                            int tby0, int tby1, int bX, float invBX) {
  const int fb = int(R.w[3].w), rangeX = int(R.w[4].x & 0xFFFFu), rangeY = int(R.w[4].x >> 16);
  const uint32_t maxZ = R.w[4].y >> 16;
  const int minY = div_bx(fb, bX, invBX), minX = fb - minY * bX;
  const int x0 = max(tbx0, minX) - tbx0, x1 = min(tbx1, minX + rangeX - 1) - tbx0;
  const int y0 = max(tby0, minY) - tby0, y1 = min(tby1, minY + rangeY - 1) - tby0;
  const int n = (x1 - x0 + 1) * (y1 - y0 + 1);
  if (minX + rangeX > bX || n > kHiddenBlocks) return false;
  bool open = false;
  int x = x0, lb = y0 * TBX + x0;
  for (int i = 0; i < n && !open; i += 4) {
    uint32_t hz[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      hz[j] = i + j < n ? uint32_t(sm.hiz[lb]) : 0xFFFFu;
      const bool wrap = x == x1;
      lb += wrap ? TBX - (x1 - x0) : 1;
      x = wrap ? x0 : x + 1;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) open |= hz[j] < 2u || hz[j] < maxZ;
  }
  return !open;
}

// Tile-overlap tests shared by the prep kernel's tile count and the frame
// kernel (they must agree exactly).
template <int TBX, int TBY>
__device__ __forceinline__ bool query_overlaps_tile(uint32_t qMinX, uint32_t qMaxX, uint32_t qMinY, uint32_t qMaxY,
                                                   uint32_t tX, uint32_t tY) {
  return tX >= (qMinX >> 3) / TBX && tX <= (qMaxX >> 3) / TBX && tY >= (qMinY >> 3) / TBY &&
         tY <= (qMaxY >> 3) / TBY;
}

// Relevance of one item to a tile: bit 0 the query rectangle overlaps it,
// bit 1 some valid quad's blocks do; status in bits 2-3; 0 when neither or
// when the item is not drawn.
template <int TBX, int TBY>
__device__ __forceinline__ uint32_t tile_relevance(const ItemState& S, uint32_t tX, uint32_t tY, int tbx0, int tbx1,
                                                   int tby0, int tby1) {
  const uint32_t status = S.status;
  if (status == kStatusSkip) return 0u;
  const bool q = status == kStatusTest && query_overlaps_tile<TBX, TBY>(S.qMinX, S.qMaxX, S.qMinY, S.qMaxY, tX, tY);
  const bool f = S.fp[0] <= S.fp[1] && int(S.fp[0]) <= tbx1 && int(S.fp[1]) >= tbx0 && int(S.fp[2]) <= tby1 &&
                 int(S.fp[3]) >= tby0;
  return (q || f) ? ((q ? 1u : 0u) | (f ? 2u : 0u) | (status << 2)) : 0u;
}

// done[i] packs, over the tiles of item i's query rectangle, the number of
// tiles that have contributed (bits 0-15) and how many found a visible pixel
// (bits 16-31).  The word is all that passes between tiles (each reads and
// writes its own depth, hiZ and winners only), so its additions and loads are
// relaxed: a release writes the XCD's L2 back before each addition and an
// acquire drops the cached records after each load.  With those, one 1080p city
// frame took 250 us, the raster launches of 20 and 128 city frames in flight
// 1.55 and 5.05 ms; without, 217 us, 0.82 and 3.08 ms.
constexpr uint32_t kDoneCountMask = 0xFFFFu;
constexpr uint32_t kDoneVisibleOne = 0x10000u;

// One screen tile of one view: items [itemBegin, itemEnd) of the launch are
// walked in draw order against the tile's depth and hiZ held in LDS, then the
// tile is written back.  Shared by the single-view frame kernel (one
// work-group per tile, gated query items) and the multi-view persistent
// kernel (work-groups take (view, tile) units from a queue).
struct TileJob {
  const ItemDesc* items;
  const ItemState* state;
  uint32_t itemBegin, itemEnd;
  int bX, bY;
  uint32_t tX, tY;
  const QuadRec* recs;
  const uint64_t* groupBox;
  const uint64_t* itemBox;  // optional: what each item may touch
  uint16_t* depth;
  uint16_t* hiz;
  uint16_t* tileMin;
  uint32_t pyrX;
  uint32_t* done;
  uint32_t* err;
  uint64_t timeoutTicks;
  uint32_t* winner;  // labelled draws: per-pixel winners (block-linear), and
  uint32_t* labels;  // per-batch counts of written blocks each batch wins
  const uint32_t* list;  // optional: this tile's relevant items, in submission order
  uint32_t listLen;
};

// LABELS (8x8-block tiles): the draw tracks each pixel's winning batch, and
// once the tile is final every written block adds one to the label of each
// distinct batch that wins one of its pixels.
//
// BOXED: with item boxes (TileJob::itemBox), which a thread tests four at a time.
template <int TBX, int TBY, int NW, bool STATS, bool LABELS, bool BOXED>
__device__ __forceinline__ void process_tile(const TileJob& J, TileSmem<TBX, TBY>& sm,
                                             const uint64_t* __restrict__ cov, bool& covLoaded,
                                             uint64_t (&ctr)[kFrameStatWords]) {
  static_assert(!LABELS || (TBX == 8 && TBY == 8), "only 8x8-block tiles hold quad numbers");
  auto stamp = []() -> uint64_t { return STATS ? __builtin_amdgcn_s_memrealtime() : 0; };
  // Opaque, so that what a tile derives from it is not held in registers across
  // the multi-view kernel's loop over tiles (at 128 registers that spilled).
  uint32_t tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  tid &= 64u * NW - 1u;
  const uint32_t lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t tX = J.tX, tY = J.tY;
  const int bX = J.bX, bY = J.bY;
  const int tbx0 = int(tX) * TBX, tby0 = int(tY) * TBY;
  const int tbx1 = min(tbx0 + TBX, bX) - 1, tby1 = min(tby0 + TBY, bY) - 1;
  const float invBX = 1.0f / float(bX);

  auto relevance = [&](uint32_t i) -> uint32_t {
    return tile_relevance<TBX, TBY>(J.state[i], tX, tY, tbx0, tbx1, tby0, tby1);
  };
  // The tile's items: its binned list (the items relevant to it, in
  // submission order) when the launch has one, else the whole item range.
  const uint32_t nList = J.list ? J.listLen : J.itemEnd - J.itemBegin;
  auto item_at = [&](uint32_t pos) -> uint32_t { return J.list ? J.list[pos] : J.itemBegin + pos; };

  int involved = 0;
  constexpr uint32_t NT = 64u * NW;
  constexpr uint32_t kItemWindow = TileSmem<TBX, TBY>::kItemWindow;
  static_assert(NT >= kItemWindow, "the item window gathers one item per thread");
  constexpr uint32_t kPerThread = BOXED ? 4 : 1;
  if (J.list) involved = nList > 0u;
  else if (BOXED)
    for (uint32_t i = 4u * tid; i < nList && !involved; i += 4u * NT)
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j)
        involved |= i + j < nList && box_touches(J.itemBox[J.itemBegin + i + j], tbx0, tbx1, tby0, tby1);
  else
    for (uint32_t i = J.itemBegin + tid; i < J.itemEnd && !involved; i += NT) involved = relevance(i) != 0u;
  if (!__syncthreads_or(involved)) return;

  const uint64_t tLoad = stamp();
  if (!covLoaded) {
    for (uint32_t i = tid; i < 4096; i += NT) sm.cov[i] = cov[i];
    covLoaded = true;
  }
  constexpr int NB = TBX * TBY;
  for (int rrow = int(tid); rrow < NB * 8; rrow += int(NT)) {
    const int lb = rrow >> 3, y = rrow & 7;
    const int gx = tbx0 + lb % TBX, gy = tby0 + lb / TBX;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (gx <= tbx1 && gy <= tby1)
      v = *reinterpret_cast<const uint4*>(J.depth + (size_t(gy) * bX + gx) * 64 + y * 8);
    *reinterpret_cast<uint4*>(&sm.depth[lb * 64 + y * 8]) = v;
  }
  for (int lb = int(tid); lb < NB; lb += int(NT)) {
    const int gx = tbx0 + lb % TBX, gy = tby0 + lb / TBX;
    sm.hiz[lb] = (gx <= tbx1 && gy <= tby1) ? J.hiz[size_t(gy) * bX + gx] : uint16_t(0xFFFF);
  }

  BlockCounters bc;
  uint32_t rPar = 0, wPar = 0;
  uint32_t fill = 0;  // quads staged in sm.recs and not yet drawn
  bool drew = false;  // before the first draw there is little to hide a quad
  // The window's current block of 64 slots: the lane's item, its flags and the
  // groups it is drawn with; masks of the items with a share of query2D in the
  // tile, with quads in it and with quads in it that need a decision.
  uint32_t block = 0, laneIndex = 0, laneFlags = 0, laneGroups = 0;
  uint64_t shares = 0, quads = 0, waits = 0;
  // Wave 0: whose share was given, which of those with quads are decided and
  // which of those visible; whose early evaluation failed since the last draw.
  uint64_t given = 0, decided = 0, visible = 0, tried = 0;
  if (STATS) {
    if (tid < 4) sm.blockStats[tid] = 0;
    __syncthreads();
    if (tid == 0) ctr[kStatLoadTicks] += stamp() - tLoad;
  }
  const uint64_t tLoop = stamp();
  for (uint32_t wbase = 0; wbase < nList;) {
    // Gather this window's items that touch the tile, in draw order: every
    // thread tests one candidate (four in turn with item boxes, of which few
    // touch the tile), the first kItemWindow relevant ones are kept, and the
    // next window starts at the first relevant candidate not kept (or after the
    // last candidate tested).
    const uint32_t pos0 = wbase + kPerThread * tid;
    uint32_t rels = 0, count = 0;  // four bits a candidate
#pragma unroll
    for (uint32_t j = 0; j < kPerThread; ++j) {
      uint32_t rel = 0;
      if (pos0 + j < nList &&
          (!BOXED || box_touches(J.itemBox[J.itemBegin + pos0 + j], tbx0, tbx1, tby0, tby1)))
        rel = relevance(item_at(pos0 + j));
      rels |= rel << (4 * j);
      count += rel != 0u;
    }
    uint32_t off, sum;  // relevant candidates of the lanes before this one, and of the wave
    if constexpr (BOXED) {
      off = __ockl_wfscan_add_u32(count, true);
      sum = readlane_u(off, 63u);
      off -= count;
    } else {
      const uint64_t m = __ballot(rels != 0u);
      off = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
      sum = uint32_t(__popcll(m));
    }
    if (lane == 0) sm.wcnt[wPar][wave] = sum;
    if (tid == 0) sm.wnext = min(wbase + kPerThread * NT, nList);
    __syncthreads();
    uint32_t nRel = 0;
#pragma unroll
    for (uint32_t w = 0; w < NW; ++w) {
      off += w < wave ? sm.wcnt[wPar][w] : 0u;
      nRel += sm.wcnt[wPar][w];
    }
    wPar ^= 1u;
    nRel = min(nRel, kItemWindow);
    for (uint32_t j = 0; j < kPerThread; ++j) {
      const uint32_t rel = (rels >> (4 * j)) & 15u;
      if (!rel) continue;
      if (off >= kItemWindow) {
        if (off == kItemWindow) sm.wnext = pos0 + j;
        break;
      }
      const uint32_t i = item_at(pos0 + j);
      const ItemState& S = J.state[i];
      ItemLocal& L = sm.items[off++];
      L.index = i;
      L.flags = rel | S.expected << 16;
      L.qMinX = S.qMinX;
      L.qMaxX = S.qMaxX;
      L.qMinY = S.qMinY;
      L.qMaxY = S.qMaxY;
      L.qMaxZ = S.qMaxZ;
      const uint32_t qb = J.items[i].quadBase, qc = J.items[i].quadCount;
      L.quadBase = qb;
      L.quadCount = qc;
      uint64_t groups = ~0ull;
      uint32_t nGroups = 0;
      if ((rel & 2u) && qc > 0) {
        const uint32_t g0 = qb >> 6, g1 = (qb + qc - 1) >> 6;
        nGroups = g1 - g0 + 1;
        if (nGroups <= 64) {
          groups = 0;
          for (uint32_t gi = g0; gi <= g1; ++gi)
            if (box_touches(J.groupBox[gi], tbx0, tbx1, tby0, tby1)) groups |= 1ull << (gi - g0);
          nGroups = uint32_t(__popcll(groups));
        }
      }
      L.groups = groups;
      L.nGroups = nGroups;
    }
    __syncthreads();
    nRel = uniform(nRel);
    const uint32_t wnext = uniform(sm.wnext);

    // The window's items in draw order, in rounds.  Wave 0 goes over the items
    // from k on: it gives the tile's share of query2D where one is due, reads
    // the decisions of query items and waits for them, up to an item that needs
    // what is to be drawn before it to be drawn (or the block's end).  All waves
    // then scan the quads of the round's visible items together and stage them
    // behind those already staged; 64 are drawn at a time, what is left before
    // wave 0 goes on if it needs it, else with the next round's.
    //
    // What bounds it: the latency of this chain, tile after tile, and the issue
    // slots that it takes from the work-group on the same CU.  So the seven
    // other waves are at a barrier meanwhile, and small items share scans and
    // draws.  (With the eight waves sharing every query2D and every poll, two
    // barriers an item, and each item scanned and drawn by itself, a 4K frame
    // of 12,000 icospheres took 1.20 ms, with this 0.72 ms (0.41 ms with
    // quad_hidden and the item boxes, which came after); the raster launches of 20
    // and 128 city frames in flight 0.83 and 3.09 ms, with this 0.78 and 3.01 ms,
    // that of 64 mixed views 0.61 and 0.51 ms.)
    bool arrived = true;  // at a block of 64 slots
    uint32_t upTo = 0;    // lane i: groups of the round's drawn items up to item block + i
    for (uint32_t k = 0;;) {
      bool drain = false;
      uint64_t draw = 0;
      if (k == nRel) {
        if (fill == 0u || wnext < nList) break;
        drain = true;
      } else {
        if (arrived) {
          arrived = false;
          block = k;
          const bool in = k + lane < nRel;
          const ItemLocal& I = sm.items[in ? k + lane : k];
          laneIndex = I.index;
          laneFlags = in ? I.flags : 0u;
          laneGroups = I.nGroups;
          shares = __ballot((laneFlags & 1u) != 0u);
          quads = __ballot((laneFlags & 2u) != 0u);
          waits = __ballot((laneFlags & 2u) && ((laneFlags >> 2) & 3u) == uint32_t(kStatusTest));
          given = decided = visible = tried = 0;
        }
        if (wave == 0) {
          uint32_t at = k - block;
          while (true) {
            // The next item with a share due or a decision open; those before it
            // are decided.
            const uint64_t rest = ~0ull << at, open = waits & ~decided & rest;
            uint64_t due = shares & ~given & rest;
            const uint64_t events = due | open;
            at = events ? uint32_t(__builtin_ctzll(events)) : min(nRel - block, 64u);
            draw |= quads & (visible | ~waits) & rest & ((1ull << (at & 63u)) - (at < 64u ? 1ull : 2ull));
            if (events == 0ull) break;
            const uint64_t turn = 1ull << at;
            const bool pending = draw != 0ull || fill != 0u;
            if (due & turn) {
              // This tile's share of query2D for the item, at its exact turn.
              if (pending) {
                drain = true;
                break;
              }
              const uint64_t tq = stamp();
              const bool found = query_tile<TBX, TBY, false>(sm.items[block + at], sm, tbx0, tbx1, tby0, tby1, lane);
              if (lane == at)
                __hip_atomic_fetch_add(&J.done[laneIndex], 1u + (found ? kDoneVisibleOne : 0u), __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
              given |= turn;
              if (found || readlane_u(laneFlags, at) >> 16 == 1u) {
                // It decides: a pixel is visible, or no other tile has a share.
                decided |= turn;
                visible |= found ? turn : 0ull;
              }
              if (STATS && lane == 0) {
                ctr[kStatQueryTicks] += stamp() - tq;
                ctr[kStatQueries]++;
              }
              continue;
            }
            // A query item is decided when every tile of its rectangle has given
            // its share, or one of them has seen a visible pixel: the counters of
            // the items up to the next share, together.
            const uint64_t ask = open & (due ? (due & (0ull - due)) - 1ull : ~0ull);
            uint32_t d = 0;
            if (__builtin_amdgcn_inverse_ballot_w64(ask))
              d = __hip_atomic_load(&J.done[laneIndex], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const uint64_t seen = __ballot(d >= kDoneVisibleOne) & ask;
            visible |= seen;
            decided |= seen | (__ballot((d & kDoneCountMask) >= laneFlags >> 16) & ask);
            if (decided & turn) continue;
            if (pending) {
              drain = true;
              break;
            }
            // Wait for it.  Meanwhile give later items' shares early where the
            // tile's state already proves that they see nothing.
            const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
            if (STATS && lane == 0) ctr[kStatWaits]++;
            const uint32_t expected = readlane_u(laneFlags, at) >> 16;
            const uint32_t* counter = &J.done[readlane_u(laneIndex, at)];
            while (true) {
              d = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              const uint32_t err = __hip_atomic_load(J.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              const uint64_t later = due & ~tried;
              if (later != 0ull) {
                const uint32_t c = uint32_t(__builtin_ctzll(later));
                const uint64_t bit = 1ull << c;
                const bool none = query_tile<TBX, TBY, true>(sm.items[block + c], sm, tbx0, tbx1, tby0, tby1, lane) == 0u;
                if (none) {
                  if (lane == c) __hip_atomic_fetch_add(&J.done[laneIndex], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                  given |= bit;
                  due &= ~bit;
                  if (readlane_u(laneFlags, c) >> 16 == 1u) decided |= bit;
                } else {
                  tried |= bit;
                }
                if (STATS && lane == 0) {
                  ctr[kStatEarlyTried]++;
                  if (none) ctr[kStatEarlyAnswered]++;
                }
              } else {
                __builtin_amdgcn_s_sleep(1);
              }
              const uint32_t now = uniform(d);
              if (now >= kDoneVisibleOne) visible |= turn;
              if (now >= kDoneVisibleOne || (now & kDoneCountMask) >= expected) break;
              if (__builtin_amdgcn_s_memrealtime() - t0 > J.timeoutTicks || uniform(err) != 0u) {
                // After one wait of the launch has timed out, the others stop
                // waiting too (the launch's result is reported as an error).
                if (lane == 0)
                  __hip_atomic_fetch_or(J.err, uint32_t(kErrTimeout), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
              }
            }
            decided |= turn;
            if (STATS && lane == 0) ctr[kStatWaitTicks] += __builtin_amdgcn_s_memrealtime() - t0;
          }
          if (lane == 0)
            sm.run[rPar] = make_uint4(at, drain ? 1u : 0u, uint32_t(draw), uint32_t(draw >> 32));
          if (STATS && lane == 0) ctr[kStatItems] += at - (k - block);
        }
        __syncthreads();
        const uint4 r = sm.run[rPar];
        rPar ^= 1u;
        const uint32_t end = uniform(r.x);
        drain = uniform(r.y) != 0u;
        draw = uniform(r.z) | uint64_t(uniform(r.w)) << 32;
        k = block + end;
        arrived = end == 64u;
      }
      uint32_t nGroups = 0;
      if (draw != 0ull) {
        upTo = __ockl_wfscan_add_u32(lane_select(draw, laneGroups), true);
        nGroups = readlane_u(upTo, 63u);
      }
      // Scan the run, one 64-quad group that may touch the tile per wave and
      // pass, and draw.
      const uint64_t tr = stamp();
      for (uint32_t f0 = 0; f0 < nGroups || (drain && fill != 0u); f0 += NW) {
        uint32_t total = fill, pos = 0, quad = 0, hidden = 0;  // hidden: pairs of a quad left out
        bool hit = false;
        if (f0 < nGroups) {
          const uint64_t tScan = stamp();
          if (STATS && tid == 0) ctr[kStatPasses]++;
          const uint32_t f = f0 + wave;
          if (f < nGroups) {
            const uint32_t r = uint32_t(__popcll(__ballot(upTo <= f)));
            const uint32_t j = f - (r ? readlane_u(upTo, r - 1u) : 0u);  // the item's j-th group
            const ItemLocal& L = sm.items[block + r];
            const uint64_t groups = L.groups;
            const uint32_t first = L.quadBase, past = first + L.quadCount;
            uint32_t g = j;
            if (((past - 1u) >> 6) - (first >> 6) < 64u) {
              const bool set = (groups >> lane) & 1ull;
              const uint32_t rank = uint32_t(__popcll(groups & ((1ull << lane) - 1ull)));
              g = uint32_t(__builtin_ctzll(__ballot(set && rank == j)));
            }
            quad = ((first >> 6) + g) * 64u + lane;
            if (quad >= first && quad < past) {
              const RecWords rec = load_rec(&J.recs[quad]);
              hit = quad_touches_tile(rec, tbx0, tbx1, tby0, tby1, bX, invBX) &&
                    !(drew && quad_hidden<TBX, TBY>(rec, sm, tbx0, tbx1, tby0, tby1, bX, invBX));
              if (STATS && !hit && quad_touches_tile(rec, tbx0, tbx1, tby0, tby1, bX, invBX))
                hidden = quad_blocks(rec, tbx0, tbx1, tby0, tby1, bX, invBX);
            }
          }
          if (STATS) {
            hidden = __ockl_wfred_add_u32(hidden);
            bc.visited += hidden;
            bc.rejected += hidden;
          }
          const uint64_t hm = __ballot(hit);
          const uint32_t hpre =
              __builtin_amdgcn_mbcnt_hi(uint32_t(hm >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(hm), 0u));
          if (lane == 0) sm.wcnt[wPar][wave] = uint32_t(__popcll(hm));
          __syncthreads();
          pos = fill + hpre;
#pragma unroll
          for (uint32_t w = 0; w < NW; ++w) {
            pos += w < wave ? sm.wcnt[wPar][w] : 0u;
            total += sm.wcnt[wPar][w];
          }
          total = uniform(total);
          wPar ^= 1u;
          if (STATS && tid == 0) ctr[kStatScanTicks] += stamp() - tScan;
        }
        for (uint32_t k0 = 0; k0 < total; k0 += kQuadChunk) {
          const uint32_t n = min(kQuadChunk, total - k0);
          // Hits reload their record (just read, so from cache) rather than
          // hold it across the compaction, which made the compiler spill it.
          if (hit && pos >= k0 && pos < k0 + n) {
            sm.recs[pos - k0] = J.recs[quad];
            if (LABELS) sm.qid[pos - k0] = quad;
          }
          fill = n;
          if (n < kQuadChunk && !(drain && f0 + NW >= nGroups)) break;
          __syncthreads();
          const uint64_t tDraw = stamp();
          const uint64_t tB = draw_chunk<TBX, TBY, NW, STATS, LABELS>(sm, n, tbx0, tbx1, tby0, tby1, bX, invBX, wave,
                                                                      lane, bc, J.winner);
          fill = 0;
          drew = true;
          tried = 0;  // the tile's state changed: early evaluations that failed may now succeed
          if (STATS && tid == 0) ctr[kStatQuads] += n;
          __syncthreads();
          if (STATS && tid == 0) {
            const uint64_t t = stamp();
            ctr[kStatDrawTicks] += t - tDraw;
            ctr[kStatChunks]++;
            ctr[kStatPhaseATicks] += tB - tDraw;
            ctr[kStatPhaseBTicks] += t - tB;
          }
        }
      }
      if (STATS && tid == 0) ctr[kStatRasterTicks] += stamp() - tr;
    }
    __syncthreads();
    wbase = wnext;
  }

  if (STATS) {
    if (tid == 0) ctr[kStatLoopTicks] += stamp() - tLoop;
    if (lane == 0) {
      atomicAdd(&sm.blockStats[0], bc.visited);
      atomicAdd(&sm.blockStats[1], bc.rejected);
      atomicAdd(&sm.blockStats[2], bc.written);
      atomicAdd(&sm.blockStats[3], bc.foldSteps);
    }
    __syncthreads();
    if (tid == 0) {
      ctr[kStatBlocksVisited] += sm.blockStats[0];
      ctr[kStatBlocksRejected] += sm.blockStats[1];
      ctr[kStatBlocksWritten] += sm.blockStats[2];
      ctr[kStatFoldSteps] += sm.blockStats[3];
    }
  }
  if constexpr (LABELS) {
    // Each block is counted by the wave that drew it, which wrote its
    // winners; blocks still cleared were not written this frame.
    for (int lb = 0; lb < NB; ++lb) {
      const int lbx = lb % TBX, lby = lb / TBX;
      if (block_owner<NW>(lbx, lby) != wave) continue;
      const int gx = tbx0 + lbx, gy = tby0 + lby;
      if (gx > tbx1 || gy > tby1 || sm.hiz[lb] == 1u) continue;
      const uint32_t w = J.winner[(size_t(gy) * size_t(bX) + size_t(gx)) * 64u + lane];
      bool active = w != kNoWinner;
      while (true) {
        const uint64_t m = __ballot(active);
        if (m == 0ull) break;
        const uint32_t v = uint32_t(__builtin_amdgcn_readlane(int(w), int(__builtin_ctzll(m))));
        if (active && w == v) active = false;
        if (lane == 0) atomicAdd(&J.labels[v], 1u);
      }
    }
  }
  // Write the tile back.
  for (int rrow = int(tid); rrow < NB * 8; rrow += int(NT)) {
    const int lb = rrow >> 3, y = rrow & 7;
    const int gx = tbx0 + lb % TBX, gy = tby0 + lb / TBX;
    if (gx <= tbx1 && gy <= tby1)
      *reinterpret_cast<uint4*>(J.depth + (size_t(gy) * bX + gx) * 64 + y * 8) =
          *reinterpret_cast<const uint4*>(&sm.depth[lb * 64 + y * 8]);
  }
  for (int lb = int(tid); lb < NB; lb += int(NT)) {
    const int gx = tbx0 + lb % TBX, gy = tby0 + lb / TBX;
    if (gx <= tbx1 && gy <= tby1) J.hiz[size_t(gy) * bX + gx] = sm.hiz[lb];
  }
  // Min hiZ of each 8x8-block sub-tile for the query kernel (blocks outside
  // the buffer hold 0xFFFF and do not lower it).
  constexpr int kSubX = TBX / 8, kSubY = TBY / 8;
  for (int sub = int(wave); sub < kSubX * kSubY; sub += NW) {
    const int sx = sub % kSubX, sy = sub / kSubX;
    const int lb = (sy * 8 + int(lane >> 3)) * TBX + sx * 8 + int(lane & 7u);
    const uint32_t mn = __ockl_wfred_min_u32(uint32_t(sm.hiz[lb]));
    const uint32_t px = tX * kSubX + uint32_t(sx), py = tY * kSubY + uint32_t(sy);
    if (lane == 0 && px < J.pyrX && py * 8 < uint32_t(bY)) J.tileMin[py * J.pyrX + px] = uint16_t(mn);
  }
}

// Two work-groups per CU, as the multi-view kernel (at most 128 VGPRs with
// eight waves per group).
template <int TBX, int TBY, int NW, bool STATS, bool BOXED>
__global__ void __launch_bounds__(64 * NW, NW == 8 ? 4 : 2) rz_frame_kernel(FrameParams p) {
  __shared__ TileSmem<TBX, TBY> sm;
  // Observability counters, kept in LDS by thread 0 (unused unless STATS).
  __shared__ uint64_t ctr[kFrameStatWords];
  if (STATS && threadIdx.x < kFrameStatWords) ctr[threadIdx.x] = 0;
  const uint64_t tEntry = STATS ? __builtin_amdgcn_s_memrealtime() : 0;
  TileJob J;
  J.items = p.items;
  J.state = p.state;
  J.itemBegin = 0;
  J.itemEnd = p.nItems;
  J.bX = int(p.bX);
  J.bY = int(p.bY);
  J.tX = blockIdx.x % p.tilesX;
  J.tY = blockIdx.x / p.tilesX;
  J.recs = p.recs;
  J.groupBox = p.groupBox;
  J.itemBox = p.itemBox;
  J.depth = p.depth;
  J.hiz = p.hiz;
  J.tileMin = p.tileMin;
  J.pyrX = p.pyrX;
  J.done = p.done;
  J.err = p.err;
  J.timeoutTicks = p.timeoutTicks;
  J.winner = nullptr;
  J.labels = nullptr;
  J.list = nullptr;
  J.listLen = 0;
  bool covLoaded = false;
  process_tile<TBX, TBY, NW, STATS, false, BOXED>(J, sm, p.cov, covLoaded, ctr);
  if (STATS && threadIdx.x == 0) {
    ctr[kStatTotalTicks] = __builtin_amdgcn_s_memrealtime() - tEntry;
    for (int k = 0; k < kFrameStatWords; ++k) p.stats[size_t(blockIdx.x) * kFrameStatWords + k] = ctr[k];
  }
}

// Multi-view persistent raster: each work-group takes (view, tile) units from
// p.queue until the queue is exhausted.  Units are handed out in view order.
// Classified items never wait.  Query-gated items (p.done) wait only on
// other tiles of the same view; when every view's tiles fit in the grid and
// the grid is co-resident (the host checks both), the earliest unfinished
// view always has all its tiles running, so every wait ends (and each is
// bounded by p.timeoutTicks in any case).
// Two work-groups per CU (the LDS allows two): with eight waves each, every
// SIMD must hold four waves, i.e. at most 128 VGPRs per lane.  NW is 2, 4 or
// 8 (the item window gathers one item per thread of its first 128).
template <int TBX, int TBY, int NW, bool STATS, bool LABELS>
__global__ void __launch_bounds__(64 * NW, NW == 8 ? 4 : 2) rz_views_kernel(ViewsParams p) {
  __shared__ TileSmem<TBX, TBY> sm;
  __shared__ uint32_t unitSh;
  __shared__ uint64_t ctr[kFrameStatWords];
  if (STATS && threadIdx.x < kFrameStatWords) ctr[threadIdx.x] = 0;
  const uint64_t tEntry = STATS ? __builtin_amdgcn_s_memrealtime() : 0;
  bool covLoaded = false;
  // With a compacted unit list, only units that have items are handed out,
  // each carrying its view; else every unit, its view found by search.
  const uint32_t nHanded = p.unitList ? *p.nActive : p.nUnits;
  while (true) {
    if (threadIdx.x == 0) {
      const uint32_t u = __hip_atomic_fetch_add(p.queue, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      unitSh = u >= nHanded ? 0xFFFFFFFFu : p.unitList ? p.unitList[u] : u;
    }
    __syncthreads();
    const uint32_t entry = __builtin_amdgcn_readfirstlane(unitSh);
    __syncthreads();
    if (entry == 0xFFFFFFFFu) break;
    uint32_t lo = 0, t = 0;
    if (p.unitList) {
      lo = entry >> 20;
      t = entry & 0xFFFFFu;
    } else {
      uint32_t hi = p.nViews - 1;
      while (lo < hi) {
        const uint32_t mid = (lo + hi + 1) >> 1;
        if (p.views[mid].unitBase <= entry) lo = mid;
        else hi = mid - 1;
      }
      t = entry - p.views[lo].unitBase;
    }
    const ViewDesc& V = p.views[lo];
    const uint32_t unit = uniform(V.unitBase) + t, tilesX = uniform(V.tilesX);
    TileJob J;
    J.items = p.items;
    J.state = p.state;
    const uint32_t first = uniform(p.batchItems ? V.batchBase : V.itemBase);
    const uint32_t count = uniform(p.batchItems ? V.nBatches : V.nItems);
    J.itemBegin = first;
    J.itemEnd = first + count;
    J.bX = int(uniform(V.bX));
    J.bY = int(uniform(V.bY));
    J.tX = t % tilesX;
    J.tY = t / tilesX;
    J.recs = p.recs;
    J.groupBox = p.groupBox;
    J.itemBox = nullptr;
    J.depth = uniform(V.depth);
    J.hiz = uniform(V.hiz);
    J.tileMin = uniform(V.tileMin);
    J.pyrX = uniform(V.pyrX);
    J.done = p.done;
    J.err = p.err;
    J.timeoutTicks = p.timeoutTicks;
    J.winner = uniform(V.winner);
    J.labels = p.labels;
    J.list = p.lists ? p.lists + uniform(V.listBase) + size_t(t) * count : nullptr;
    J.listLen = p.lists ? uniform(p.listLen[unit]) : 0u;
    process_tile<TBX, TBY, NW, STATS, LABELS, false>(J, sm, p.cov, covLoaded, ctr);
    __syncthreads();
  }
  if (STATS) {
    // Words 0-2: block-loop counters; 3 onwards: the per-tile counters of
    // every unit summed, word 3 + kStatTotalTicks being the work-groups'
    // lifetimes.
    __syncthreads();
    if (threadIdx.x == 0) ctr[kStatTotalTicks] = __builtin_amdgcn_s_memrealtime() - tEntry;
    __syncthreads();
    if (threadIdx.x < kFrameStatWords)
      atomicAdd(&p.stats[3 + threadIdx.x], (unsigned long long)ctr[threadIdx.x]);
    if (threadIdx.x == 0) {
      atomicAdd(&p.stats[0], (unsigned long long)ctr[kStatBlocksVisited]);
      atomicAdd(&p.stats[1], (unsigned long long)ctr[kStatBlocksRejected]);
      atomicAdd(&p.stats[2], (unsigned long long)ctr[kStatBlocksWritten]);
    }
  }
}

// The units of one view (one work-group per view) that have items, in tile
// order, as view << 20 | tile, at unitTmp[view's unitBase ...], and their
// count in p.unitCounts[view].
__global__ void __launch_bounds__(256) rz_views_compact_kernel(ViewsParams p, uint32_t* __restrict__ unitTmp) {
  __shared__ uint32_t wcnt[4];
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
  const uint32_t v = blockIdx.x;
  const ViewDesc& V = p.views[v];
  // Units with more items first (buckets of floor(log2(items)), 8 and up
  // together at the top), tile order within a bucket: the tiles that the
  // others' query waits depend on most start first.  Any order within a view
  // keeps every wait finite (all of the earliest view's tiles run).
  uint32_t n = 0;
  for (int bucket = 7; bucket >= 0; --bucket) {
    for (uint32_t base = 0; base < V.nUnits; base += 256u) {
      const uint32_t t = base + tid;
      const uint32_t len = t < V.nUnits ? p.listLen[V.unitBase + t] : 0u;
      const int lg = len ? min(31 - __builtin_clz(len), 7) : -1;
      const bool has = lg == bucket;
      const uint64_t m = __ballot(has);
      const uint32_t pre = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
      if (lane == 0) wcnt[wave] = uint32_t(__popcll(m));
      __syncthreads();
      uint32_t off = n, total = 0;
#pragma unroll
      for (uint32_t w = 0; w < 4; ++w) {
        off += w < wave ? wcnt[w] : 0u;
        total += wcnt[w];
      }
      if (has) unitTmp[V.unitBase + off + pre] = (v << 20) | t;
      n += total;
      __syncthreads();
    }
  }
  if (tid == 0) p.unitCounts[v] = n;
}

// Concatenates the views' compacted units in view order into p.unitList
// (one work-group per view); the last view also writes the total.
__global__ void __launch_bounds__(256) rz_views_gather_kernel(ViewsParams p, const uint32_t* __restrict__ unitTmp) {
  const uint32_t v = blockIdx.x;
  uint32_t off = 0;
  for (uint32_t w = 0; w < v; ++w) off += p.unitCounts[w];
  const uint32_t n = p.unitCounts[v];
  const uint32_t src = p.views[v].unitBase;
  for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) p.unitList[off + k] = unitTmp[src + k];
  if (v == p.nViews - 1 && threadIdx.x == 0) *p.nActive = off + n;
}

__global__ void __launch_bounds__(256) rz_item_boxes_kernel(const ItemState* __restrict__ state, uint32_t n,
                                                            uint64_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const ItemState& S = state[i];
  uint32_t c0 = 0xFFFFu, c1 = 0u, r0 = 0xFFFFu, r1 = 0u;
  if (S.status != kStatusSkip) {
    if (S.fp[0] <= S.fp[1]) {
      c0 = S.fp[0];
      c1 = S.fp[1];
      r0 = S.fp[2];
      r1 = S.fp[3];
    }
    if (S.status == kStatusTest) {
      c0 = min(c0, S.qMinX >> 3);
      c1 = max(c1, S.qMaxX >> 3);
      r0 = min(r0, S.qMinY >> 3);
      r1 = max(r1, S.qMaxY >> 3);
    }
  }
  out[i] = c0 <= c1 ? uint64_t(c0) | uint64_t(c1) << 16 | uint64_t(r0) << 32 | uint64_t(r1) << 48 : kEmptyBox;
}

// Per item of a multi-view launch, the box in 8x8-block tiles (u16 x0, x1,
// y0, y1) that bounds every tile it is relevant to: the union of its
// footprint's tiles and, for a query-gated item, its query rectangle's;
// empty (x0 > x1) when the item is not drawn.
__global__ void __launch_bounds__(256) rz_item_tiles_kernel(ViewsParams p, uint32_t n, uint64_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const ItemState& S = p.state[i];
  // Tiles of tileB blocks: block >> sh, pixel >> (sh + 3).
  const uint32_t sh = p.views[p.items[i].view].tileB == 16u ? 4u : 3u;
  uint32_t x0 = 0xFFFFu, x1 = 0u, y0 = 0xFFFFu, y1 = 0u;
  if (S.status != kStatusSkip) {
    if (S.fp[0] <= S.fp[1]) {
      x0 = S.fp[0] >> sh;
      x1 = S.fp[1] >> sh;
      y0 = S.fp[2] >> sh;
      y1 = S.fp[3] >> sh;
    }
    if (S.status == kStatusTest) {
      x0 = min(x0, S.qMinX >> (sh + 3u));
      x1 = max(x1, S.qMaxX >> (sh + 3u));
      y0 = min(y0, S.qMinY >> (sh + 3u));
      y1 = max(y1, S.qMaxY >> (sh + 3u));
    }
  }
  out[i] = uint64_t(min(x0, 0xFFFFu)) | uint64_t(min(x1, 0xFFFFu)) << 16 | uint64_t(min(y0, 0xFFFFu)) << 32 |
           uint64_t(min(y1, 0xFFFFu)) << 48;
}

// Per-tile item lists of a multi-view launch: for each (view, tile) unit, the
// indices of the view's items whose tile box (rz_item_tiles_kernel) holds the
// tile, in submission order, at lists[views[v].listBase + tile * (items in
// view)], and their count in listLen[unit].  A box can hold a tile the item is
// not relevant to; the raster kernel's exact test drops those.  One wave per
// unit tests the items 64 at a time and compacts them with ballots (no
// barriers: a view's items are about a hundred, so a work-group per unit
// spent its time being scheduled).
__global__ void __launch_bounds__(256) rz_views_bin_kernel(ViewsParams p, const uint64_t* __restrict__ tileBox) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
  for (uint32_t unit = blockIdx.x * 4u + wave; unit < p.nUnits; unit += gridDim.x * 4u) {
    uint32_t lo = 0, hi = p.nViews - 1;
    while (lo < hi) {
      const uint32_t mid = (lo + hi + 1) >> 1;
      if (p.views[mid].unitBase <= unit) lo = mid;
      else hi = mid - 1;
    }
    const ViewDesc& V = p.views[lo];
    const uint32_t t = unit - V.unitBase;
    const uint32_t tX = t % V.tilesX, tY = t / V.tilesX;
    const uint32_t begin = p.batchItems ? V.batchBase : V.itemBase;
    const uint32_t end = begin + (p.batchItems ? V.nBatches : V.nItems);
    uint32_t* out = p.lists + V.listBase + size_t(t) * (end - begin);
    uint32_t n = 0;
    for (uint32_t base = begin; base < end; base += 64u) {
      const uint32_t i = base + lane;
      bool rel = false;
      if (i < end) {
        const uint64_t b = tileBox[i];
        rel = uint32_t(b & 0xFFFF) <= tX && tX <= uint32_t((b >> 16) & 0xFFFF) && uint32_t((b >> 32) & 0xFFFF) <= tY &&
              tY <= uint32_t(b >> 48);
      }
      const uint64_t m = __ballot(rel);
      const uint32_t pre = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
      if (rel) out[n + pre] = i;
      n += uint32_t(__popcll(m));
    }
    if (lane == 0) p.listLen[unit] = n;
  }
}

hipError_t launch_views_bin(const ViewsParams& p, uint32_t nItems, uint64_t* tileBox, hipStream_t stream) {
  if (p.nUnits == 0 || !p.lists) return hipSuccess;
  if (nItems) hipLaunchKernelGGL(rz_item_tiles_kernel, dim3((nItems + 255) / 256), dim3(256), 0, stream, p, nItems, tileBox);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(rz_views_bin_kernel, dim3(std::min<uint32_t>((p.nUnits + 3u) / 4u, 65535u)), dim3(256), 0,
                     stream, p, tileBox);
  return hipGetLastError();
}

hipError_t launch_views_compact(const ViewsParams& p, uint32_t* unitTmp, hipStream_t stream) {
  if (p.nUnits == 0 || !p.unitList) return hipSuccess;
  hipLaunchKernelGGL(rz_views_compact_kernel, dim3(p.nViews), dim3(256), 0, stream, p, unitTmp);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(rz_views_gather_kernel, dim3(p.nViews), dim3(256), 0, stream, p, static_cast<const uint32_t*>(unitTmp));
  return hipGetLastError();
}

// Per-item draw status of a frame: 0 not drawn, 1 rasterize<false>,
// 2 rasterize<true>.
__global__ void rz_status_kernel(const ItemState* __restrict__ state, const uint32_t* __restrict__ visible,
                                 uint32_t n, uint8_t* __restrict__ out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint32_t st = state[i].status;
  out[i] = uint8_t(st == kStatusTest ? ((visible[i] >> 16) != 0u ? 1u : 0u) : st);
}

// ---------------------------------------------------------------------------
// Queries, readback, clear.
// ---------------------------------------------------------------------------
// queryVisibility (Rasterizer.cpp:123-281) of a batch: lanes 0..BPW-1 of a
// wave each take one box for the depth-independent part (projection,
// frustum, near plane, rectangle), then the wave runs query2D for those that
// need it (query2d_boxes).  launch_query chooses BPW and WHOLE.
template <uint32_t BPW, bool WHOLE>
__global__ void __launch_bounds__(256) rz_query_kernel(QueryParams p) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t q = ((blockIdx.x * blockDim.x + threadIdx.x) >> 6) * BPW + lane;
  const bool valid = lane < BPW && q < p.n;
  QueryPre Q = {0, 0, 0, 0, 0, 0};
  if (valid) {
    const float* b = p.bounds + 8 * size_t(q);
    const float bmin[4] = {b[0], b[1], b[2], b[3]};
    const float bmax[4] = {b[4], b[5], b[6], b[7]};
    Q = query_pre(p.mvp, bmin, bmax, p.width, p.height, p.rcp);
  }
  const uint32_t clip = Q.kind == 1 ? 1u : 0u;
  const QueryBufs B = {p.depth, p.hiz, p.tileMin, p.bX, p.pyrX};
  const uint32_t vis = query2d_boxes<WHOLE>(Q, valid && Q.kind == 3, B, lane) ? 1u : clip;
  if (valid) {
    p.visible[q] = uint8_t(vis);
    if (p.needsClipping) p.needsClipping[q] = uint8_t(clip);
  }
  // The draws that set the error word have completed.
  if (p.words.out && blockIdx.x == 0 && threadIdx.x == 0) p.words.out[0] = *p.words.err;
}

// queryVisibility of one box, by one wave: the box comes with the launch and
// the answer goes straight to host memory, so a blocking call is one launch
// and one wait.  Latency bound: rz_query takes 15 us on an idle stream.  (With
// a copy of the box before it, and copies of the answer and of the error word
// after it, it took 41 us.)
__global__ void __launch_bounds__(64) rz_query_one_kernel(QueryParams p, QueryBox box) {
  const QueryPre Q = query_pre(p.mvp, box.lo, box.hi, p.width, p.height, p.rcp);
  const uint32_t clip = Q.kind == 1 ? 1u : 0u;
  uint32_t vis = clip;
  if (Q.kind == 3) {  // the same in every lane
    const QueryBufs B = {p.depth, p.hiz, p.tileMin, p.bX, p.pyrX};
    vis = query2d_wave(Q.minX, Q.maxX, Q.minY, Q.maxY, Q.maxZ, B, threadIdx.x) ? 1u : 0u;
  }
  if (threadIdx.x == 0) {
    // bit 0 visible, bit 1 needsClipping, bit 2 needsClipping was written
    p.words.out[1] = vis | (clip << 1) | (Q.kind != 0 ? 4u : 0u);
    p.words.out[0] = *p.words.err;
  }
}

__global__ void rz_host_words_kernel(HostWords words) { words.out[0] = *words.err; }

// queryVisibility over the queries of every view of a multi-view launch;
// blockIdx.y is the view.  A step holds many boxes, so one lane per box does
// the depth-independent part (projection, frustum, near plane, rectangle)
// and the wave then runs query2D for its boxes that need it.
__global__ void __launch_bounds__(256) rz_views_query_kernel(ViewsQueryParams p) {
  // The raster launch that sets the error word has completed.
  if (p.errOut && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) *p.errOut = *p.err;
  const uint32_t lane = threadIdx.x & 63u;
  const ViewDesc& V = p.views[blockIdx.y];
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;  // 64 boxes per wave
  const bool valid = k < V.nQueries;
  QueryPre Q = {0, 0, 0, 0, 0, 0};
  if (valid) {
    const float* b = V.queryBounds + 8 * size_t(k);
    const float bmin[4] = {b[0], b[1], b[2], b[3]};
    const float bmax[4] = {b[4], b[5], b[6], b[7]};
    Q = query_pre(V.mvp, bmin, bmax, V.width, V.height, p.rcp);
  }
  const uint32_t clip = Q.kind == 1 ? 1u : 0u;
  const QueryBufs B = {V.depth, V.hiz, V.tileMin, V.bX, V.pyrX};
  const uint32_t vis = query2d_boxes<false>(Q, valid && Q.kind == 3, B, lane) ? 1u : clip;
  if (valid) {
    V.queryVisible[k] = uint8_t(vis);
    V.queryClip[k] = uint8_t(clip);
  }
}

// clear (Rasterizer.cpp:107-121) of every view (blockIdx.y): hiZ := 1, the
// cleared mark, eight entries per 16-byte store (each view's hiZ buffer is its
// own allocation, holding whole groups of eight), and the per-tile min hiZ
// := 1.  The view table comes from `src`, the host's pinned copy with this
// step's matrices, read through its device mapping; the first work-group of
// each view copies the view's entry to `views`, which every later kernel of
// the step reads (no copy before the launch).
__global__ void rz_views_clear_kernel(const ViewDesc* __restrict__ src, ViewDesc* __restrict__ views) {
  const ViewDesc& V = src[blockIdx.y];
  if (blockIdx.x == 0 && threadIdx.x < sizeof(ViewDesc) / 16)
    reinterpret_cast<uint4*>(views + blockIdx.y)[threadIdx.x] =
        reinterpret_cast<const uint4*>(src + blockIdx.y)[threadIdx.x];
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (V.bX * V.bY + 8u) / 8u) reinterpret_cast<uint4*>(V.hiz)[i] = make_uint4(0x10001u, 0x10001u, 0x10001u, 0x10001u);
  if (i < V.pyrX * V.pyrY) V.tileMin[i] = 1;
}

__global__ void rz_query2d_kernel(uint32_t minX, uint32_t maxX, uint32_t minY, uint32_t maxY, uint32_t maxZ,
                                  QueryParams p) {
  const bool v = query2d_wave(minX, maxX, minY, maxY, maxZ, {p.depth, p.hiz, p.tileMin, p.bX, p.pyrX}, threadIdx.x);
  if (threadIdx.x == 0) {
    p.words.out[1] = v ? 1u : 0u;
    p.words.out[0] = *p.words.err;
  }
}

// Min of hiZ over each 8x8-block tile, one wave per tile.
__global__ void rz_tile_min_kernel(const uint16_t* __restrict__ hiz, uint32_t bX, uint32_t bY,
                                   uint16_t* __restrict__ tileMin, uint32_t pyrX, uint32_t pyrY) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t t = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  if (t >= pyrX * pyrY) return;
  const uint32_t bx = (t % pyrX) * 8 + (lane & 7u), by = (t / pyrX) * 8 + (lane >> 3);
  const uint32_t v = (bx < bX && by < bY) ? uint32_t(hiz[by * bX + bx]) : 0xFFFFu;
  const uint32_t mn = __ockl_wfred_min_u32(v);
  if (lane == 0) tileMin[t] = uint16_t(mn);
}

// readBackDepth (Rasterizer.cpp:351-399), one pixel per thread.
__global__ void __launch_bounds__(256) rz_readback_kernel(const uint16_t* __restrict__ depth,
                                                          const uint16_t* __restrict__ hiz, uint32_t width,
                                                          uint32_t height, uint32_t bX, uint32_t* __restrict__ rgba,
                                                          HostWords words) {
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) words.out[0] = *words.err;
  const uint32_t px = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t py = blockIdx.y;
  if (px >= width || py >= height) return;
  const uint32_t b = (py >> 3) * bX + (px >> 3);
  uint32_t out = 0;
  if (hiz[b] != 1u) {
    const uint32_t v = depth[size_t(b) * 64 + (py & 7u) * 8 + (px & 7u)];
    const float f = bitsf(v << 12) * 3.9623753e+28f;
    const float l = 0.5f / (1000.25f - (1.0f - f) * 999.75f);
    const uint32_t d = uint32_t(25600.0f * l);
    out = (d / 100u & 0xFFu) | ((d % 256u) << 8) | 0xFF000000u;
  }
  rgba[size_t(py) * width + px] = out;
}

// clear (Rasterizer.cpp:107-121) of a single view: hiZ and the per-tile min
// hiZ := 1 (the cleared mark), both arrays in one launch; hiZ (whole groups
// of eight entries, in its own allocation) eight entries per 16-byte store.
__global__ void rz_clear_kernel(uint4* hiz, uint32_t nHiz8, uint16_t* tileMin, uint32_t nMin) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nHiz8) hiz[i] = make_uint4(0x10001u, 0x10001u, 0x10001u, 0x10001u);
  else if (i - nHiz8 < nMin) tileMin[i - nHiz8] = 1;
}

// ---------------------------------------------------------------------------
// Draw-order labels and batch features.
// ---------------------------------------------------------------------------
// Item whose quad range holds quad g (items are in quad order).
// 16 features per batch, from its quads' setup records and packets and the
// labels of the previous step:
//  0 drawn quads / 8          1 log2(1 + union block-box area)
//  2 min packed maxZ / 65535  3 max packed maxZ / 65535   4 mean packed maxZ / 65535
//  5 log2(1 + sum of block-box areas)  6 drawn with rasterize<true>
//  7, 8 union box centre / buffer size (x, y)   9 log2(1 + |W| of the batch centroid)
// 10 log2(1 + previous step's label)  11-13 mean, min, max of (unit quad normal . view direction)
// 14 position of the batch in the view's plain order   15 fraction of Convex quads
// Writes batch b's features; returns whether its occluder is drawn.
__device__ bool batch_features(const LearnParams& p, uint32_t b) {
  const uint32_t item = item_of_quad(p.items, p.nItems, b * 8u, p.groupItem);
  const ItemDesc& D = p.items[item];
  const ItemState& S = p.state[item];
  const ViewDesc& V = p.views[D.view];
  float f[kFeatures];
#pragma unroll
  for (int k = 0; k < kFeatures; ++k) f[k] = 0.0f;
  uint32_t n = 0, convex = 0;
  uint32_t c0 = 0xFFFFu, c1 = 0, r0 = 0xFFFFu, r1 = 0;
  float zmin = 1.0f, zmax = 0.0f, zsum = 0.0f, areaSum = 0.0f;
  const float vlen = sqrtf(V.mvp.raw[12] * V.mvp.raw[12] + V.mvp.raw[13] * V.mvp.raw[13] + V.mvp.raw[14] * V.mvp.raw[14]);
  const float vd[3] = {V.mvp.raw[12] / vlen, V.mvp.raw[13] / vlen, V.mvp.raw[14] / vlen};
  float ndSum = 0.0f, ndMin = 1.0f, ndMax = -1.0f, cen[3] = {0.0f, 0.0f, 0.0f};
  float ext[3];
#pragma unroll
  for (int j = 0; j < 3; ++j) ext[j] = D.refMax[j] - D.refMin[j];
  // The batch's 4 packets of 8 quads: 32 contiguous words (word 8j + k is
  // vertex j of quad k), read as 16-byte loads.
  uint32_t W[32];
  {
    const uint4* src = reinterpret_cast<const uint4*>(D.packets + size_t(b * 8u - D.quadBase) * 4u);
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const uint4 x = src[v];
      W[4 * v] = x.x;
      W[4 * v + 1] = x.y;
      W[4 * v + 2] = x.z;
      W[4 * v + 3] = x.w;
    }
  }
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k) {
    const uint32_t g = b * 8u + k;
    float P[4][3];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t w = W[8 * j + k];
      const float X = float((int32_t(w) >> 21) + 1024), Y = float((w >> 10) & 2047u), Z = float(w & 1023u);
      P[j][0] = D.refMin[0] + X * (ext[0] / 2047.0f);
      P[j][1] = D.refMin[1] + Y * (ext[1] / 2047.0f);
      P[j][2] = D.refMin[2] + Z * (ext[2] / 1023.0f);
#pragma unroll
      for (int a = 0; a < 3; ++a) cen[a] += P[j][a] * (1.0f / 32.0f);
    }
    if (S.status == kStatusSkip) continue;  // not drawn: no valid quads (records not written)
    const uint32_t fz = p.featZ[g];
    if (!(fz & kFeatValid)) continue;  // empty rectangle
    ++n;
    const uint64_t bb = p.bbox[g];
    const uint32_t bc0 = uint32_t(bb & 0xFFFF), bc1 = uint32_t((bb >> 16) & 0xFFFF);
    const uint32_t br0 = uint32_t((bb >> 32) & 0xFFFF), br1 = uint32_t(bb >> 48);
    c0 = min(c0, bc0);
    c1 = max(c1, bc1);
    r0 = min(r0, br0);
    r1 = max(r1, br1);
    areaSum += float((bc1 - bc0 + 1) * (br1 - br0 + 1));
    const float z = float(fz >> 16) * (1.0f / 65535.0f);
    zmin = fminf(zmin, z);
    zmax = fmaxf(zmax, z);
    zsum += z;
    convex += (fz & 0xFFu) == kModeConvex ? 1u : 0u;
    float e1[3], e2[3], e3[3], nrm[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      e1[a] = P[1][a] - P[0][a];
      e2[a] = P[2][a] - P[0][a];
      e3[a] = P[3][a] - P[0][a];
    }
    nrm[0] = (e1[1] * e2[2] - e1[2] * e2[1]) + (e2[1] * e3[2] - e2[2] * e3[1]);
    nrm[1] = (e1[2] * e2[0] - e1[0] * e2[2]) + (e2[2] * e3[0] - e2[0] * e3[2]);
    nrm[2] = (e1[0] * e2[1] - e1[1] * e2[0]) + (e2[0] * e3[1] - e2[1] * e3[0]);
    const float nl = sqrtf(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
    const float nd = nl > 0.0f ? (nrm[0] * vd[0] + nrm[1] * vd[1] + nrm[2] * vd[2]) / nl : 0.0f;
    ndSum += nd;
    ndMin = fminf(ndMin, nd);
    ndMax = fmaxf(ndMax, nd);
  }
  f[0] = float(n) * 0.125f;
  if (n > 0) {
    f[1] = log2f(1.0f + float((c1 - c0 + 1) * (r1 - r0 + 1)));
    f[2] = zmin;
    f[3] = zmax;
    f[4] = zsum / float(n);
    f[5] = log2f(1.0f + areaSum);
    f[7] = (0.5f * float(c0 + c1) + 0.5f) / float(V.bX);
    f[8] = (0.5f * float(r0 + r1) + 0.5f) / float(V.bY);
    f[11] = ndSum / float(n);
    f[12] = ndMin;
    f[13] = ndMax;
    f[15] = float(convex) / float(n);
  } else {
    f[7] = f[8] = 0.5f;
  }
  f[6] = S.status == kStatusClip ? 1.0f : 0.0f;
  const float w = cen[0] * V.mvp.raw[12] + cen[1] * V.mvp.raw[13] + cen[2] * V.mvp.raw[14] + V.mvp.raw[15];
  f[9] = log2f(1.0f + fabsf(w));
  f[10] = log2f(1.0f + float(p.labels[b]));
  f[14] = V.nBatches > 1 ? float(b - V.batchBase) / float(V.nBatches - 1) : 0.0f;
#pragma unroll
  for (int k = 0; k < kFeatures; ++k) p.features[size_t(b) * kFeatures + k] = f[k];
  return S.status != kStatusSkip;
}

__global__ void __launch_bounds__(256) rz_features_kernel(LearnParams p, uint32_t nBatches) {
  __shared__ uint32_t wgCount, wgBase;
  const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
  const bool drawn = b < nBatches && batch_features(p, b);
  if (!p.drawn) return;
  // Append the work-group's drawn batches to the list with one atomic on the
  // list's count (the count is a single word: one atomic per wave serialised
  // there).
  if (threadIdx.x == 0) wgCount = 0;
  __syncthreads();
  const uint64_t m = __ballot(drawn);
  uint32_t waveOff = 0;
  if ((threadIdx.x & 63u) == 0 && m != 0ull) waveOff = atomicAdd(&wgCount, uint32_t(__popcll(m)));
  waveOff = uint32_t(__builtin_amdgcn_readlane(int(waveOff), 0));
  __syncthreads();
  if (threadIdx.x == 0) wgBase = wgCount != 0 ? atomicAdd(p.nDrawn, wgCount) : 0u;
  __syncthreads();
  const uint32_t pre = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
  if (drawn) p.drawn[wgBase + waveOff + pre] = b;
}

// Item k of a reordered draw: batch order[k] alone, with its occluder's
// classification and the footprint of the batch's drawn quads.
__global__ void __launch_bounds__(256) rz_batch_items_kernel(LearnParams p, const uint32_t* __restrict__ order,
                                                              uint32_t nBatches, ItemDesc* __restrict__ outItems,
                                                              ItemState* __restrict__ outState) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= nBatches) return;
  const uint32_t b = order[k];
  const uint32_t item = item_of_quad(p.items, p.nItems, b * 8u, p.groupItem);
  ItemDesc D = p.items[item];
  ItemState S = p.state[item];
  D.quadBase = b * 8u;
  D.quadCount = 8u;
  uint32_t c0 = 0xFFFFFFFFu, c1 = 0, r0 = 0xFFFFFFFFu, r1 = 0;
  for (uint32_t j = 0; j < 8 && S.status != kStatusSkip; ++j) {  // no boxes are written for skipped occluders
    const uint64_t bb = p.bbox[b * 8u + j];
    const uint32_t bc0 = uint32_t(bb & 0xFFFF), bc1 = uint32_t((bb >> 16) & 0xFFFF);
    if (bc0 > bc1) continue;  // empty box: quad not drawn
    c0 = min(c0, bc0);
    c1 = max(c1, bc1);
    r0 = min(r0, uint32_t((bb >> 32) & 0xFFFF));
    r1 = max(r1, uint32_t(bb >> 48));
  }
  S.fp[0] = c0;
  S.fp[1] = c1;
  S.fp[2] = r0;
  S.fp[3] = r1;
  outItems[k] = D;
  outState[k] = S;
}

__global__ void __launch_bounds__(256) rz_item_scores_kernel(LearnParams p, const float* __restrict__ batchScores,
                                                              float* __restrict__ itemScores) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= p.nItems) return;
  const ItemDesc& D = p.items[i];
  float best = -3.402823466e+38f;
  for (uint32_t b = D.quadBase / 8u; b < (D.quadBase + D.quadCount) / 8u; ++b) best = fmaxf(best, batchScores[b]);
  itemScores[i] = best;
}

__global__ void __launch_bounds__(256) rz_sort_keys_kernel(const ViewDesc* __restrict__ views, uint32_t nViews,
                                                           const float* __restrict__ scores, uint32_t n, bool items,
                                                           uint64_t* __restrict__ keys) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint32_t lo = 0, hi = nViews - 1;
  while (lo < hi) {
    const uint32_t mid = (lo + hi + 1) >> 1;
    if ((items ? views[mid].itemBase : views[mid].batchBase) <= i) lo = mid;
    else hi = mid - 1;
  }
  const uint32_t u = __float_as_uint(scores[i]);
  const uint32_t ordered = (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // ascending with the float order
  keys[i] = (uint64_t(lo) << 32) | uint64_t(~ordered);
}

// Squared distance of Main.cpp:184-190: _mm_dp_ps(d, d, 0x7f) sums the x
// and y products, then adds z's (each rounded; compiled without
// contraction, so no fused multiply-add).
__global__ void __launch_bounds__(256) rz_f2b_keys_kernel(const ItemDesc* __restrict__ items, uint32_t n,
                                                          const float* __restrict__ eyes, uint64_t* __restrict__ keys) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const ItemDesc& D = items[i];
  const float* e = eyes + 4 * D.view;
  uint32_t bits = 0;
  if (e[3] != 0.0f) {
    float p[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float c = (D.boundsMax[a] + D.boundsMin[a]) * 0.5f;
      const float d = c - e[a];
      p[a] = d * d;
    }
    bits = __float_as_uint((p[0] + p[1]) + p[2]);  // >= +0 (or NaN, last): its bits order as the value
  }
  keys[i] = (uint64_t(D.view) << 32) | uint64_t(bits);
}

__global__ void __launch_bounds__(256) rz_item_reorder_kernel(LearnParams p, const uint32_t* __restrict__ order,
                                                               ItemDesc* __restrict__ outItems,
                                                               ItemState* __restrict__ outState) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= p.nItems) return;
  const uint32_t i = order[k];
  outItems[k] = p.items[i];
  outState[k] = p.state[i];
}

__global__ void rz_fill_u32_kernel(uint32_t* p, uint32_t n, uint32_t v) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------
static inline uint32_t groups(uint32_t n, uint32_t per) { return (n + per - 1) / per; }

hipError_t launch_prep(const PrepParams& p, hipStream_t stream) {
  if (p.nItems == 0) return hipSuccess;
  // One wave per work-group: a frame's few hundred items then spread over as
  // many CUs, each with its own reads in flight (from host memory, for
  // single-view draws).
  hipLaunchKernelGGL(rz_prep_kernel, dim3(groups(p.nItems, 64)), dim3(64), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_setup(const SetupParams& p, hipStream_t stream) {
  if (p.nQuads == 0 || p.nItems == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_setup_kernel, dim3(groups(p.nQuads, 256)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

template <int T, int NW>
static const void* frame_fn(bool stats, bool boxed) {
  if (stats)
    return boxed ? reinterpret_cast<const void*>(&rz_frame_kernel<T, T, NW, true, true>)
                 : reinterpret_cast<const void*>(&rz_frame_kernel<T, T, NW, true, false>);
  return boxed ? reinterpret_cast<const void*>(&rz_frame_kernel<T, T, NW, false, true>)
               : reinterpret_cast<const void*>(&rz_frame_kernel<T, T, NW, false, false>);
}

static const void* frame_kernel_fn(int tileW, int waves, bool stats, bool boxed) {
  if (tileW == 8)
    return waves == 8 ? frame_fn<8, 8>(stats, boxed)
           : waves == 4 ? frame_fn<8, 4>(stats, boxed)
           : waves == 2 ? frame_fn<8, 2>(stats, boxed)
                        : nullptr;
  if (tileW == 16)
    return waves == 8 ? frame_fn<16, 8>(stats, boxed)
           : waves == 4 ? frame_fn<16, 4>(stats, boxed)
           : waves == 2 ? frame_fn<16, 2>(stats, boxed)
                        : nullptr;
  return nullptr;
}

// Launches a grid that the host has sized to be co-resident, cooperatively
// when asked.  The runtime can refuse a cooperative launch while another
// process on the device holds its cooperative (global wave sync) resources;
// the grid is then dispatched plainly, which the kernels allow: they never
// synchronise the whole grid, and each of their cross-tile waits is bounded
// in time (a grid that another process kept from being co-resident reports
// RZ_ERR_TIMEOUT instead of hanging).
static hipError_t launch_coresident(const void* fn, dim3 grid, dim3 block, void** args, hipStream_t stream,
                                    bool cooperative) {
  if (cooperative) {
    const hipError_t e = hipLaunchCooperativeKernel(fn, grid, block, args, 0, stream);
    if (e != hipErrorIllegalState && e != hipErrorCooperativeLaunchTooLarge) return e;
    (void)hipGetLastError();  // the refusal is handled: clear it
  }
  return hipLaunchKernel(fn, grid, block, args, 0, stream);
}

hipError_t launch_frame(const FrameParams& p, int tileW, hipStream_t stream, bool cooperative, int waves) {
  if (p.nItems == 0) return hipSuccess;
  FrameParams local = p;
  void* args[] = {&local};
  const dim3 grid(p.tilesX * p.tilesY), block(64 * waves);
  const void* fn = frame_kernel_fn(tileW, waves, p.stats != nullptr, p.itemBox != nullptr);
  if (!fn) return hipErrorInvalidValue;
  return launch_coresident(fn, grid, block, args, stream, cooperative);
}

hipError_t frame_max_groups(int tileW, int waves, int* maxGroups) {
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  int perCU = 1 << 30;
  for (int variant = 0; variant < 4; ++variant) {
    const void* fn = frame_kernel_fn(tileW, waves, variant & 1, variant & 2);
    if (!fn) return hipErrorInvalidValue;
    int n = 0;
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, 64 * waves, 0);
    if (e != hipSuccess) return e;
    perCU = n < perCU ? n : perCU;
  }
  *maxGroups = perCU * cus;
  return hipSuccess;
}

hipError_t launch_item_boxes(const ItemState* state, uint32_t n, uint64_t* out, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_item_boxes_kernel, dim3(groups(n, 256)), dim3(256), 0, stream, state, n, out);
  return hipGetLastError();
}

hipError_t launch_status(const ItemState* state, const uint32_t* visible, uint32_t n, uint8_t* out,
                         hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_status_kernel, dim3(groups(n, 256)), dim3(256), 0, stream, state, visible, n, out);
  return hipGetLastError();
}

hipError_t launch_query(const QueryParams& p, hipStream_t stream) {
  if (p.n == 0) return hipSuccess;
  // Small batches leave wave slots (8,192) idle: a wave a box or four, each with
  // the whole wave, is the shortest chain.  Larger ones get as many boxes per
  // wave as fill the slots once, eight rectangles at a time: fewer leave most
  // lanes of the projection idle, more leave slots idle and make longer waves.
  // Device batches of city boxes over the 1080p buffer, us per call back to back:
  //   boxes      1 whole  4 whole  8 boxes  16    32    64
  //   1,000      5.7      7.4      9.3      9.9   9.2   10.4
  //   8,192      7.7      6.8      9.5      9.6   10.6  11.8
  //   32,768     15.4     10.0     14.9     14.7  15.1  15.6
  //   65,536     25.7     14.4     14.8     15.0  15.1  15.9
  //   131,072    45.9     23.9     18.2     14.9  14.9  15.7
  //   262,144    87.1     41.8     30.3     19.8  14.9  15.3
  //   1,000,003  332      155      106      60.8  36.3  24.3
  constexpr uint32_t kWaves = 8192;
  auto go = [&](auto kernel, uint32_t bpw) {
    hipLaunchKernelGGL(kernel, dim3(groups(groups(p.n, bpw), 4)), dim3(256), 0, stream, p);
  };
  if (p.n <= kWaves / 2) go(rz_query_kernel<1, true>, 1);
  else if (p.n <= 8 * kWaves) go(rz_query_kernel<4, true>, 4);
  else if (p.n <= 16 * kWaves) go(rz_query_kernel<16, false>, 16);
  else if (p.n <= 32 * kWaves) go(rz_query_kernel<32, false>, 32);
  else go(rz_query_kernel<64, false>, 64);
  return hipGetLastError();
}

hipError_t launch_query_one(const QueryParams& p, const QueryBox& box, hipStream_t stream) {
  hipLaunchKernelGGL(rz_query_one_kernel, dim3(1), dim3(64), 0, stream, p, box);
  return hipGetLastError();
}

hipError_t launch_query2d(uint32_t minX, uint32_t maxX, uint32_t minY, uint32_t maxY, uint32_t maxZ,
                          const QueryParams& p, hipStream_t stream) {
  hipLaunchKernelGGL(rz_query2d_kernel, dim3(1), dim3(64), 0, stream, minX, maxX, minY, maxY, maxZ, p);
  return hipGetLastError();
}

hipError_t launch_host_words(const HostWords& words, hipStream_t stream) {
  hipLaunchKernelGGL(rz_host_words_kernel, dim3(1), dim3(1), 0, stream, words);
  return hipGetLastError();
}

hipError_t launch_tile_min(const uint16_t* hiz, uint32_t bX, uint32_t bY, uint16_t* tileMin, uint32_t pyrX,
                           uint32_t pyrY, hipStream_t stream) {
  hipLaunchKernelGGL(rz_tile_min_kernel, dim3(groups(pyrX * pyrY, 4)), dim3(256), 0, stream, hiz, bX, bY, tileMin,
                     pyrX, pyrY);
  return hipGetLastError();
}

hipError_t launch_readback(const uint16_t* depth, const uint16_t* hiz, uint32_t width, uint32_t height, uint32_t bX,
                           uint32_t* rgba, const HostWords& words, hipStream_t stream) {
  hipLaunchKernelGGL(rz_readback_kernel, dim3(groups(width, 256), height), dim3(256), 0, stream, depth, hiz, width,
                     height, bX, rgba, words);
  return hipGetLastError();
}

hipError_t launch_clear(uint16_t* hiz, uint32_t nHiz, uint16_t* tileMin, uint32_t nMin, hipStream_t stream) {
  if (nHiz % 8 != 0 || reinterpret_cast<uintptr_t>(hiz) % 16 != 0) return hipErrorInvalidValue;
  const uint32_t n = nHiz / 8 + nMin;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_clear_kernel, dim3(groups(n, 256)), dim3(256), 0, stream, reinterpret_cast<uint4*>(hiz),
                     nHiz / 8, tileMin, nMin);
  return hipGetLastError();
}

// Labelled draws need 8x8-block tiles (the block-major draw); 16x16-block
// tiles have no labelled variant.
template <int NW>
static const void* views_fn(int tileB, bool stats, bool labels) {
  if (tileB == 16)
    return stats ? reinterpret_cast<const void*>(&rz_views_kernel<16, 16, NW, true, false>)
                 : reinterpret_cast<const void*>(&rz_views_kernel<16, 16, NW, false, false>);
  if (labels)
    return stats ? reinterpret_cast<const void*>(&rz_views_kernel<8, 8, NW, true, true>)
                 : reinterpret_cast<const void*>(&rz_views_kernel<8, 8, NW, false, true>);
  return stats ? reinterpret_cast<const void*>(&rz_views_kernel<8, 8, NW, true, false>)
               : reinterpret_cast<const void*>(&rz_views_kernel<8, 8, NW, false, false>);
}

hipError_t launch_views(const ViewsParams& p, uint32_t nGroups, hipStream_t stream, bool cooperative) {
  if (p.nUnits == 0 || nGroups == 0) return hipSuccess;
  const bool st = p.stats != nullptr, lab = p.labels != nullptr;
  if (p.tileB != 8 && (p.tileB != 16 || lab)) return hipErrorInvalidValue;
  const int tb = int(p.tileB);
  if (p.waves != 2 && p.waves != 4 && p.waves != 8) return hipErrorInvalidValue;
  const void* fn = p.waves == 8 ? views_fn<8>(tb, st, lab) : p.waves == 4 ? views_fn<4>(tb, st, lab)
                                                                          : views_fn<2>(tb, st, lab);
  ViewsParams local = p;
  void* args[] = {&local};
  const dim3 grid(nGroups), block(64 * p.waves);
  return launch_coresident(fn, grid, block, args, stream, cooperative);
}

hipError_t views_max_groups(int tileB, int waves, int* maxGroups) {
  int dev = 0, cus = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e != hipSuccess) return e;
  int perCU = 1 << 30;
  for (int variant = 0; variant < (tileB == 16 ? 2 : 4); ++variant) {
    int n = 0;
    const bool stats = variant & 1, labels = variant & 2;
    if (waves != 2 && waves != 4 && waves != 8) return hipErrorInvalidValue;
    const void* fn = waves == 8 ? views_fn<8>(tileB, stats, labels)
                     : waves == 4 ? views_fn<4>(tileB, stats, labels)
                                  : views_fn<2>(tileB, stats, labels);
    e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, 64 * waves, 0);
    if (e != hipSuccess) return e;
    perCU = n < perCU ? n : perCU;
  }
  *maxGroups = perCU * cus;
  return hipSuccess;
}

hipError_t launch_views_query(const ViewsQueryParams& p, hipStream_t stream) {
  if (p.nViews == 0 || (p.nQueries == 0 && !p.errOut)) return hipSuccess;
  hipLaunchKernelGGL(rz_views_query_kernel, dim3(std::max(groups(p.maxPerView, 256), 1u), p.nViews), dim3(256), 0,
                     stream, p);
  return hipGetLastError();
}

hipError_t launch_features(const LearnParams& p, uint32_t nBatches, hipStream_t stream) {
  if (nBatches == 0 || p.nItems == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_features_kernel, dim3(groups(nBatches, 256)), dim3(256), 0, stream, p, nBatches);
  return hipGetLastError();
}

hipError_t launch_batch_items(const LearnParams& p, const uint32_t* order, uint32_t nBatches, ItemDesc* outItems,
                              ItemState* outState, hipStream_t stream) {
  if (nBatches == 0 || p.nItems == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_batch_items_kernel, dim3(groups(nBatches, 256)), dim3(256), 0, stream, p, order, nBatches,
                     outItems, outState);
  return hipGetLastError();
}

hipError_t launch_item_scores(const LearnParams& p, const float* batchScores, float* itemScores,
                              hipStream_t stream) {
  if (p.nItems == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_item_scores_kernel, dim3(groups(p.nItems, 256)), dim3(256), 0, stream, p, batchScores,
                     itemScores);
  return hipGetLastError();
}

hipError_t launch_sort_keys(const ViewDesc* views, uint32_t nViews, const float* scores, uint32_t n, bool items,
                            uint64_t* keys, hipStream_t stream) {
  if (n == 0 || nViews == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_sort_keys_kernel, dim3(groups(n, 256)), dim3(256), 0, stream, views, nViews, scores, n, items,
                     keys);
  return hipGetLastError();
}

hipError_t launch_f2b_keys(const ItemDesc* items, uint32_t n, const float* eyes, uint64_t* keys, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_f2b_keys_kernel, dim3(groups(n, 256)), dim3(256), 0, stream, items, n, eyes, keys);
  return hipGetLastError();
}

hipError_t launch_item_reorder(const LearnParams& p, const uint32_t* order, ItemDesc* outItems, ItemState* outState,
                               hipStream_t stream) {
  if (p.nItems == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_item_reorder_kernel, dim3(groups(p.nItems, 256)), dim3(256), 0, stream, p, order, outItems,
                     outState);
  return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_fill_u32_kernel, dim3(groups(n, 256)), dim3(256), 0, stream, p, n, v);
  return hipGetLastError();
}

hipError_t launch_views_clear(const ViewDesc* src, ViewDesc* views, uint32_t nViews, uint32_t maxEntries,
                              hipStream_t stream) {
  if (nViews == 0) return hipSuccess;
  hipLaunchKernelGGL(rz_views_clear_kernel, dim3(groups(std::max(maxEntries, 1u), 256), nViews), dim3(256), 0, stream,
                     src, views);
  return hipGetLastError();
}

}  // namespace rzd
