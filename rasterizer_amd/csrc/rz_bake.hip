// Occluder::bake (Occluder.cpp:7-181) on the device, for occluders baked at
// run time: per-quad normals, the reference's k-means over six axis seeds,
// the stable regroup by cluster, the 11/11/10-bit packing against the
// reference box, and the bounds.  One wave per occluder.  Bit-exact with the
// host bake: SSE arithmetic is IEEE single precision (compiled without
// contraction), RSQRTPS comes from the host's table, and every sum that the
// reference makes in order is made in the same order.
#include <hip/hip_runtime.h>

#include "rz_kernels.h"
#include "rz_x86.h"

namespace rzd {

namespace {

// First occurrence of the smallest (largest) value in vertex order, as the
// reference's sequential _mm_min_ps(v, acc) (_mm_max_ps) keeps it: a value
// replaces the accumulator only when strictly smaller; NaNs never do.
struct Ext {
  float v;
  uint32_t i;
};
__device__ __forceinline__ Ext pick_min(Ext a, Ext b) { return (b.v < a.v || (b.v == a.v && b.i < a.i)) ? b : a; }
__device__ __forceinline__ Ext pick_max(Ext a, Ext b) { return (b.v > a.v || (b.v == a.v && b.i < a.i)) ? b : a; }
template <bool MIN>
__device__ __forceinline__ float wave_extreme(Ext e) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    Ext o{__shfl_xor(e.v, off), uint32_t(__shfl_xor(int(e.i), off))};
    e = MIN ? pick_min(e, o) : pick_max(e, o);
  }
  return e.v;
}

}  // namespace

namespace {

// One occluder by one wave.  N, order and C are per quad, in LDS (with the
// normals in cluster order in M) or, for an occluder too large for that, in
// the caller's scratch memory (M null).
__device__ __forceinline__ void bake_occluder(const BakeParams& p, uint32_t o, float4* N, float4* M, uint32_t* ord,
                                              uint32_t* C) {
  const uint32_t lane = threadIdx.x;
  const uint32_t v0 = p.offsets[o], n = p.offsets[o + 1] - v0, quads = n / 4;
  const float4* V = reinterpret_cast<const float4*>(p.vertices) + v0;

  // Quad normals: the two triangle normals summed, then normalized
  // (Occluder.cpp:11-21).  The bounds over the input vertices (:159-178) are
  // taken on the way.
  Ext mn[3], mx[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    mn[a] = {__builtin_inff(), 0xFFFFFFFFu};
    mx[a] = {-__builtin_inff(), 0xFFFFFFFFu};
  }
  for (uint32_t q = lane; q < quads; q += 64) {
    const float4 P[4] = {V[4 * q], V[4 * q + 1], V[4 * q + 2], V[4 * q + 3]};
    const V3 a = cross3(sub3(P[1], P[0]), sub3(P[2], P[0])), b = cross3(sub3(P[2], P[0]), sub3(P[3], P[0]));
    const V3 s = approx_normalize({a.x + b.x, a.y + b.y, a.z + b.z}, p.rsqrt);
    N[q] = make_float4(s.x, s.y, s.z, 0.0f);
    C[q] = 0u;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const float c[3] = {P[k].x, P[k].y, P[k].z};
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        if (c[j] < mn[j].v) mn[j] = {c[j], 4 * q + k};
        if (c[j] > mx[j].v) mx[j] = {c[j], 4 * q + k};
      }
    }
  }
  __syncthreads();

  // K-means over six axis seeds, at most 10 rounds (Occluder.cpp:23-78):
  // each quad takes the last seed with the largest dot product; each seed
  // becomes the normalized sum of its quads' normals, summed in quad order
  // (lane k sums seed k).  The quads are regrouped by cluster, stably, in
  // every round that changes a cluster: the sums then run over consecutive
  // normals, and the last regrouping is the packing's (:80-93).
  V3 seed[6] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {0, -1, 0}, {0, 0, -1}, {-1, 0, 0}};
  for (int round = 0; round < 10; ++round) {
    bool mine = false;
    uint32_t size[6] = {0, 0, 0, 0, 0, 0};
    for (uint32_t base = 0; base < quads; base += 64) {
      const uint32_t q = base + lane;
      uint32_t pick = 6;
      if (q < quads) {
        const float4 nq = N[q];
        const V3 v{nq.x, nq.y, nq.z};
        float best = -__builtin_inff();
        pick = 0;
#pragma unroll
        for (uint32_t k = 0; k < 6; ++k) {
          const float d = dp3(seed[k], v);
          if (d >= best) {
            best = d;
            pick = k;
          }
        }
        if (C[q] != pick) {
          C[q] = pick;
          mine = true;
        }
      }
#pragma unroll
      for (uint32_t k = 0; k < 6; ++k) size[k] += uint32_t(__popcll(__ballot(pick == k)));
    }
    const bool changed = __ballot(mine) != 0ull;
    if (!changed && round > 0) break;
    uint32_t at[6], begin = 0, end = 0;
#pragma unroll
    for (uint32_t k = 0, sum = 0; k < 6; ++k) {
      at[k] = sum;
      if (lane == k) {
        begin = sum;
        end = sum + size[k];
      }
      sum += size[k];
    }
    __syncthreads();
    for (uint32_t base = 0; base < quads; base += 64) {
      const uint32_t q = base + lane, pick = q < quads ? C[q] : 6u;
      uint32_t pos = 0;
#pragma unroll
      for (uint32_t k = 0; k < 6; ++k) {
        const uint64_t m = __ballot(pick == k);
        if (pick == k)
          pos = at[k] + __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u));
        at[k] += uint32_t(__popcll(m));
      }
      if (q < quads) {
        ord[pos] = q;
        if (M) M[pos] = N[q];
      }
    }
    __syncthreads();
    if (!changed || round == 9) break;  // the seeds are not read again
    V3 sum{0.0f, 0.0f, 0.0f};
    uint32_t i = begin;
    for (; i + 8 <= end; i += 8) {
      float4 x[8];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) x[j] = M ? M[i + j] : N[ord[i + j]];
#pragma unroll
      for (uint32_t j = 0; j < 8; ++j) sum = {sum.x + x[j].x, sum.y + x[j].y, sum.z + x[j].z};
    }
    for (; i < end; ++i) {
      const float4 x = M ? M[i] : N[ord[i]];
      sum = {sum.x + x.x, sum.y + x.y, sum.z + x.z};
    }
    const V3 c = approx_normalize(sum, p.rsqrt);
#pragma unroll
    for (int k = 0; k < 6; ++k) seed[k] = {__shfl(c.x, k), __shfl(c.y, k), __shfl(c.z, k)};
  }

  // Packing (Occluder.cpp:95-157): word (4b + k) * 8 + l is vertex k of
  // regrouped quad 8b + l, quantized to 11/11/10 bits of the reference box.
  const float* ref = p.ref + 8 * o;
  const float lo[3] = {ref[0], ref[1], ref[2]};
  const float inv[3] = {1.0f / (ref[4] - ref[0]), 1.0f / (ref[5] - ref[1]), 1.0f / (ref[6] - ref[2])};
  for (uint32_t w = lane; w < n; w += 64) {
    const uint32_t b = w >> 5, k = (w >> 3) & 3u, l = w & 7u;
    const float4 vx = V[4 * ord[8 * b + l] + k];
    const float tx = (vx.x - lo[0]) * inv[0], ty = (vx.y - lo[1]) * inv[1], tz = (vx.z - lo[2]) * inv[2];
    const uint32_t qx = uint32_t(cvtt_x86(__builtin_fmaf(tx, 2047.0f, 0.5f)) - 1024);
    const uint32_t qy = uint32_t(cvtt_x86(__builtin_fmaf(ty, 2047.0f, 0.5f)));
    const uint32_t qz = uint32_t(cvtt_x86(__builtin_fmaf(tz, 1023.0f, 0.5f)));
    p.packets[v0 + w] = (qx << 21) | (qy << 10) | qz;
  }

  // Bounds, w set to 1, and the centre.
  float bmin[3], bmax[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    bmin[a] = wave_extreme<true>(mn[a]);
    bmax[a] = wave_extreme<false>(mx[a]);
  }
  if (lane == 0) {
    float* out = p.bounds + 12 * o;
    for (int a = 0; a < 3; ++a) {
      out[a] = bmin[a];
      out[4 + a] = bmax[a];
      out[8 + a] = (bmax[a] + bmin[a]) * 0.5f;
    }
    out[3] = out[7] = 1.0f;
    out[11] = (1.0f + 1.0f) * 0.5f;
  }
}

}  // namespace

// What bounds it: the sequential sums of the k-means rounds, up to an
// occluder's quads long (one wave per occluder, a few hundred occluders).
// From LDS, over consecutive normals, 878 city occluders take 60 us; with
// each seed's lane walking every quad's cluster and normal in global memory
// they took 256.  The LDS is what the launch's largest such occluder needs (40
// bytes a quad: the normals, the normals in cluster order, the order and the
// clusters), so that small ones leave room for many waves on a CU: rz_bake_device
// of 12,000 occluders of 8 quads takes 76 us, and 120 with room for 1,024 quads
// each, which was slower than from global memory (104).
__global__ void __launch_bounds__(64) rz_bake_kernel(BakeParams p) {
  extern __shared__ float4 bakeLds[];
  const uint32_t o = blockIdx.x, v0 = p.offsets[o], quads = (p.offsets[o + 1] - v0) / 4, n = p.ldsQuads;
  uint32_t* words = reinterpret_cast<uint32_t*>(bakeLds + 2 * n);
  if (quads <= n)
    bake_occluder(p, o, bakeLds, bakeLds + n, words, words + n);
  else
    bake_occluder(p, o, p.normals + v0 / 4, nullptr, p.order + v0 / 4, p.cluster + v0 / 4);
}

hipError_t launch_bake(const BakeParams& p, uint32_t nOccluders, hipStream_t stream) {
  if (nOccluders == 0) return hipSuccess;
  if (p.ldsQuads > kBakeLdsQuads) return hipErrorInvalidValue;
  hipLaunchKernelGGL(rz_bake_kernel, dim3(nOccluders), dim3(64), size_t(p.ldsQuads) * kBakeLdsBytes, stream, p);
  return hipGetLastError();
}

}  // namespace rzd
