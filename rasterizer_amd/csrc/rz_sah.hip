// SurfaceAreaHeuristic::generateBatches (SurfaceAreaHeuristic.cpp:10-104) on
// the device, for occluder sets built at run time.
//
// The reference recurses depth first; each call sorts its index range stably
// by box centre along x, then y, then z, scores every split position that is
// a multiple of the granularity with prefix and suffix box areas, and sorts
// the range once more along the winning axis.
//
// Nothing is sorted per call here: every order that a call can see is the
// restriction of one of a few orders of the whole set, which are sorted once.
// Write (x, z, y) for the lexicographic order by those centres, ties by input
// index.  A range sorted along a winning axis is in (x, z, y), (y, z, x) or
// (z, y, x), since that last sort is stable over the z sort, which is stable
// over the y sort, which is stable over the x sort; equal centres never
// change places.  Its child calls then see, for the x scoring, (x, z, y) (or
// (x, y, z) when the range was last sorted along y), for the y scoring
// (y, x, z) and for the z scoring (z, y, x).  Only the first call sees the
// input order: (x, index) and (y, x, index).  So the five orders are kept as
// five index arrays, and a split is a stable partition of each.
//
// One level of the recursion is one round over all open ranges ("segments")
// at once, without the host:
//   - the boxes of chunks of gran positions, since every split falls between
//     chunks, in the three scoring orders;
//   - per segment and axis one work-group: prefix and suffix areas over the
//     chunks (min and max are exact, so the order in which boxes are merged
//     does not change them) and the split costs.  The best (cost, axis, index)
//     is a 64-bit minimum, which keeps the reference's first strict minimum in
//     (axis, index) order; the last of the segment's three work-groups splits
//     it;
//   - a flag per element (right of the split or not) from the winning order,
//     one prefix sum of those flags over all five arrays, and the partition.
// Segments stay in the arrays where the depth-first recursion would emit
// them, so the batches are the final segments, left to right.
//
// What bounds it: launches and latency (six short launches a level, 12 levels
// for 286,000 quads), then the random reads of the boxes.  Four device sorts
// and four scans by key per axis and level, as the reference's sorts would
// translate to, took 6.2 ms of kernels for 240,000 box quads; this takes
// 1.4 ms.
#include <hip/hip_runtime.h>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>
#include <rocprim/iterator/counting_iterator.hpp>
#include <rocprim/iterator/transform_iterator.hpp>

#include <algorithm>
#include <cstdint>
#include <memory>
#include <new>
#include <type_traits>

#include "rasterizer_amd.h"
#include "rz_kernels.h"
#include "rz_scratch.h"

extern "C" __device__ uint32_t __ockl_wfred_min_u32(uint32_t);
extern "C" __device__ uint32_t __ockl_wfred_max_u32(uint32_t);

namespace rzd {

namespace {

constexpr uint32_t kMaxSahItems = 1u << 28;
constexpr float kMaxSahCoordinate = 1099511627776.0f;  // 2^40

struct Ext6 {
  float mn[3], mx[3];
};

struct MergeExt {
  __device__ Ext6 operator()(const Ext6& a, const Ext6& b) const {
    Ext6 r;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      r.mn[j] = fminf(a.mn[j], b.mn[j]);
      r.mx[j] = fmaxf(a.mx[j], b.mx[j]);
    }
    return r;
  }
};

__device__ __forceinline__ Ext6 load_ext(const float* __restrict__ boxes, uint32_t e) {
  const float4 lo = reinterpret_cast<const float4*>(boxes)[2 * size_t(e)];
  const float4 hi = reinterpret_cast<const float4*>(boxes)[2 * size_t(e) + 1];
  return {{lo.x, lo.y, lo.z}, {hi.x, hi.y, hi.z}};
}

// Aabb::surfaceArea (VectorMath.h:57-62): DPPS(ext, ext.yzx, 0x7F), summed
// (x + y) + (z + the masked lane's 0).
__device__ __forceinline__ float surface_area(const Ext6& b) {
  const float e0 = b.mx[0] - b.mn[0], e1 = b.mx[1] - b.mn[1], e2 = b.mx[2] - b.mn[2];
  const float p0 = e0 * e1, p1 = e1 * e2, p2 = e2 * e0;
  return (p0 + p1) + (p2 + 0.0f);
}

// Sort key of a centre coordinate: ascending in float order, with -0 and +0
// equal, as the reference's _mm_cmplt_ps comparator sees them.
__device__ __forceinline__ uint32_t centre_key(float c) {
  const uint32_t u = __float_as_uint(c == 0.0f ? 0.0f : c);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__global__ void __launch_bounds__(256) sah_check_kernel(const float* __restrict__ boxes, uint32_t n,
                                                        uint32_t* __restrict__ bad) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const Ext6 b = load_ext(boxes, i);
  bool ok = true;
#pragma unroll
  for (int j = 0; j < 3; ++j)
    ok = ok && fabsf(b.mn[j]) <= kMaxSahCoordinate && fabsf(b.mx[j]) <= kMaxSahCoordinate && b.mn[j] <= b.mx[j];
  if (!ok) *bad = 1u;
}

__global__ void __launch_bounds__(256) sah_iota_kernel(uint32_t* __restrict__ idx, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) idx[i] = i;
}

// The five orders, and the three the winning axis chooses from.
enum Order : int { kXzy = 0, kYzx = 1, kZyx = 2, kXyz = 3, kYxz = 4, kOrders = 5 };

// One array of a sorting round: the elements in the order they come in (null:
// input order) and the axis of the centre to sort by.
struct SortPart {
  const uint32_t* in;
  int axis;
};
struct SortRound {
  SortPart part[3];
};

// Radix keys (part << 32 | centre key) and values of a round's parts, one
// after another: one stable sort then sorts each part by itself.
__global__ void __launch_bounds__(256) sah_round_keys_kernel(SortRound r, const float* __restrict__ boxes, uint32_t n,
                                                             uint64_t* __restrict__ keys,
                                                             uint32_t* __restrict__ values) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, p = blockIdx.y;
  if (i >= n) return;
  const uint32_t e = r.part[p].in ? r.part[p].in[i] : i;
  const int a = r.part[p].axis;
  const float c = boxes[8 * size_t(e) + a] + boxes[8 * size_t(e) + 4 + a];  // Aabb::getCenter
  keys[size_t(p) * n + i] = uint64_t(p) << 32 | centre_key(c);
  values[size_t(p) * n + i] = e;
}

constexpr uint32_t kClosed = ~0u;

// An open segment of a level: its positions and the axis its elements were
// last sorted along (3: the whole set in input order).
struct Segment {
  uint32_t start, len, axis;
};
// Its split: left part's length, winning axis, and its children's numbers in
// the next level (kClosed: a batch).
struct Split {
  uint32_t k, axis, child[2];
};

struct SahLevel {
  const float* boxes;
  uint32_t n, nChunks, gran, target;
  uint32_t* orders;       // kOrders arrays of n
  uint32_t* nextOrders;   // the same after the level's splits
  const uint32_t* rootX;  // (x, index) and (y, x, index), for the first level
  const uint32_t* rootY;
  uint32_t* chunkSeg;     // per chunk: open segment or kClosed
  uint32_t* nextChunkSeg;
  Segment* segs;
  Segment* nextSegs;
  unsigned long long* best;      // per open segment
  unsigned long long* nextBest;
  uint32_t* arrived;             // work-groups of the segment that are done
  uint32_t* nextArrived;
  uint32_t* nOpen;
  uint32_t* nextNOpen;
  Split* splits;
  Ext6* chunkBox;        // per axis and chunk, in the axis's scoring order
  float* rightArea;      // per axis and chunk: area of the boxes from the chunk to the segment's end
  uint8_t* side;         // per element: right of its segment's split
  const uint32_t* lefts; // per order and position: elements left of their split before it
  uint8_t* starts;       // per chunk: a batch starts here
  uint8_t* batchAxis;    // per chunk: the axis its batch was last sorted along
  uint32_t* err;
};

__device__ __forceinline__ const uint32_t* scoring_order(const SahLevel& L, uint32_t axis, uint32_t lastAxis) {
  if (axis == 2u) return L.orders + size_t(kZyx) * L.n;
  if (lastAxis == 3u) return axis == 0u ? L.rootX : L.rootY;
  if (axis == 1u) return L.orders + size_t(kYxz) * L.n;
  return L.orders + size_t(lastAxis == 1u ? kXyz : kXzy) * L.n;
}

// Boxes of each open segment's chunks of gran positions, in the three scoring
// orders (blockIdx.y).  Every segment starts at a multiple of gran (the root
// at 0, each split gran times an integer further on), so no chunk spans two
// segments.
__global__ void __launch_bounds__(256) sah_chunks_kernel(SahLevel L) {
  const uint32_t c = blockIdx.x * blockDim.x + threadIdx.x, axis = blockIdx.y;
  if (c >= L.nChunks) return;
  const uint32_t s = L.chunkSeg[c];
  if (s == kClosed) return;
  const uint32_t* order = scoring_order(L, axis, L.segs[s].axis);
  const uint32_t i0 = c * L.gran, i1 = min(i0 + L.gran, L.n);
  Ext6 b = load_ext(L.boxes, order[i0]);
  const MergeExt merge;
  for (uint32_t i = i0 + 1; i < i1; ++i) b = merge(b, load_ext(L.boxes, order[i]));
  L.chunkBox[size_t(axis) * L.nChunks + c] = b;
}

__device__ __forceinline__ uint64_t wave_min_u64(uint64_t v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const uint32_t lo = uint32_t(__shfl_xor(int(uint32_t(v)), off));
    const uint32_t hi = uint32_t(__shfl_xor(int(uint32_t(v >> 32)), off));
    const uint64_t o = (uint64_t(hi) << 32) | lo;
    v = o < v ? o : v;
  }
  return v;
}

// sahSplit's cost loop (SurfaceAreaHeuristic.cpp:46-64) for one open segment
// and axis, by one work-group: split position k of a segment of len items
// costs area(items [0, k)) * k + area(items [k, len)) * (len - k), for k =
// gran, 2 gran, ... < len - gran.  Each thread takes a run of consecutive
// chunks; the runs' boxes are scanned in both directions in LDS, then each
// thread walks its run backwards for the right areas and forwards for the left
// ones and the costs.  The key orders by cost (non-negative, -0 folded into
// +0), then axis, then k, so the minimum is the reference's first strict
// minimum.  The last of the segment's three work-groups splits it.
//
// NT threads: the first levels' few long segments take 1024, so that a run is
// short; later ones 256, so that many segments share a CU.
template <uint32_t NT>
__global__ void __launch_bounds__(NT) sah_split_kernel(SahLevel L) {
  const uint32_t s = blockIdx.x, axis = blockIdx.y, t = threadIdx.x;
  if (s >= *L.nOpen) return;
  __shared__ Ext6 pre[2][NT], suf[2][NT];
  __shared__ uint64_t waveBest[NT / 64];
  const Segment S = L.segs[s];
  const uint32_t c0 = S.start / L.gran, nc = (S.len + L.gran - 1) / L.gran;
  const uint32_t per = (nc + NT - 1) / NT, r0 = min(t * per, nc), r1 = min(r0 + per, nc);
  const Ext6* box = L.chunkBox + size_t(axis) * L.nChunks + c0;
  float* right = L.rightArea + size_t(axis) * L.nChunks + c0;
  const MergeExt merge;
  const float inf = __builtin_inff();
  const Ext6 empty = {{inf, inf, inf}, {-inf, -inf, -inf}};
  Ext6 run = empty;
  for (uint32_t c = r0; c < r1; ++c) run = merge(run, box[c]);
  pre[0][t] = suf[0][t] = run;
  __syncthreads();
  uint32_t cur = 0;
  for (uint32_t d = 1; d < NT; d <<= 1) {
    pre[cur ^ 1][t] = t >= d ? merge(pre[cur][t - d], pre[cur][t]) : pre[cur][t];
    suf[cur ^ 1][t] = t + d < NT ? merge(suf[cur][t], suf[cur][t + d]) : suf[cur][t];
    cur ^= 1;
    __syncthreads();
  }
  run = t + 1 < NT ? suf[cur][t + 1] : empty;
  for (uint32_t c = r1; c > r0; --c) {
    run = merge(run, box[c - 1]);
    right[c - 1] = surface_area(run);
  }
  run = t > 0 ? pre[cur][t - 1] : empty;
  uint64_t key = ~0ull;
  for (uint32_t c = r0; c < r1; ++c) {
    const uint32_t k = c * L.gran;
    if (k >= L.gran && k + L.gran < S.len) {
      float cost = surface_area(run) * float(int(k)) + right[c] * float(int(S.len - k));
      if (cost == 0.0f) cost = 0.0f;
      const uint64_t mine = (uint64_t(__float_as_uint(cost)) << 32) | (uint64_t(axis) << 30) | k;
      key = mine < key ? mine : key;
    }
    run = merge(run, box[c]);
  }
  key = wave_min_u64(key);
  if ((t & 63u) == 0u) waveBest[t >> 6] = key;
  __syncthreads();
  if (t != 0u) return;
  for (uint32_t w = 1; w < NT / 64; ++w) key = waveBest[w] < key ? waveBest[w] : key;
  atomicMin(&L.best[s], static_cast<unsigned long long>(key));
  if (__hip_atomic_fetch_add(&L.arrived[s], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) != 2u) return;
  // All three axes are in.
  const uint64_t best = __hip_atomic_load(&L.best[s], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  Split P = {uint32_t(best & 0x3FFFFFFFu), uint32_t(best >> 30) & 3u, {kClosed, kClosed}};
  if (best == ~0ull) {
    // Every open segment has a split position: the root holds more than 2 gran
    // items and a child stays open only with target > 2 gran items.
    atomicOr(L.err, 1u);
    P = {S.len, 0u, {kClosed, kClosed}};
  }
  const uint32_t start[2] = {S.start, S.start + P.k}, len[2] = {P.k, S.len - P.k};
  for (int i = 0; i < 2; ++i) {
    // A child recurses when it holds target items or more
    // (SurfaceAreaHeuristic.cpp:81-92).
    if (len[i] >= L.target && best != ~0ull) {
      const uint32_t id = atomicAdd(L.nextNOpen, 1u);
      P.child[i] = id;
      L.nextSegs[id] = {start[i], len[i], P.axis};
      L.nextBest[id] = ~0ull;
      L.nextArrived[id] = 0u;
    }
  }
  if (best != ~0ull) L.starts[start[1] / L.gran] = 1;
  L.splits[s] = P;
}

// Which elements lie right of their segment's split, in the winning order.
__global__ void __launch_bounds__(256) sah_sides_kernel(SahLevel L) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= L.n) return;
  const uint32_t s = L.chunkSeg[p / L.gran];
  if (s == kClosed) return;
  const Split P = L.splits[s];
  L.side[L.orders[size_t(P.axis) * L.n + p]] = p - L.segs[s].start >= P.k;
}

// 1 for an element left of its split, 0 right of it or in a batch: the input
// of the prefix sum over all five arrays.
struct IsLeft {
  const uint32_t* orders;
  const uint32_t* chunkSeg;
  const uint8_t* side;
  uint32_t n, gran;
  __device__ uint32_t operator()(uint32_t i) const {
    const uint32_t a = i / n, p = i - a * n;
    if (chunkSeg[p / gran] == kClosed) return 0u;
    return side[orders[i]] ? 0u : 1u;
  }
};

// The stable partition of every open segment in each order (blockIdx.y), and
// the next level's segment of every chunk.
__global__ void __launch_bounds__(256) sah_partition_kernel(SahLevel L) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x, a = blockIdx.y;
  if (p == 0u && a == 0u) *L.nOpen = 0u;  // this level's count is the one after next's
  if (p >= L.n) return;
  const uint32_t* in = L.orders + size_t(a) * L.n;
  uint32_t* out = L.nextOrders + size_t(a) * L.n;
  const uint32_t c = p / L.gran, s = L.chunkSeg[c], e = in[p];
  const bool first = a == 0u && p == c * L.gran;
  if (s == kClosed) {
    out[p] = e;
    if (first) L.nextChunkSeg[c] = kClosed;
    return;
  }
  const Split P = L.splits[s];
  const uint32_t start = L.segs[s].start, at = p - start;
  const uint32_t* lefts = L.lefts + size_t(a) * L.n;
  const uint32_t l = lefts[p] - lefts[start];
  out[start + (L.side[e] ? P.k + (at - l) : l)] = e;
  if (first) {
    const uint32_t child = P.child[at >= P.k ? 1 : 0];
    L.nextChunkSeg[c] = child;
    if (child == kClosed) L.batchAxis[c] = uint8_t(P.axis);
  }
}

// The batches' elements: each batch in the order it was last sorted in.
__global__ void __launch_bounds__(256) sah_emit_kernel(const uint32_t* __restrict__ orders,
                                                       const uint8_t* __restrict__ batchAxis, uint32_t n,
                                                       uint32_t gran, uint32_t* __restrict__ out) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) out[p] = orders[size_t(batchAxis[p / gran]) * n + p];
}

uint32_t grid_of(uint32_t n) { return (n + 255u) / 256u; }

}  // namespace

#define SAH_HIP(call)                                  \
  do {                                                 \
    if ((call) != hipSuccess) return RZ_ERR_DEVICE;    \
  } while (0)

int sah_batches_run(hipStream_t stream, Scratch& scratch, uint32_t n, const float* d_boxes, uint32_t target,
                    uint32_t gran, uint32_t* d_indices, uint32_t* batchOffsets, uint32_t* nBatches) {
  if (gran == 0 || target <= 2 * uint64_t(gran)) return RZ_ERR_INVALID_ARGUMENT;
  if (n > kMaxSahItems) return RZ_ERR_TOO_LARGE;
  batchOffsets[0] = 0;
  if (n == 0) {
    *nBatches = 0;
    return RZ_OK;
  }
  const bool whole = n <= 2 * gran;  // no split position (see below)
  const uint32_t nChunks = (n + gran - 1) / gran;
  const uint32_t maxOpen = n / target + 1;  // every open segment but the root holds target items or more
  const size_t n3 = size_t(3) * n;
  SahLevel A{}, B{};  // the levels' two views of the buffers
  uint64_t *keys = nullptr, *keysOut = nullptr;
  uint32_t *values = nullptr, *round1 = nullptr, *round2 = nullptr, *lefts = nullptr;
  unsigned char* temp = nullptr;
  size_t sortBytes = 0, scanBytes = 0;
  auto left_iterator = [&](const SahLevel& L) {
    return rocprim::make_transform_iterator(rocprim::counting_iterator<uint32_t>(0u),
                                            IsLeft{L.orders, L.chunkSeg, L.side, n, gran});
  };
  if (!whole) {
    for (uint32_t parts = 2; parts <= 3; ++parts) {
      size_t bytes = 0;
      SAH_HIP(rocprim::radix_sort_pairs(nullptr, bytes, keys, keysOut, values, values, size_t(parts) * n, 0u, 34u,
                                        stream));
      sortBytes = std::max(sortBytes, bytes);
    }
    SAH_HIP(rocprim::exclusive_scan(nullptr, scanBytes, left_iterator(A), lefts, 0u, size_t(kOrders) * n,
                                    rocprim::plus<uint32_t>(), stream));
  }
  const size_t tempBytes = std::max(sortBytes, scanBytes);
  Scratch::Frame frame(scratch);
  bool ok = true;
  auto take = [&](auto** p, size_t count) {
    *p = scratch.take<std::remove_pointer_t<std::remove_pointer_t<decltype(p)>>>(count);
    ok = ok && *p != nullptr;
  };
  take(&A.err, 4);  // the error word, the range check's, and the two open counts
  if (!whole) {
    take(&A.orders, size_t(kOrders) * n);
    take(&A.nextOrders, size_t(kOrders) * n);
    take(&keys, n3);
    take(&keysOut, n3);
    take(&values, n3);
    take(&round1, size_t(2) * n);
    take(&round2, n3);
    take(&lefts, size_t(kOrders) * n);
    take(&temp, tempBytes);
    take(&A.chunkSeg, nChunks);
    take(&A.nextChunkSeg, nChunks);
    take(&A.segs, maxOpen);
    take(&A.nextSegs, maxOpen);
    take(&A.best, maxOpen);
    take(&A.nextBest, maxOpen);
    take(&A.arrived, maxOpen);
    take(&A.nextArrived, maxOpen);
    take(&A.splits, maxOpen);
    take(&A.chunkBox, size_t(3) * nChunks);
    take(&A.rightArea, size_t(3) * nChunks);
    take(&A.side, n);
    take(&A.starts, nChunks);
    take(&A.batchAxis, nChunks);
  }
  if (!ok) return RZ_ERR_OUT_OF_MEMORY;
  A.nOpen = A.err + 2;
  A.nextNOpen = A.err + 3;
  uint32_t words[4] = {0, 0, 1, 0};
  SAH_HIP(hipMemcpyAsync(A.err, words, sizeof words, hipMemcpyHostToDevice, stream));
  sah_check_kernel<<<grid_of(n), 256, 0, stream>>>(d_boxes, n, A.err + 1);
  SAH_HIP(hipGetLastError());
  if (whole) {
    // No split position exists, so the reference's recursion is undefined
    // here (bestIndex stays -1); the whole set is one batch in input order.
    SAH_HIP(hipMemcpyAsync(words, A.err, sizeof words, hipMemcpyDeviceToHost, stream));
    SAH_HIP(hipStreamSynchronize(stream));
    if (words[1]) return RZ_ERR_INVALID_ARGUMENT;
    sah_iota_kernel<<<grid_of(n), 256, 0, stream>>>(d_indices, n);
    SAH_HIP(hipGetLastError());
    SAH_HIP(hipStreamSynchronize(stream));
    batchOffsets[1] = n;
    *nBatches = 1;
    return RZ_OK;
  }

  // The orders, in four rounds of stable sorts, each sorting two or three
  // arrays at once:
  //   (x)        (z)
  //   (y, x)     (y, z)     (x, z)
  //   (z, y, x)  (x, y, z)  (y, x, z)
  //   (x, z, y)  (y, z, x)
  auto sort_round = [&](const SortRound& r, uint32_t parts, uint32_t* out) -> hipError_t {
    sah_round_keys_kernel<<<dim3(grid_of(n), parts), 256, 0, stream>>>(r, d_boxes, n, keys, values);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t bytes = tempBytes;
    return rocprim::radix_sort_pairs(temp, bytes, keys, keysOut, values, out, size_t(parts) * n, 0u, 34u, stream);
  };
  auto order = [&](int o) { return A.orders + size_t(o) * n; };
  // The third round's results are not neighbours in `orders`: it goes through
  // nextOrders, which the levels only write.
  uint32_t* round3 = A.nextOrders;
  SAH_HIP(sort_round({{{nullptr, 0}, {nullptr, 2}, {nullptr, 0}}}, 2, round1));
  SAH_HIP(sort_round({{{round1, 1}, {round1 + n, 1}, {round1 + n, 0}}}, 3, round2));
  SAH_HIP(sort_round({{{round2, 2}, {round2 + n, 0}, {round2 + 2 * size_t(n), 1}}}, 3, round3));
  static_assert(kYzx == kXzy + 1 && kXyz == kZyx + 1 && kYxz == kZyx + 2, "the rounds write neighbouring orders");
  SAH_HIP(sort_round({{{round3, 0}, {round3, 1}, {nullptr, 0}}}, 2, order(kXzy)));
  SAH_HIP(hipMemcpyAsync(order(kZyx), round3, n3 * 4, hipMemcpyDeviceToDevice, stream));

  // The root is split whatever its size (generateBatches calls the recursion
  // on it directly).
  const Segment root = {0u, n, 3u};
  const unsigned long long none = ~0ull;
  SAH_HIP(hipMemcpyAsync(A.segs, &root, sizeof root, hipMemcpyHostToDevice, stream));
  SAH_HIP(hipMemcpyAsync(A.best, &none, sizeof none, hipMemcpyHostToDevice, stream));
  SAH_HIP(hipMemsetAsync(A.arrived, 0, 4, stream));
  SAH_HIP(hipMemsetAsync(A.chunkSeg, 0, size_t(nChunks) * 4, stream));
  SAH_HIP(hipMemsetAsync(A.starts, 0, nChunks, stream));
  SAH_HIP(hipMemsetAsync(A.starts, 1, 1, stream));
  A.boxes = d_boxes;
  A.n = n;
  A.nChunks = nChunks;
  A.gran = gran;
  A.target = target;
  A.rootX = round1;
  A.rootY = round2;
  A.lefts = lefts;
  B = A;
  std::swap(B.orders, B.nextOrders);
  std::swap(B.chunkSeg, B.nextChunkSeg);
  std::swap(B.segs, B.nextSegs);
  std::swap(B.best, B.nextBest);
  std::swap(B.arrived, B.nextArrived);
  std::swap(B.nOpen, B.nextNOpen);
  // Levels until none is open: the host looks after as many as even splits
  // need, then after every second one (a level without open segments only
  // copies the orders).
  uint32_t level = 0, look = 1;
  while ((uint64_t(target) << look) <= n) ++look;
  while (true) {
    const SahLevel& L = level & 1u ? B : A;
    sah_chunks_kernel<<<dim3(grid_of(nChunks), 3), 256, 0, stream>>>(L);
    SAH_HIP(hipGetLastError());
    const uint32_t open = level < 31u ? std::min(maxOpen, 1u << level) : maxOpen;
    if (level < 4u)
      sah_split_kernel<1024><<<dim3(open, 3), 1024, 0, stream>>>(L);
    else
      sah_split_kernel<256><<<dim3(open, 3), 256, 0, stream>>>(L);
    SAH_HIP(hipGetLastError());
    sah_sides_kernel<<<grid_of(n), 256, 0, stream>>>(L);
    SAH_HIP(hipGetLastError());
    size_t bytes = tempBytes;
    SAH_HIP(rocprim::exclusive_scan(temp, bytes, left_iterator(L), lefts, 0u, size_t(kOrders) * n,
                                    rocprim::plus<uint32_t>(), stream));
    sah_partition_kernel<<<dim3(grid_of(n), kOrders), 256, 0, stream>>>(L);
    SAH_HIP(hipGetLastError());
    ++level;
    if (level < look) continue;
    look = level + 2;
    SAH_HIP(hipMemcpyAsync(words, A.err, sizeof words, hipMemcpyDeviceToHost, stream));
    SAH_HIP(hipStreamSynchronize(stream));
    if (words[1]) return RZ_ERR_INVALID_ARGUMENT;
    if (words[0]) return RZ_ERR_DEVICE;
    if (words[2] == 0 && words[3] == 0) break;
  }
  sah_emit_kernel<<<grid_of(n), 256, 0, stream>>>(level & 1u ? B.orders : A.orders, A.batchAxis, n, gran, d_indices);
  SAH_HIP(hipGetLastError());
  const std::unique_ptr<uint8_t[]> starts(new (std::nothrow) uint8_t[nChunks]);
  if (!starts) return RZ_ERR_OUT_OF_MEMORY;
  SAH_HIP(hipMemcpyAsync(starts.get(), A.starts, nChunks, hipMemcpyDeviceToHost, stream));
  SAH_HIP(hipStreamSynchronize(stream));
  uint32_t count = 0;
  for (uint32_t c = 1; c < nChunks; ++c)
    if (starts[c]) batchOffsets[++count] = c * gran;
  batchOffsets[++count] = n;
  *nBatches = count;
  return RZ_OK;
}

// ---------------------------------------------------------------------------
// Scene preparation around the SAH pass (Main.cpp:86-128): padded quad
// boxes, the scene box, and the vertices gathered into batch order.
// ---------------------------------------------------------------------------
namespace {

// Ascending-order key of a float (for exact, order-independent min and max
// with atomics; -0 sorts below +0).
__device__ __forceinline__ uint32_t ordered_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Quad j < nPad: padded quads (j >= nQuads) are four copies of vertex 0, as
// Main.cpp:90-94 pads the index buffer with indices[0].
__device__ __forceinline__ float4 padded_vertex(const float4* __restrict__ v, uint32_t nQuads, uint32_t j, uint32_t k) {
  return j < nQuads ? v[4 * size_t(j) + k] : v[0];
}

// A thread's share of the scene box (Main.cpp:109-113) as ordered keys, and
// whether it met a vertex that the SAH costs cannot take (they need finite
// boxes of bounded size, as rz_sah_batches checks; NaN would also escape the
// fminf/fmaxf boxes).
struct SceneShare {
  uint32_t mn[4] = {~0u, ~0u, ~0u, ~0u}, mx[4] = {0u, 0u, 0u, 0u};
  bool bad = false;
  __device__ void add(float4 v) {
    const float c[4] = {v.x, v.y, v.z, v.w};
    bad = bad || !(fabsf(v.x) <= 0x1p40f) || !(fabsf(v.y) <= 0x1p40f) || !(fabsf(v.z) <= 0x1p40f);
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      mn[l] = min(mn[l], ordered_key(c[l]));
      mx[l] = max(mx[l], ordered_key(c[l]));
    }
  }
};

// The work-group's (256 threads) share as nine words: minima, maxima, bad.
__device__ void reduce_share(const SceneShare& s, uint32_t* __restrict__ out) {
  __shared__ uint32_t part[4][9];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    const uint32_t a = __ockl_wfred_min_u32(s.mn[l]), b = __ockl_wfred_max_u32(s.mx[l]);
    if (lane == 0u) {
      part[wave][l] = a;
      part[wave][4 + l] = b;
    }
  }
  const uint64_t bad = __ballot(s.bad);
  if (lane == 0u) part[wave][8] = bad != 0ull ? 1u : 0u;
  __syncthreads();
  if (threadIdx.x < 9u) {
    uint32_t v = part[0][threadIdx.x];
    for (int w = 1; w < 4; ++w) v = threadIdx.x < 4u ? min(v, part[w][threadIdx.x]) : max(v, part[w][threadIdx.x]);
    out[threadIdx.x] = v;
  }
}

// Main.cpp:96-105: the quads' Aabbs over their four vertices (all lanes), and
// the scene box over those vertices and boxVertices (a whole vertex buffer can
// hold vertices no quad references).  Each work-group writes its share of the
// scene box; one atomic per wave and word on the same eight words took 0.83 ms
// of the city mesh's preparation.
__global__ void __launch_bounds__(256) scene_boxes_kernel(const float4* __restrict__ vertices, uint32_t nQuads,
                                                          uint32_t nPad, const float4* __restrict__ boxVertices,
                                                          uint32_t nBox, float4* __restrict__ boxes,
                                                          uint32_t* __restrict__ partials) {
  const uint32_t first = blockIdx.x * blockDim.x + threadIdx.x, step = gridDim.x * blockDim.x;
  SceneShare s;
  for (uint32_t j = first; j < nPad; j += step) {  // nPad is at most 2^28
    float4 mn = make_float4(INFINITY, INFINITY, INFINITY, INFINITY);
    float4 mx = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const float4 v = padded_vertex(vertices, nQuads, j, k);
      mn = make_float4(fminf(mn.x, v.x), fminf(mn.y, v.y), fminf(mn.z, v.z), fminf(mn.w, v.w));
      mx = make_float4(fmaxf(mx.x, v.x), fmaxf(mx.y, v.y), fmaxf(mx.z, v.z), fmaxf(mx.w, v.w));
      s.add(v);
    }
    boxes[2 * size_t(j)] = mn;
    boxes[2 * size_t(j) + 1] = mx;
  }
  for (size_t j = first; j < nBox; j += step) s.add(boxVertices[j]);  // nBox can be up to 2^32 - 1
  reduce_share(s, partials + 9 * size_t(blockIdx.x));
}

// The scene box from the work-groups' shares.
__global__ void __launch_bounds__(256) scene_keys_kernel(const uint32_t* __restrict__ partials, uint32_t parts,
                                                         uint32_t* __restrict__ sceneKeys) {
  SceneShare s;
  for (uint32_t p = threadIdx.x; p < parts; p += blockDim.x) {
    const uint32_t* w = partials + 9 * size_t(p);
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      s.mn[l] = min(s.mn[l], w[l]);
      s.mx[l] = max(s.mx[l], w[4 + l]);
    }
    s.bad = s.bad || w[8] != 0u;
  }
  reduce_share(s, sceneKeys);
}

__global__ void __launch_bounds__(256) scene_gather_kernel(const float4* __restrict__ vertices, uint32_t nQuads,
                                                           uint32_t nPad, const uint32_t* __restrict__ order,
                                                           float4* __restrict__ out) {
  const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 4 * nPad) return;
  out[t] = padded_vertex(vertices, nQuads, order[t >> 2], t & 3u);
}

}  // namespace

hipError_t launch_scene_boxes(const float* vertices, uint32_t nQuads, uint32_t nPad, const float* boxVertices,
                              uint32_t nBox, float* boxes, uint32_t* partials, uint32_t* sceneKeys,
                              hipStream_t stream) {
  const size_t items = std::max<size_t>(nPad, boxVertices ? nBox : 0u);
  const uint32_t parts = uint32_t(std::min<size_t>((items + 255u) / 256u, kSceneParts));
  scene_boxes_kernel<<<parts, 256, 0, stream>>>(reinterpret_cast<const float4*>(vertices), nQuads, nPad,
                                                reinterpret_cast<const float4*>(boxVertices), boxVertices ? nBox : 0u,
                                                reinterpret_cast<float4*>(boxes), partials);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  scene_keys_kernel<<<1, 256, 0, stream>>>(partials, parts, sceneKeys);
  return hipGetLastError();
}

hipError_t launch_scene_gather(const float* vertices, uint32_t nQuads, uint32_t nPad, const uint32_t* order,
                               float* out, hipStream_t stream) {
  scene_gather_kernel<<<grid_of(4 * nPad), 256, 0, stream>>>(reinterpret_cast<const float4*>(vertices), nQuads, nPad,
                                                             order, reinterpret_cast<float4*>(out));
  return hipGetLastError();
}

}  // namespace rzd
