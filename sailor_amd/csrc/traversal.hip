// Ray / voxel intersection (Amanatides-Woo DDA over the coarse grid), per-ray
// adaptive sampling inside the hit intervals, and the per-ray sort.
//
// Follows c_lib/VoxelEncoding/src/intersection_kernel.cu (ray_voxel_traversal
// :286-439, RayVoxelIntersectionNodeListNew :128-284, RayVoxelIntersection
// :36-71) and c_lib/VoxelEncoding/src/sampling_kernel.cu
// (ray_voxels_sampling_uniform_kernel :1070-1177, sort_samplings :1308-1329).
//
// Differences from the reference (all deliberate):
//  * the slab test uses the IEEE reciprocal 1.0f/d instead of __fdividef;
//  * the child weight and the start-level voxel scale use the tree's `rate`
//    instead of the literal 4 (identical for rate 4);
//  * hit lists are bounded by n_max_hits with an overflow flag instead of
//    writing past the end of the row;
//  * the sort is stable (ties keep slot order) so the permutation is unique.
// Compiled with -ffp-contract=off: intervals, valid lengths and sample counts
// are reproduced bit for bit by the CPU oracle.
#include "common.h"
#include "traversal_common.h"

namespace {

constexpr int kThreads = 256;

using sailor::LaneGroup;
using sailor::SampleRow;

constexpr int kWalkThreads = 64;   // one wave: rays differ widely in length

__global__ void fill_lists(int* __restrict__ idx, float* __restrict__ a, float* __restrict__ b,
                           long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    idx[i] = -1;
    a[i] = -1.0f;
    b[i] = -1.0f;
  }
}

template <int G>
struct ListSink {
  int* idx;
  float* tmin;
  float* tmax;
  int cap;
  bool overflow;
  const LaneGroup<G>& grp;
  __device__ __forceinline__ void store(int pos, int node, float t0, float t1) {
    if (pos < cap) {
      idx[pos] = node;
      tmin[pos] = t0;
      tmax[pos] = t1;
    } else {
      overflow = true;
    }
  }
  __device__ __forceinline__ void put(int pos, int node, float t0, float t1) {
    if (grp.sub == 0) store(pos, node, t0, t1);
  }
  __device__ __forceinline__ void put_lanes(int pos, int node, float t0, float t1, bool hit,
                                            unsigned votes) {
    if (hit) store(pos + grp.before(votes), node, t0, t1);
  }
  __device__ __forceinline__ bool stop() const { return false; }
};

// G lanes per ray (traversal_common.h); each wave then fills what its rows have
// left with -1.  The rows are what bounds the call (n_max 1024: 12 KB a ray), so
// they are written once: a fill of all rows before a lane-per-ray walk took
// 225 + 256 us for 102,400 rays, this kernel 239 us (5.3 TB/s).  A lane per ray
// (G = 1) finds its rows filled.
template <int G>
__global__ void __launch_bounds__(kWalkThreads)
traversal_kernel(const int* __restrict__ vc, const float4* __restrict__ node_pos,
                 const int4* __restrict__ node_info, int n_nodes,
                 const float* __restrict__ vol_bbox,
                 const float* __restrict__ voxel_size, long long first, long long ray_end,
                 int dim_fine, int dim_coarse, int rate, const float* __restrict__ ray_ori,
                 const float* __restrict__ ray_dir, int R, int n_max,
                 int th_early_stop, int is_training, int opt_num,
                 int* __restrict__ hit_idx, float* __restrict__ tmin,
                 float* __restrict__ tmax, float* __restrict__ valid_len,
                 int* __restrict__ status) {
  constexpr int kRays = kWalkThreads / G;
  const LaneGroup<G> grp;
  const long long ray = first + (long long)blockIdx.x * kRays + threadIdx.x / G;
  int count = 0, filled = n_max;
  bool overflow = false;
  if (ray < ray_end) {
    const int b = (int)(ray / R);
    sailor::RayCtx ctx;
    ctx.init(vc, node_pos, node_info, n_nodes, vol_bbox, voxel_size, b, dim_fine,
             dim_coarse, rate, ray_ori + ray * 3, ray_dir + ray * 3);
    ListSink<G> sink{hit_idx + ray * n_max, tmin + ray * n_max, tmax + ray * n_max,
                     n_max, false, grp};
    float vl = 0.0f;
    count = sailor::traverse(ctx, grp, th_early_stop, is_training != 0, opt_num, sink, &vl);
    if (grp.sub == 0) valid_len[ray] = vl;
    overflow = sink.overflow;
    if (G > 1) filled = min(count, n_max);
  }
  const int lane = threadIdx.x & 63;
  const long long ray0 = ray - grp.base / G;
#pragma unroll 1
  for (int k = 0; k < (G > 1 ? 64 / G : 0); ++k) {
    const int from = __builtin_amdgcn_readlane(filled, k * G);
    if (from >= n_max) continue;
    const long long row = (ray0 + k) * n_max;
    sailor::fill_row(reinterpret_cast<unsigned*>(hit_idx + row), from, n_max, 0xffffffffu, lane);
    sailor::fill_row(reinterpret_cast<unsigned*>(tmin + row), from, n_max, 0xbf800000u, lane);
    sailor::fill_row(reinterpret_cast<unsigned*>(tmax + row), from, n_max, 0xbf800000u, lane);
  }
  // global max hit count (reference: atomicMax per step, :405) and overflow
  int m = count;
  for (int o = 32; o > 0; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
  unsigned long long ov = __ballot(overflow);
  if (lane == 0) {
    if (m > 0) atomicMax(status, m);
    if (ov) atomicOr(status + 1, 1);
  }
}

// G lanes per ray, G hits at a time; the row's unused slots are -1.
template <int G>
__global__ void __launch_bounds__(kWalkThreads)
sampling_kernel(const int* __restrict__ hit_idx, const float* __restrict__ tmin,
                const float* __restrict__ tmax, const float* __restrict__ noise,
                const float* __restrict__ valid_len,
                const float4* __restrict__ node_pos,
                const float* __restrict__ voxel_size, long long first, long long ray_end, int R,
                int n_max, int S, int start_scale, int* __restrict__ sidx,
                float* __restrict__ st) {
  constexpr int kRays = kWalkThreads / G;
  const LaneGroup<G> grp;
  const long long ray = first + (long long)blockIdx.x * kRays + threadIdx.x / G;
  int has = S;   // rows past the batch have no tail
  if (ray < ray_end) {
    const int b = (int)(ray / R);
    const int* hi = hit_idx + ray * n_max;
    const float* h0 = tmin + ray * n_max;
    const float* h1 = tmax + ray * n_max;
    SampleRow row;
    row.init(valid_len[ray], voxel_size[b] * (float)start_scale, S, noise + ray * S,
             sidx + ray * S, st + ray * S);
    if (hi[0] >= 0) {
      bool end = false;   // a slot without a hit ends the list
      for (int i0 = 0; i0 < n_max && !end && row.has < S; i0 += G) {
        const int i = i0 + grp.sub;
        int v = -1;
        float mn = -1.0f, mx = -1.0f;
        if (i < n_max) {
          v = hi[i];
          mn = h0[i];
          mx = h1[i];
        }
        const unsigned gone = grp.vote(v < 0 || mn < 0 || mx < 0);
        end = gone != 0;
        const bool on = !end || grp.sub < __ffs(gone) - 1;
        row.intervals(grp, on, v, mn, mx, on ? node_pos[v].w : 1.0f);
      }
      // leftover slots: one midpoint sample per hit, in hit order (:1156-1174)
      const int left = min(S - row.has, n_max);
      int placed = 0;
      end = false;
      for (int i0 = 0; i0 < left && !end; i0 += G) {
        const int i = i0 + grp.sub;
        int v = -1;
        float mn = -1.0f, mx = -1.0f;
        if (i < left) {
          v = hi[i];
          mn = h0[i];
          mx = h1[i];
        }
        const unsigned gone = grp.vote(v < 0 || mn < 0 || mx < 0);
        const int n = gone ? __ffs(gone) - 1 : G;
        end = gone != 0;
        if (grp.sub < n) row.leftover(row.has + i, v, mn, mx);
        placed += n;
      }
      row.has += placed;
    }
    has = row.has;
  }
  if constexpr (G == 1) {
    for (int j = has; j < S; ++j) {
      sidx[ray * S + j] = -1;
      st[ray * S + j] = -1.0f;
    }
    return;
  }
  const int lane = threadIdx.x & 63;
  const long long ray0 = ray - grp.base / G;
#pragma unroll
  for (int k = 0; k < 64 / G; ++k) {
    const int hk = __builtin_amdgcn_readlane(has, k * G);
    for (int j = hk + lane; j < S; j += 64) {
      sidx[(ray0 + k) * S + j] = -1;
      st[(ray0 + k) * S + j] = -1.0f;
    }
  }
}

// Stable ascending sort of each row; one wave per row, rank counting in LDS.
constexpr int kSortMaxS = 1024;
__global__ void __launch_bounds__(kThreads)
sort_rows(const float* __restrict__ t, int n_rows, int S, float* __restrict__ out,
          int* __restrict__ order) {
  __shared__ float s_v[kThreads / 64][kSortMaxS];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const long long row = (long long)blockIdx.x * (kThreads / 64) + wid;
  const bool active = row < n_rows;
  float* sv = s_v[wid];
  if (active) {
    const float* src = t + row * S;
    for (int i = lane; i < S; i += 64) sv[i] = src[i];
  }
  __syncthreads();
  if (!active) return;
  // A row already in non-decreasing order (every row without samples, all
  // -1) is its own stable sort: rank of element i = i.  (A NaN fails the
  // test and takes the rank loop, as before.)
  bool out_of_order = false;
  for (int i = lane; i + 1 < S; i += 64) out_of_order |= !(sv[i] <= sv[i + 1]);
  if (__ballot(out_of_order) == 0) {
    for (int i = lane; i < S; i += 64) {
      out[row * S + i] = sv[i];
      order[row * S + i] = i;
    }
    return;
  }
  for (int i = lane; i < S; i += 64) {
    float v = sv[i];
    int r = 0;
    for (int j = 0; j < S; ++j) {
      float u = sv[j];
      r += (u < v) || (u == v && j < i);
    }
    out[row * S + r] = v;
    order[row * S + r] = i;
  }
}

// Lanes per ray.  With is_training a node's children are not tested, so there is
// nothing to share; wide rows are bound by their writes.  8 lanes and (lanes
// taken), us: is_training, rate 4, n_max 128, random rays 4,096 33 and (1) 34,
// 16,384 50 and 36, 1,048,576 1514 and 526; n_max 1024 16,384 58 and 64, 65,536
// 193 and 178.  Otherwise, n_max 128, rate 2 65,536 167 and (2) 151, 131,072 259
// and 181, 1,048,576 1585 and 947; rate 4 262,144 in raster order 279 and (4)
// 286, 524,288 random 742 and 571; rate 8 1,048,576 1521 and (4) 1723; n_max 1024
// rate 2 262,144 734 and (2) 802.
int traversal_lanes(long long rays, int rate, int n_max, bool training) {
  const bool narrow = n_max < 512;
  if (training) return rays >= (narrow ? 8192 : 65536) ? 1 : 8;
  if (narrow && rate < 4 && rays >= 1 << 17) return 2;
  if (narrow && rate < 8 && rays >= 1 << 19) return 4;
  return 8;
}

}  // namespace

extern "C" int sailor_octree_voxel_traversal(
    const int32_t* vol_coarse, const float* node_pos, const int32_t* node_info,
    int n_nodes, const float* vol_bbox, const float* voxel_size, int B, int dim_fine,
    int dim_coarse, int rate, const float* ray_ori, const float* ray_dir, int R,
    int n_max_hits, int th_early_stop, int is_training, int opt_num_intersected,
    int32_t* hit_idx, float* tmin, float* tmax, float* valid_len,
    int32_t* status, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && n_max_hits > 0, "voxel_traversal: bad sizes");
  SAILOR_REQUIRE(dim_coarse > 0 && rate >= 1, "voxel_traversal: bad tree dims");
  hipStream_t st = sailor::as_stream(stream);
  if (R == 0) return SAILOR_OK;
  const long long rays = (long long)B * R;
  const int lanes = traversal_lanes(rays, rate, n_max_hits, is_training != 0);
  auto kern = traversal_kernel<8>;
  if (lanes == 4) kern = traversal_kernel<4>;
  if (lanes == 2) kern = traversal_kernel<2>;
  if (lanes == 1) {
    kern = traversal_kernel<1>;
    const long long n = rays * n_max_hits;
    hipLaunchKernelGGL(fill_lists,
                       dim3((unsigned)std::min<long long>((n + kThreads - 1) / kThreads, 65535)),
                       dim3(kThreads), 0, st, hit_idx, tmin, tmax, n);
    if (int e = sailor::check_launch("voxel_traversal (fill)")) return e;
  }
  return sailor::in_parts(rays, [&](long long first, long long n) {
    hipLaunchKernelGGL(kern, dim3(sailor::ceil_div(n, kWalkThreads / lanes)), dim3(kWalkThreads), 0,
                       st, vol_coarse, reinterpret_cast<const float4*>(node_pos),
                       reinterpret_cast<const int4*>(node_info), n_nodes, vol_bbox, voxel_size,
                       first, first + n, dim_fine, dim_coarse, rate, ray_ori, ray_dir, R,
                       n_max_hits, th_early_stop, is_training, opt_num_intersected, hit_idx,
                       tmin, tmax, valid_len, status);
    return sailor::check_launch("voxel_traversal");
  });
}

extern "C" int sailor_octree_sampling_coarse(
    const int32_t* hit_idx, const float* tmin, const float* tmax,
    const float* noise, const float* valid_len, const float* node_pos,
    const float* voxel_size, int B, int R, int n_max_hits, int S, int start_scale,
    int32_t* sampled_idx, float* sampled_t, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && S > 0 && n_max_hits > 0, "sampling: bad sizes");
  if (R == 0) return SAILOR_OK;
  // 8 lanes and a lane per ray, us: 131,072 rays of 1 sample 13 and 7.5, of 4
  // 14 and 11; 524,288 of 1 sample 36 and 22, of 2 26 and 42
  const int lanes = S == 1 || (S <= 4 && (long long)B * R < 1 << 18) ? 1 : sailor::kGroup;
  auto kern = sampling_kernel<8>;
  if (lanes == 1) kern = sampling_kernel<1>;
  return sailor::in_parts((long long)B * R, [&](long long first, long long n) {
    hipLaunchKernelGGL(kern, dim3(sailor::ceil_div(n, kWalkThreads / lanes)), dim3(kWalkThreads), 0,
                       sailor::as_stream(stream), hit_idx, tmin, tmax, noise, valid_len,
                       reinterpret_cast<const float4*>(node_pos), voxel_size, first, first + n,
                       R, n_max_hits, S, start_scale, sampled_idx, sampled_t);
    return sailor::check_launch("sampling_coarse");
  });
}

extern "C" int sailor_sort_samplings(const float* t, int n_rows, int S, float* sorted,
                                     int32_t* order, void* stream) {
  SAILOR_REQUIRE(S > 0 && S <= kSortMaxS, "sort_samplings: S must be in [1, %d]", kSortMaxS);
  if (n_rows <= 0) return SAILOR_OK;
  hipLaunchKernelGGL(sort_rows, dim3(sailor::ceil_div(n_rows, kThreads / 64)),
                     dim3(kThreads), 0, sailor::as_stream(stream), t, n_rows, S, sorted,
                     order);
  return sailor::check_launch("sort_samplings");
}
