// Fused per-ray trace: camera ray -> coarse-grid DDA -> length-weighted
// sampling, without materialising the reference's [B, R, 1024] hit lists.
//
// The reference chain is rays_calculating (sampling_kernel.cu:411-486) ->
// voxel_traversal (intersection_kernel.cu:827-895) ->
// ray_voxels_points_sampling_coarse (sampling_kernel.cu:1070-1177).  The
// sampler needs the total weighted valid length of a ray before it can place
// the first sample, so instead of storing every hit in HBM the walk is done
// in passes: pass 1 accumulates the valid length, pass 2 emits samples
// (stopping once all S slots are used), and a third pass places the leftover
// midpoint samples.  8 lanes walk a ray together, 4 or 2 in large targets of
// trees with few children per node (traversal_common.h).  Pass 1
// keeps up to kHitCache hits per ray in LDS, and rays within that take passes
// 2 and 3 from there, a hit per lane; longer rays walk again.  Every
// expression is the one of the separate kernels, so the samples are
// bit-identical to the unfused path.
// Bound by the latency of the walk (few of 262,144 rays meet the performer):
// one lane per ray took 551 us for a 512^2 target of a 256^3 grid, 8
// lanes 289 us.
// Compiled with -ffp-contract=off.
#include "common.h"
#include "traversal_common.h"

namespace {

using sailor::LaneGroup;
using sailor::SampleRow;

// One wave per workgroup, 8 rays: waves differ widely in how much of the
// performer they meet, and a workgroup holds its place until its last wave is
// done (512^2 target: 16 rays x 4 tiles of two waves 487, 16 rays 380, this
// 300 us).
constexpr int kThreads = 64;

// Hits of walk 1 kept in LDS (up to kHitCache per ray): rays with at most that
// many place their samples from there instead of walking the DDA again.  44
// leaves no ray of the 512^2 workload walking again and keeps the second walk
// covered by the test scene, whose longest ray has 46 hits.
constexpr int kHitCache = 44;

// With fewer than 8 lanes per ray a wave has more rays and keeps the nodes
// alone; an interval is the slab test of the node again, by the same code.
template <int G>
struct CacheSink {
  static constexpr int kRays = kThreads / G;
  static constexpr bool kIntervals = G == 8;
  int* node;     // [kHitCache] of this ray, one slot every kRays words
  float *t0, *t1;
  const LaneGroup<G>& grp;
  __device__ __forceinline__ void keep(int pos, int nd, float a, float b) {
    if (pos < kHitCache) {
      node[pos * kRays] = nd;
      if constexpr (kIntervals) {
        t0[pos * kRays] = a;
        t1[pos * kRays] = b;
      }
    }
  }
  // hit k: its interval and, in the last component, its node's size
  __device__ __forceinline__ float3 hit(const sailor::RayCtx& c, int k) const {
    const int nd = node[k * kRays];
    if constexpr (kIntervals) return make_float3(t0[k * kRays], t1[k * kRays], c.np[nd].w);
    const float4 q = c.np[nd];
    const float2 v = sailor::slab_test(c.o, c.inv, make_float3(q.x, q.y, q.z), q.w);
    return make_float3(v.x, v.y, q.w);
  }
  __device__ __forceinline__ void put(int pos, int nd, float a, float b) {
    if (grp.sub == 0) keep(pos, nd, a, b);
  }
  __device__ __forceinline__ void put_lanes(int pos, int nd, float a, float b, bool hit,
                                            unsigned votes) {
    if (hit) keep(pos + grp.before(votes), nd, a, b);
  }
  __device__ __forceinline__ bool stop() const { return false; }
};

// Second walk of a ray with more hits: samples as they come.
template <int G>
struct SampleSink {
  SampleRow& row;
  const float4* np;
  const LaneGroup<G>& grp;
  __device__ __forceinline__ void put(int, int nd, float a, float b) {
    if (row.has < row.S) row.intervals(grp, grp.sub == 0, nd, a, b, np[nd].w);
  }
  __device__ __forceinline__ void put_lanes(int, int nd, float a, float b, bool hit, unsigned) {
    if (row.has < row.S) row.intervals(grp, hit, nd, a, b, hit ? np[nd].w : 1.0f);
  }
  __device__ __forceinline__ bool stop() const { return row.has >= row.S; }
};

// Third walk: hit number pos < left takes slot has + pos.
template <int G>
struct LeftoverSink {
  SampleRow& row;
  const LaneGroup<G>& grp;
  int left;
  int seen;
  __device__ __forceinline__ void put(int pos, int nd, float a, float b) {
    if (grp.sub == 0 && pos < left) row.leftover(row.has + pos, nd, a, b);
    seen = pos + 1;
  }
  __device__ __forceinline__ void put_lanes(int pos, int nd, float a, float b, bool hit,
                                            unsigned votes) {
    const int k = pos + grp.before(votes);
    if (hit && k < left) row.leftover(row.has + k, nd, a, b);
  }
  __device__ __forceinline__ bool stop() const { return seen >= left; }
};

__device__ __forceinline__ void inv3(const float* M, float* out) {
  float a1 = M[0], b1 = M[1], c1 = M[2];
  float a2 = M[3], b2 = M[4], c2 = M[5];
  float a3 = M[6], b3 = M[7], c3 = M[8];
  float det = a1 * (b2 * c3 - c2 * b3) - a2 * (b1 * c3 - c1 * b3) +
              a3 * (b1 * c2 - c1 * b2);
  out[0] = (b2 * c3 - c2 * b3) / det;
  out[1] = (b3 * c1 - c3 * b1) / det;
  out[2] = (b1 * c2 - c1 * b2) / det;
  out[3] = (a3 * c2 - c3 * a2) / det;
  out[4] = (a1 * c3 - c1 * a3) / det;
  out[5] = (a2 * c1 - c2 * a1) / det;
  out[6] = (a2 * b3 - b2 * a3) / det;
  out[7] = (b1 * a3 - a1 * b3) / det;
  out[8] = (b2 * a1 - a2 * b1) / det;
}

// grid = (ceil(pixels / kRays), B), pixels from `first` on; G lanes per target
// pixel.
template <int G>
__global__ void __launch_bounds__(kThreads, 6)
trace_kernel(const float* __restrict__ K, const float* __restrict__ Rm,
             const float* __restrict__ Tv, int H, int W, int first,
             const int* __restrict__ vc, const float4* __restrict__ node_pos,
             const int4* __restrict__ node_info, int n_nodes,
             const float* __restrict__ vol_bbox, const float* __restrict__ voxel_size,
             int dim_fine, int dim_coarse, int rate, int start_scale, int S,
             const float* __restrict__ noise, float* __restrict__ rays_out,
             int* __restrict__ sidx, float* __restrict__ st, float* __restrict__ vl_out) {
  constexpr int kRays = kThreads / G;
  constexpr int kHits = CacheSink<G>::kIntervals ? kHitCache * kRays : 1;
  __shared__ float s_m[18];
  __shared__ int s_node[kHitCache * kRays];
  __shared__ float s_t0[kHits], s_t1[kHits];
  const int b = blockIdx.y;
  if (threadIdx.x < 2) inv3((threadIdx.x ? Rm : K) + (size_t)b * 9, s_m + 9 * threadIdx.x);
  __syncthreads();
  const LaneGroup<G> grp;
  const int slot = threadIdx.x / G;
  const int HW = H * W;
  const long long p64 = first + (long long)blockIdx.x * kRays + slot;
  // groups past the image carry no ray but stay for the wave's tail fill
  const bool live = p64 < HW;
  const int p = (int)p64;
  const long long ray = (long long)b * HW + p64;
  int has = S;   // samples placed; rows past the image have no tail
  if (live) {
    // ---- camera ray (rays_calculating_kernel, :443-484)
    const int h = p / W, w = p - h * W;
    const float* ki = s_m;
    const float* ri = s_m + 9;
    const float* t = Tv + (size_t)b * 3;
    float o[3], cd[3], wd[3], d[3];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      o[k] = -ri[3 * k + 0] * t[0] - ri[3 * k + 1] * t[1] - ri[3 * k + 2] * t[2];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      cd[k] = (float)w * ki[3 * k + 0] + (float)h * ki[3 * k + 1] + 1.0f * ki[3 * k + 2];
#pragma unroll
    for (int k = 0; k < 3; ++k)
      wd[k] = cd[0] * ri[3 * k + 0] + cd[1] * ri[3 * k + 1] + cd[2] * ri[3 * k + 2];
    const float nrm = sqrtf(wd[0] * wd[0] + wd[1] * wd[1] + wd[2] * wd[2]);
    const double den = (double)nrm + 1e-10;
#pragma unroll
    for (int k = 0; k < 3; ++k) d[k] = (float)((double)wd[k] / den);
    for (int k = rays_out ? grp.sub : 6; k < 6; k += G)
      rays_out[ray * 6 + k] = k == 0 ? o[0] : k == 1 ? o[1] : k == 2 ? o[2]
                              : k == 3 ? d[0] : k == 4 ? d[1] : d[2];
    // ---- walk 1: weighted valid length
    sailor::RayCtx ctx;
    ctx.init(vc, node_pos, node_info, n_nodes, vol_bbox, voxel_size, b, dim_fine, dim_coarse,
             rate, o, d);
    CacheSink<G> cs{s_node + slot, s_t0 + slot, s_t1 + slot, grp};
    float vl = 0.0f;
    const int count = sailor::traverse(ctx, grp, -1, false, -1, cs, &vl);
    sailor::wave_fence();
    if (vl_out && grp.sub == 0) vl_out[ray] = vl;
    has = 0;
    if (count > 0) {
      SampleRow row;
      row.init(vl, voxel_size[b] * (float)start_scale, S, noise + ray * S, sidx + ray * S,
               st + ray * S);
      if (count <= kHitCache) {
        // ---- samples (sampling_kernel.cu:1125-1154) ...
        for (int k0 = 0; k0 < count && row.has < S; k0 += G) {
          const int k = k0 + grp.sub;
          const bool on = k < count;
          const float3 hit = on ? cs.hit(ctx, k) : make_float3(0.0f, 0.0f, 1.0f);
          row.intervals(grp, on, on ? cs.node[k * kRays] : 0, hit.x, hit.y, hit.z);
        }
        // ---- ... and leftover midpoints (:1156-1174)
        const int left = min(S - row.has, count);
        for (int k = grp.sub; k < left; k += G) {
          const float3 hit = cs.hit(ctx, k);
          row.leftover(row.has + k, cs.node[k * kRays], hit.x, hit.y);
        }
        row.has += left;
      } else {
        float dummy;
        SampleSink<G> ss{row, node_pos, grp};
        sailor::traverse(ctx, grp, -1, false, -1, ss, &dummy);
        if (row.has < S) {
          LeftoverSink<G> ls{row, grp, S - row.has, 0};
          sailor::traverse(ctx, grp, -1, false, -1, ls, &dummy);
          row.has += min(S - row.has, count);
        }
      }
      has = row.has;
    }
  }
  // ---- the rest of every row is -1, written row by row by the whole wave
  // (most rays have no sample: their rows are one stretch of memory)
  const int lane = threadIdx.x;
#pragma unroll
  for (int k = 0; k < 64 / G; ++k) {
    const int hk = __builtin_amdgcn_readlane(has, k * G);
    if (hk >= S) continue;
    const long long rk = ray - grp.base / G + k;
    for (int j = hk + lane; j < S; j += 64) {
      sidx[rk * S + j] = -1;
      st[rk * S + j] = -1.0f;
    }
  }
}

// Lanes per ray.  8 and fewer lanes, us, with 4, 16 and 48 samples a ray: rate 2
// 320^2 158, 184, 259 and (2 lanes) 165, 215, 374; 512^2 277, 312, 421 and 204,
// 256, 397; 1024^2 832, 874, 1099 and 469, 573, 901.  Rate 4 512^2 211, 235, 318
// and (4 lanes) 228, 264, 387; 1024^2 549, 574, 750 and 459, 522, 736.  Rate 8
// 1024^2 589, 627, 784 and (4 lanes) 687, 748, 977.
int trace_lanes(long long rays, int rate) {
  if (rate < 4 && rays >= 1 << 18) return 2;
  if (rate < 8 && rays >= 1 << 19) return 4;
  return 8;
}

}  // namespace

extern "C" int sailor_trace_sample(const float* K, const float* R, const float* T, int B,
                                   int H, int W, const int32_t* vol_coarse,
                                   const float* node_pos, const int32_t* node_info,
                                   int n_nodes, const float* vol_bbox,
                                   const float* voxel_size, int dim_fine, int dim_coarse,
                                   int start_scale, int S, const float* noise,
                                   float* rays_out, int32_t* sampled_idx, float* sampled_t,
                                   float* valid_len, void* stream) {
  SAILOR_REQUIRE(B > 0 && H > 0 && W > 0 && S > 0, "trace_sample: bad sizes");
  SAILOR_REQUIRE(dim_coarse > 0 && dim_fine % dim_coarse == 0, "trace_sample: bad dims");
  const int rate = dim_fine / dim_coarse;
  const int lanes = trace_lanes((long long)B * H * W, rate);
  auto kern = trace_kernel<8>;
  if (lanes == 4) kern = trace_kernel<4>;
  if (lanes == 2) kern = trace_kernel<2>;
  return sailor::in_parts((long long)H * W, [&](long long first, long long n) {
    hipLaunchKernelGGL(kern, dim3(sailor::ceil_div(n, kThreads / lanes), B), dim3(kThreads), 0,
                       sailor::as_stream(stream), K, R, T, H, W, (int)first, vol_coarse,
                       reinterpret_cast<const float4*>(node_pos),
                       reinterpret_cast<const int4*>(node_info), n_nodes, vol_bbox, voxel_size,
                       dim_fine, dim_coarse, rate, start_scale, S, noise, rays_out, sampled_idx,
                       sampled_t, valid_len);
    return sailor::check_launch("trace_sample");
  });
}
