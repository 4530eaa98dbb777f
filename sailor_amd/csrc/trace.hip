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
// midpoint samples.  8 lanes walk a ray together (traversal_common.h).  Pass 1
// keeps up to kHitCache hits per ray in LDS, and rays within that take passes
// 2 and 3 from there, 8 hits at a time; longer rays walk again.  Every
// expression is the one of the separate kernels, so the samples are
// bit-identical to the unfused path.
// Bound by the latency of the walk (few of 262,144 rays meet the performer):
// one lane per ray took 551 us for a 512^2 target of a 256^3 grid, 8
// lanes 289 us.
// Compiled with -ffp-contract=off.
#include "common.h"
#include "traversal_common.h"

namespace {

using sailor::kGroup;
using sailor::LaneGroup;
using sailor::SampleRow;

// One wave per workgroup, 8 rays: waves differ widely in how much of the
// performer they meet, and a workgroup holds its place until its last wave is
// done (512^2 target: 16 rays x 4 tiles of two waves 487, 16 rays 380, this
// 300 us).
constexpr int kThreads = 64;
constexpr int kRays = kThreads / kGroup;

// Hits of walk 1 kept in LDS (up to kHitCache per ray): rays with at most that
// many place their samples from there instead of walking the DDA again.  44
// leaves no ray of the 512^2 workload walking again and keeps the second walk
// covered by the test scene, whose longest ray has 46 hits.
constexpr int kHitCache = 44;

struct CacheSink {
  int* node;     // [kHitCache] of this ray, one slot every kRays words
  float *t0, *t1;
  const LaneGroup& grp;
  __device__ __forceinline__ void keep(int pos, int nd, float a, float b) {
    if (pos < kHitCache) {
      node[pos * kRays] = nd;
      t0[pos * kRays] = a;
      t1[pos * kRays] = b;
    }
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
struct SampleSink {
  SampleRow& row;
  const float4* np;
  const LaneGroup& grp;
  __device__ __forceinline__ void put(int, int nd, float a, float b) {
    if (row.has < row.S) row.intervals(grp, grp.sub == 0, nd, a, b, np[nd].w);
  }
  __device__ __forceinline__ void put_lanes(int, int nd, float a, float b, bool hit, unsigned) {
    if (row.has < row.S) row.intervals(grp, hit, nd, a, b, hit ? np[nd].w : 1.0f);
  }
  __device__ __forceinline__ bool stop() const { return row.has >= row.S; }
};

// Third walk: hit number pos < left takes slot has + pos.
struct LeftoverSink {
  SampleRow& row;
  const LaneGroup& grp;
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

// grid = (ceil(pixels / kRays), B), pixels from `first` on; 8 lanes per target
// pixel.
__global__ void __launch_bounds__(kThreads, 6)
trace_kernel(const float* __restrict__ K, const float* __restrict__ Rm,
             const float* __restrict__ Tv, int H, int W, int first,
             const int* __restrict__ vc, const float4* __restrict__ node_pos,
             const int4* __restrict__ node_info, int n_nodes,
             const float* __restrict__ vol_bbox, const float* __restrict__ voxel_size,
             int dim_fine, int dim_coarse, int rate, int start_scale, int S,
             const float* __restrict__ noise, float* __restrict__ rays_out,
             int* __restrict__ sidx, float* __restrict__ st, float* __restrict__ vl_out) {
  __shared__ float s_m[18];
  __shared__ int s_node[kHitCache * kRays];
  __shared__ float s_t0[kHitCache * kRays], s_t1[kHitCache * kRays];
  const int b = blockIdx.y;
  if (threadIdx.x < 2) inv3((threadIdx.x ? Rm : K) + (size_t)b * 9, s_m + 9 * threadIdx.x);
  __syncthreads();
  const LaneGroup grp;
  const int slot = threadIdx.x / kGroup;
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
    if (rays_out && grp.sub < 6) {
      const int k = grp.sub;
      rays_out[ray * 6 + k] = k == 0 ? o[0] : k == 1 ? o[1] : k == 2 ? o[2]
                              : k == 3 ? d[0] : k == 4 ? d[1] : d[2];
    }
    // ---- walk 1: weighted valid length
    sailor::RayCtx ctx;
    ctx.init(vc, node_pos, node_info, n_nodes, vol_bbox, voxel_size, b, dim_fine, dim_coarse,
             rate, o, d);
    CacheSink cs{s_node + slot, s_t0 + slot, s_t1 + slot, grp};
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
        for (int k0 = 0; k0 < count && row.has < S; k0 += kGroup) {
          const int k = k0 + grp.sub;
          const bool on = k < count;
          const int nd = on ? cs.node[k * kRays] : 0;
          const float a0 = on ? cs.t0[k * kRays] : 0.0f, a1 = on ? cs.t1[k * kRays] : 0.0f;
          row.intervals(grp, on, nd, a0, a1, on ? node_pos[nd].w : 1.0f);
        }
        // ---- ... and leftover midpoints (:1156-1174)
        const int left = min(S - row.has, count);
        for (int k = grp.sub; k < left; k += kGroup)
          row.leftover(row.has + k, cs.node[k * kRays], cs.t0[k * kRays], cs.t1[k * kRays]);
        row.has += left;
      } else {
        float dummy;
        SampleSink ss{row, node_pos, grp};
        sailor::traverse(ctx, grp, -1, false, -1, ss, &dummy);
        if (row.has < S) {
          LeftoverSink ls{row, grp, S - row.has, 0};
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
  for (int k = 0; k < 64 / kGroup; ++k) {
    const int hk = __builtin_amdgcn_readlane(has, k * kGroup);
    if (hk >= S) continue;
    const long long rk = ray - grp.base / kGroup + k;
    for (int j = hk + lane; j < S; j += 64) {
      sidx[rk * S + j] = -1;
      st[rk * S + j] = -1.0f;
    }
  }
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
  return sailor::in_parts((long long)H * W, [&](long long first, long long n) {
    hipLaunchKernelGGL(trace_kernel, dim3(sailor::ceil_div(n, kRays), B), dim3(kThreads), 0,
                       sailor::as_stream(stream), K, R, T, H, W, (int)first, vol_coarse,
                       reinterpret_cast<const float4*>(node_pos),
                       reinterpret_cast<const int4*>(node_info), n_nodes, vol_bbox, voxel_size,
                       dim_fine, dim_coarse, rate, start_scale, S, noise, rays_out, sampled_idx,
                       sampled_t, valid_len);
    return sailor::check_launch("trace_sample");
  });
}
