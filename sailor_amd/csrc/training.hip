// Training-only kernels of the octree path: the recursive octree traversal,
// the adaptive (length- and size-weighted) point sampling and the trilinear
// aggregation of per-corner features with its backward.
//
// Follows c_lib/VoxelEncoding/src/intersection_kernel.cu (octree_traversal
// :738-825, ray_octree_traversal :441-643, RayVoxelIntersectionNodeList
// :72-126) and c_lib/VoxelEncoding/src/sampling_kernel.cu
// (ray_voxels_points_sampling :1178-1248 with ray_voxels_sampling_kernel
// :911-982 and ray_voxels_further_sampling_kernel :984-1068,
// trilinear_aggregate_features[_backward] :162-327, 1384-1462).
//
// The reference appends per-ray entries and samples through atomicAdd
// queues from one thread per (ray, coarse hit) and accumulates the ray's
// valid length with float atomics, so its entry order and the low bits of
// the valid length depend on scheduling.  Here a ray's lanes
// append in coarse-hit order, which is one of the orders the reference can
// produce, and the result is reproducible bit for bit.  Lists are bounded by
// their capacity with an overflow flag (the reference writes past the row;
// its DFS buffers hold 8 entries).  Compiled with -ffp-contract=off.
#include "common.h"
#include "traversal_common.h"

namespace {

constexpr int kThreads = 256;

using sailor::kGroup;
using sailor::LaneGroup;

constexpr int kWalkThreads = 64;   // one wave: rays differ widely in length
constexpr int kEntries = 32;       // entries of a coarse hit kept in LDS per ray

// Receives the coarse hits of the DDA (RayVoxelIntersectionNodeList) and
// expands each into its fine entries right away: the coarse entry, then the
// children in stack order (last child first) that the slab test hits; an
// interval equal to one already listed for this coarse hit keeps the
// smaller node (ray_octree_traversal :518-567).  The ray's G lanes test G
// children at a time and compare a hit with G listed entries at a time; a
// coarse hit's entries are kept in LDS, those past kEntries are read back from
// their row: a ray in general position meets at most 3 n - 2 of n^3 children (22
// at rate 8, 46 at rate 16), one along shared faces or edges more.
template <int G>
struct TreeSink {
  static constexpr int kRays = kWalkThreads / G;
  const float4* np;
  const int4* ni;
  int n_nodes;
  float3 o, inv;
  int* idx_c;
  float* t0_c;
  float* t1_c;
  int cap_c;
  int* idx;
  float* t0;
  float* t1;
  int cap;
  const LaneGroup<G>& grp;
  int* e_node;     // [kEntries] of this ray, one slot every kRays words
  float *e_t0, *e_t1;
  int cnt;
  float vl;
  bool overflow;

  // entry `pos` of the row, `k`-th of this coarse hit, by one lane
  __device__ __forceinline__ void store(int pos, int k, int node, float a, float b) {
    if (grp.sub != 0) return;
    if (pos < cap) {
      idx[pos] = node;
      t0[pos] = a;
      t1[pos] = b;
    }
    if (k < kEntries) {
      e_node[k * kRays] = node;
      e_t0[k * kRays] = a;
      e_t1[k * kRays] = b;
    }
  }
  __device__ __forceinline__ void put(int pos, int node, float a, float b) {
    if (pos < cap_c) {
      if (grp.sub == 0) {
        idx_c[pos] = node;
        t0_c[pos] = a;
        t1_c[pos] = b;
      }
    } else {
      overflow = true;
    }
    const float start_vs = np[node].w;
    const int g0 = cnt;
    sailor::wave_fence();   // the last coarse hit's entries are no longer read
    store(cnt, 0, node, a, b);
    cnt += 1;
    const int4 info = ni[node];
    if (info.z >= 0) {
      const int last = min(info.z + info.w, n_nodes) - 1;
      int ch = last - grp.sub;
      float4 qn = ch >= info.z ? np[ch] : make_float4(0.f, 0.f, 0.f, 0.f);
      for (int ch0 = last; ch0 >= info.z; ch0 -= G, ch -= G) {
        const float4 q = qn;
        if (ch - G >= info.z) qn = np[ch - G];
        const float2 cd = sailor::slab_test(o, inv, make_float3(q.x, q.y, q.z), q.w);
        unsigned votes = grp.vote(ch >= info.z && !(cd.x == -1.0f || cd.y == -1.0f));
        while (votes) {
          const int i = __ffs(votes) - 1;
          votes &= votes - 1;
          const float c0 = grp.from(cd.x, i), c1 = grp.from(cd.y, i), cs = grp.from(q.w, i);
          sailor::wave_fence();   // entries stored so far
          // the first listed entry of this coarse hit with the same interval
          const int lim = cnt < cap ? cnt : cap;
          int same = -1;
          for (int j0 = g0; j0 < lim && same < 0; j0 += G) {
            const int j = j0 + grp.sub, k = j - g0;
            bool eq = false;
            if (j < lim) {
              if (k < kEntries) {
                eq = e_t0[k * kRays] == c0 && e_t1[k * kRays] == c1;
              } else {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
                eq = t0[j] == c0 && t1[j] == c1;
              }
            }
            const unsigned e = grp.vote(eq);
            if (e) same = j0 + __ffs(e) - 1;
          }
          if (same < 0) {
            store(cnt, cnt - g0, ch0 - i, c0, c1);
            cnt += 1;
          } else if (grp.sub == 0) {
            const int k = same - g0;
            const int held = k < kEntries ? e_node[k * kRays] : idx[same];
            if (np[held].w > cs) {
              idx[same] = ch0 - i;
              if (k < kEntries) e_node[k * kRays] = ch0 - i;
            }
          }
        }
      }
    }
    if (cnt > cap) overflow = true;
    // valid length of the listed entries, in order
    const int lim = cnt < cap ? cnt : cap;
    sailor::wave_fence();
    for (int j0 = g0; j0 < lim; j0 += G) {
      const int j = j0 + grp.sub, k = j - g0;
      float part = 0.0f;
      if (j < lim) {
        float a0, a1;
        int nd;
        if (k < kEntries) {
          a0 = e_t0[k * kRays];
          a1 = e_t1[k * kRays];
          nd = e_node[k * kRays];
        } else {
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
          a0 = t0[j];
          a1 = t1[j];
          nd = idx[j];
        }
        const float scale = start_vs / np[nd].w;
        part = (a1 - a0) * scale;
      }
      const int n = min(G, lim - j0);
      for (int i = 0; i < n; ++i) vl += grp.from(part, i);
    }
  }
  __device__ __forceinline__ void put_lanes(int, int, float, float, bool, unsigned) {}
  __device__ __forceinline__ bool stop() const { return false; }
};

// G lanes per ray (traversal_common.h); each wave then fills what its rows have
// left with -1.  20,000 random rays through a 128^3 tree filled 79 of 256
// CUs with a lane per ray and took 1221 us after two fills, now 171 us in all.
template <int G>
__global__ void __launch_bounds__(kWalkThreads)
octree_traversal_kernel(const int* __restrict__ vc, const float4* __restrict__ node_pos,
                        const int4* __restrict__ node_info, int n_nodes,
                        const float* __restrict__ vol_bbox, const float* __restrict__ voxel_size,
                        long long first, long long ray_end, int dim_fine, int dim_coarse, int rate,
                        const float* __restrict__ ray_ori, const float* __restrict__ ray_dir,
                        int R, int n_max_c, int n_max, int th_early_stop, int opt_num,
                        int* __restrict__ idx_c, float* __restrict__ t0_c,
                        float* __restrict__ t1_c, int* __restrict__ idx,
                        float* __restrict__ t0, float* __restrict__ t1,
                        float* __restrict__ valid_len, int* __restrict__ status) {
  constexpr int kRays = kWalkThreads / G;
  __shared__ int s_node[kEntries * kRays];
  __shared__ float s_t0[kEntries * kRays], s_t1[kEntries * kRays];
  const LaneGroup<G> grp;
  const int slot = threadIdx.x / G;
  const long long ray = first + (long long)blockIdx.x * kRays + slot;
  int n_coarse = 0, n_fine = 0, filled_c = n_max_c, filled = n_max;
  bool overflow = false;
  if (ray < ray_end) {
    const int b = (int)(ray / R);
    sailor::RayCtx ctx;
    ctx.init(vc, node_pos, node_info, n_nodes, vol_bbox, voxel_size, b, dim_fine, dim_coarse,
             rate, ray_ori + ray * 3, ray_dir + ray * 3);
    TreeSink<G> sink{node_pos, node_info, n_nodes, ctx.o, ctx.inv,
                  idx_c + ray * n_max_c, t0_c + ray * n_max_c, t1_c + ray * n_max_c, n_max_c,
                  idx + ray * n_max, t0 + ray * n_max, t1 + ray * n_max, n_max,
                  grp, s_node + slot, s_t0 + slot, s_t1 + slot,
                  0, 0.0f, false};
    float vl_coarse = 0.0f;  // the coarse pass adds no valid length (:90-126)
    n_coarse = sailor::traverse(ctx, grp, th_early_stop, true, opt_num, sink, &vl_coarse);
    if (grp.sub == 0) valid_len[ray] = sink.vl;
    n_fine = sink.cnt;
    overflow = sink.overflow;
    filled_c = min(n_coarse, n_max_c);
    filled = min(n_fine, n_max);
  }
  const long long ray0 = ray - grp.base / G;
  auto fill = [&](int used, int cap, int* ids, float* a, float* c) {
#pragma unroll 1
    for (int k = 0; k < 64 / G; ++k) {
      const int from = __builtin_amdgcn_readlane(used, k * G);
      if (from >= cap) continue;
      const long long row = (ray0 + k) * cap;
      const int lane = threadIdx.x & 63;
      sailor::fill_row(reinterpret_cast<unsigned*>(ids + row), from, cap, 0xffffffffu, lane);
      sailor::fill_row(reinterpret_cast<unsigned*>(a + row), from, cap, 0xbf800000u, lane);
      sailor::fill_row(reinterpret_cast<unsigned*>(c + row), from, cap, 0xbf800000u, lane);
    }
  };
  fill(filled_c, n_max_c, idx_c, t0_c, t1_c);
  fill(filled, n_max, idx, t0, t1);
  int mc = n_coarse, mf = n_fine;
  for (int o = 32; o > 0; o >>= 1) {
    mc = max(mc, __shfl_xor(mc, o, 64));
    mf = max(mf, __shfl_xor(mf, o, 64));
  }
  const unsigned long long ov = __ballot(overflow);
  if ((threadIdx.x & 63) == 0) {
    if (mc > 0) atomicMax(status, mc);
    if (mf > 0) atomicMax(status + 1, mf);
    if (ov) atomicOr(status + 2, 1);
  }
}

// ray_voxels_sampling_kernel over the hits in order, then
// ray_voxels_further_sampling_kernel, by 8 lanes per ray: 8 hits at a time
// (their slots by a prefix sum), slots written 8 at a time.  A lane per ray,
// every row access in another line, took 92 us for 20,000 rays, this 20 us.
__global__ void __launch_bounds__(kWalkThreads)
adaptive_sampling_kernel(const int* __restrict__ hit_idx, const float* __restrict__ tmin,
                         const float* __restrict__ tmax, const float* __restrict__ noise,
                         const float* __restrict__ valid_len,
                         const float4* __restrict__ node_pos, int n_nodes,
                         const float* __restrict__ voxel_size, long long first, long long ray_end,
                         int R, int n_max, int max_hits, int S, int start_scale, int* __restrict__ sidx,
                         float* __restrict__ st) {
  constexpr int kRays = kWalkThreads / kGroup;
  const LaneGroup<kGroup> grp;
  const long long ray = first + (long long)blockIdx.x * kRays + threadIdx.x / kGroup;
  if (ray >= ray_end) return;   // whole groups
  const int b = (int)(ray / R);
  const int* hi = hit_idx + ray * n_max;
  const float* mn_ = tmin + ray * n_max;
  const float* mx_ = tmax + ray * n_max;
  const float* rnd = noise + ray * S;
  int* oi = sidx + ray * S;
  float* ot = st + ray * S;
  const float vlen = valid_len[ray];
  const float start_vs = voxel_size[b] * (float)start_scale;
  int cnt = 0;
  // ray_voxels_sampling_kernel visits the first max_hits slots of every ray
  // (num_max_intersected_voxels_fine, :944)
  for (int i0 = 0; i0 < max_hits && cnt < S; i0 += kGroup) {
    const int i = i0 + grp.sub;
    const int vi = i < max_hits ? hi[i] : -1;
    const bool on = vi >= 0 && vi < n_nodes;
    int n = 0;
    float mn = 0.0f, off = 0.0f;
    if (on) {
      mn = mn_[i];
      const float mx = mx_[i];
      const float rate = start_vs / node_pos[vi].w;
      n = sailor::sat_f2i((mx - mn) * rate * (float)S / vlen);
      n = n >= 1 ? n : 1;
      off = (mx - mn) / (float)(n + 1);
    }
    const int want = n < S ? n : S;
    const int end = grp.inclusive_sum(want);
    const int slot = cnt + end - want;
    for (int j = 0; j < want && slot + j < S; ++j) {
      const float u = rnd[slot + j];
      const float basic = mn + off * (float)(j + 1);
      ot[slot + j] = (float)((double)basic - (double)off / 2.0 + (double)(off * u));
      oi[slot + j] = vi;
    }
    cnt = min(S, cnt + grp.from(end, kGroup - 1));
  }
  // the first of the smallest nodes' hits with the smallest midpoint: each
  // lane's own hits in order, then the lanes'
  float min_mid = 99999.0f, min_vs = 99999.0f, z0 = -1.0f, z1 = -1.0f;
  int min_idx = -1, min_at = n_max;
  bool nan_mid = false;
  bool end = cnt >= S;   // no slot left to fill
  for (int i0 = 0; i0 < n_max && !end; i0 += kGroup) {
    const int i = i0 + grp.sub;
    const int vi = i < n_max ? hi[i] : -1;
    const unsigned gone = grp.vote(vi == -1);
    end = gone != 0;
    if (vi < 0 || vi >= n_nodes || (gone && grp.sub >= __ffs(gone) - 1)) continue;
    const float vs = node_pos[vi].w;
    if (!(vs <= min_vs)) continue;
    const float a = mn_[i], c = mx_[i];
    const float mid = (float)((double)(a + c) / 2.0);
    nan_mid |= mid != mid;
    if (vs < min_vs || mid < min_mid) {
      min_mid = mid;
      z0 = a;
      z1 = c;
      min_idx = vi;
      min_at = i;
    }
    min_vs = vs;
  }
  // a NaN midpoint (lists of another origin) stays if it comes first and never
  // replaces another: the hits of all lanes in order, by every lane
  if (grp.vote(nan_mid)) {
    min_mid = min_vs = 99999.0f;
    min_idx = -1;
    for (int i = 0; i < n_max && hi[i] != -1; ++i) {
      const int vi = hi[i];
      if (vi < 0 || vi >= n_nodes) continue;
      const float vs = node_pos[vi].w;
      if (!(vs <= min_vs)) continue;
      const float a = mn_[i], c = mx_[i];
      const float mid = (float)((double)(a + c) / 2.0);
      if (vs < min_vs || mid < min_mid) {
        min_mid = mid;
        z0 = a;
        z1 = c;
        min_idx = vi;
      }
      min_vs = vs;
    }
    min_at = 0;   // all lanes agree
  }
#pragma unroll
  for (int o = 1; o < kGroup; o <<= 1) {
    const float vs = __shfl_xor(min_vs, o, kGroup), mid = __shfl_xor(min_mid, o, kGroup);
    const float a = __shfl_xor(z0, o, kGroup), c = __shfl_xor(z1, o, kGroup);
    const int vi = __shfl_xor(min_idx, o, kGroup), at = __shfl_xor(min_at, o, kGroup);
    const bool take = vi >= 0 && (min_idx < 0 || vs < min_vs ||
                                  (vs == min_vs && (mid < min_mid ||
                                                    (mid == min_mid && at < min_at))));
    if (take) {
      min_vs = vs;
      min_mid = mid;
      z0 = a;
      z1 = c;
      min_idx = vi;
      min_at = at;
    }
  }
  const int n_new = S - cnt;
  const float off = (z1 - z0) / (float)(n_new + 1);
  for (int i = cnt + grp.sub; i < S; i += kGroup) {
    float z = -1.0f;
    if (min_idx >= 0) {
      const float basic = z0 + off * (float)(i - cnt + 1);
      const float u = rnd[i];
      z = (float)((double)basic - (double)off / 2.0 + (double)(off * u));
    }
    ot[i] = z;
    oi[i] = min_idx;
  }
}

// Interpolation weights of the point ori + dir * t in node p (corners at
// centre +- size / 2; corner id 4 x + 2 y + z): tx, and ty / tz from the
// mean corner coordinates in double (sampling_kernel.cu:216-227).
__device__ __forceinline__ void tri_weights(float4 p, const float* __restrict__ o,
                                            const float* __restrict__ d, float t, float& tx,
                                            float& ty, float& tz) {
  const float px = o[0] + d[0] * t, py = o[1] + d[1] * t, pz = o[2] + d[2] * t;
  const float h_lo = ((float)(-1) * p.w) / 2.0f, h_hi = ((float)(1) * p.w) / 2.0f;
  const float xl = p.x + h_lo, xh = p.x + h_hi;
  const float yl = p.y + h_lo, yh = p.y + h_hi;
  const float zl = p.z + h_lo, zh = p.z + h_hi;
  tx = (px - xl) / (xh - xl);
  const double ym = (double)(yl + yl) / 2.0, yp = (double)(yh + yh) / 2.0;
  ty = (float)(((double)py - ym) / (yp - ym));
  const double zm = (double)(((zl + zl) + zl) + zl) / 4.0;
  const double zp = (double)(((zh + zh) + zh) + zh) / 4.0;
  tz = (float)(((double)pz - zm) / (zp - zm));
}

__device__ __forceinline__ float lerp1(float a, float b, float t) { return a * (1 - t) + b * t; }

// One thread per sample (b, r, s), looping over the C channels: the 8
// corner values of a channel are one 32-byte read, consecutive samples are
// consecutive in every channel plane.
__global__ void __launch_bounds__(kThreads)
trilinear_fwd_kernel(const float4* __restrict__ node_pos, int n_nodes,
                     const float* __restrict__ ray_ori, const float* __restrict__ ray_dir,
                     const int* __restrict__ sidx, const float* __restrict__ st,
                     const float4* __restrict__ feats, int B, int R, int S, int C,
                     float* __restrict__ out) {
  const long long RS = (long long)R * S;
  const long long total = (long long)B * RS;
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < total;
       k += (long long)gridDim.x * blockDim.x) {
    const long long b = k / RS, rs = k - b * RS, r = rs / S;
    const int vi = sidx[k];
    const bool ok = vi >= 0 && vi < n_nodes;
    float tx = 0.0f, ty = 0.0f, tz = 0.0f;
    if (ok) tri_weights(node_pos[vi], ray_ori + 3 * (b * R + r), ray_dir + 3 * (b * R + r), st[k],
                        tx, ty, tz);
    for (int c = 0; c < C; ++c) {
      const long long oi = (b * C + c) * RS + rs;
      float v = 0.0f;
      if (ok) {
        const float4 lo = feats[2 * oi], hi = feats[2 * oi + 1];
        const float x04 = lerp1(lo.x, hi.x, tx), x15 = lerp1(lo.y, hi.y, tx);
        const float x26 = lerp1(lo.z, hi.z, tx), x37 = lerp1(lo.w, hi.w, tx);
        const float y0 = lerp1(x04, x26, ty), y1 = lerp1(x15, x37, ty);
        v = lerp1(y0, y1, tz);
      }
      out[oi] = v;
    }
  }
}

__global__ void __launch_bounds__(kThreads)
trilinear_bwd_kernel(const float4* __restrict__ node_pos, int n_nodes,
                     const float* __restrict__ ray_ori, const float* __restrict__ ray_dir,
                     const int* __restrict__ sidx, const float* __restrict__ st,
                     const float* __restrict__ grad, int B, int R, int S, int C,
                     float4* __restrict__ grad_feats) {
  const long long RS = (long long)R * S;
  const long long total = (long long)B * RS;
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < total;
       k += (long long)gridDim.x * blockDim.x) {
    const long long b = k / RS, rs = k - b * RS, r = rs / S;
    const int vi = sidx[k];
    const bool ok = vi >= 0 && vi < n_nodes;
    float w[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (ok) {
      float tx, ty, tz;
      tri_weights(node_pos[vi], ray_ori + 3 * (b * R + r), ray_dir + 3 * (b * R + r), st[k], tx,
                  ty, tz);
      // sampling_kernel.cu:293-316
      const float z1 = tz, z0 = 1 - tz, y26 = ty, y04 = 1 - ty, y37 = ty, y15 = 1 - ty;
      const float x4 = tx, x0 = 1 - tx, x6 = tx, x2 = 1 - tx, x5 = tx, x1 = 1 - tx, x7 = tx,
                  x3 = 1 - tx;
      w[0] = x0 * y04 * z0;
      w[1] = x1 * y15 * z1;
      w[2] = x2 * y26 * z0;
      w[3] = x3 * y37 * z1;
      w[4] = x4 * y04 * z0;
      w[5] = x5 * y15 * z1;
      w[6] = x6 * y26 * z0;
      w[7] = x7 * y37 * z1;
    }
    for (int c = 0; c < C; ++c) {
      const long long gi = (b * C + c) * RS + rs;
      float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
      if (ok) {
        const float g = grad[gi];
        lo = make_float4(g * w[0], g * w[1], g * w[2], g * w[3]);
        hi = make_float4(g * w[4], g * w[5], g * w[6], g * w[7]);
      }
      grad_feats[2 * gi] = lo;
      grad_feats[2 * gi + 1] = hi;
    }
  }
}

// project_xyz (sampling_kernel.cu:55-157): one thread per (batch, view,
// ray, sample); the point ori + dir * t (and with corners, the node's 8
// corners, id 4 x + 2 y + z) through [R | T] and K, divided by the third
// coordinate and mapped to [-1, 1] as (p - w / 2.0) / (w / 2.0) in double.
// Samples with index -1 keep the -1 fill.
__global__ void __launch_bounds__(kThreads)
project_kernel(const float4* __restrict__ node_pos, int n_nodes,
               const float* __restrict__ ray_ori, const float* __restrict__ ray_dir,
               const float* __restrict__ Ks, const float* __restrict__ RTs,
               const int* __restrict__ sidx, const float* __restrict__ st, int B, int V, int R,
               int S, int ori_w, int ori_h, int corners, float* __restrict__ xy,
               float* __restrict__ z) {
  const long long total = (long long)B * V * R * S;
  const int np_ = corners ? 9 : 1;
  for (long long k = (long long)blockIdx.x * blockDim.x + threadIdx.x; k < total;
       k += (long long)gridDim.x * blockDim.x) {
    const long long rs = k % ((long long)R * S);
    const long long bv = k / ((long long)R * S);
    const long long b = bv / V;
    const long long r = rs / S;
    const long long si = b * R * S + rs;
    const int vi = sidx[si];
    if (vi == -1) continue;
    const float* RT = RTs + bv * 12;
    const float* K = Ks + bv * 9;
    const float* o = ray_ori + (b * R + r) * 3;
    const float* d = ray_dir + (b * R + r) * 3;
    const float t = st[si];
    const float pt[3] = {o[0] + d[0] * t, o[1] + d[1] * t, o[2] + d[2] * t};
    const float4 nd = (vi >= 0 && vi < n_nodes) ? node_pos[vi] : make_float4(0.f, 0.f, 0.f, 0.f);
    const bool corner_ok = corners && vi >= 0 && vi < n_nodes;
    const double hw = (double)ori_w / 2.0, hh = (double)ori_h / 2.0;
    for (int c = 0; c < np_; ++c) {
      float q[3];
      if (c == 0) {
        q[0] = pt[0];
        q[1] = pt[1];
        q[2] = pt[2];
      } else {
        if (!corner_ok) break;
        const int id = c - 1;
        q[0] = nd.x + ((float)((id >> 2) & 1 ? 1 : -1) * nd.w) / 2.0f;
        q[1] = nd.y + ((float)((id >> 1) & 1 ? 1 : -1) * nd.w) / 2.0f;
        q[2] = nd.z + ((float)(id & 1 ? 1 : -1) * nd.w) / 2.0f;
      }
      const float cx = RT[0] * q[0] + RT[1] * q[1] + RT[2] * q[2] + RT[3];
      const float cy = RT[4] * q[0] + RT[5] * q[1] + RT[6] * q[2] + RT[7];
      const float cz = RT[8] * q[0] + RT[9] * q[1] + RT[10] * q[2] + RT[11];
      float px = K[0] * cx + K[1] * cy + K[2] * cz;
      float py = K[3] * cx + K[4] * cy + K[5] * cz;
      const float pz = K[6] * cx + K[7] * cy + K[8] * cz;
      px = px / pz;
      py = py / pz;
      const long long o2 = (k * np_ + c) * 2;
      xy[o2] = (float)(((double)px - hw) / hw);
      xy[o2 + 1] = (float)(((double)py - hh) / hh);
      z[k * np_ + c] = cz;
    }
  }
}

__global__ void fill_value(float* __restrict__ a, long long n, float v) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x)
    a[i] = v;
}

unsigned grid_of(long long work) {
  return (unsigned)std::max<long long>(
      1, std::min<long long>((work + kThreads - 1) / kThreads, 256 * 32));
}

}  // namespace

extern "C" int sailor_octree_traversal(
    const int32_t* vol_coarse, const float* node_pos, const int32_t* node_info, int n_nodes,
    const float* vol_bbox, const float* voxel_size, int B, int dim_fine, int dim_coarse,
    int rate, const float* ray_ori, const float* ray_dir, int R, int n_max_hits_coarse,
    int n_max_hits, int th_early_stop, int opt_num_intersected, int32_t* hit_idx_coarse,
    float* tmin_coarse, float* tmax_coarse, int32_t* hit_idx, float* tmin, float* tmax,
    float* valid_len, int32_t* status, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && n_max_hits_coarse > 0 && n_max_hits > 0,
                 "octree_traversal: bad sizes");
  SAILOR_REQUIRE(dim_coarse > 0 && rate >= 1 && n_nodes >= 0, "octree_traversal: bad tree dims");
  if (R == 0) return SAILOR_OK;
  hipStream_t st = sailor::as_stream(stream);
  // 8 and 4 lanes, us, rows of 128 + 128: rate 2 32,768 random rays 175 and 169,
  // 65,536 263 and 221, 1,048,576 2789 and 1858 (2 lanes 2140); rate 4 131,072
  // in raster order 321 and 360, random 437 and 318, 1,048,576 3244 and 1766;
  // rate 8 1,048,576 in raster order 1274 and 1310, random 3309 and 2447
  const long long rays = (long long)B * R;
  const int lanes = rate < 8 && rays >= (rate < 4 ? 1 << 16 : 1 << 18) ? 4 : kGroup;
  auto kern = octree_traversal_kernel<8>;
  if (lanes == 4) kern = octree_traversal_kernel<4>;
  return sailor::in_parts(rays, [&](long long first, long long n) {
    hipLaunchKernelGGL(kern, dim3(sailor::ceil_div(n, kWalkThreads / lanes)),
                       dim3(kWalkThreads), 0, st, vol_coarse,
                       reinterpret_cast<const float4*>(node_pos),
                       reinterpret_cast<const int4*>(node_info), n_nodes, vol_bbox, voxel_size,
                       first, first + n, dim_fine, dim_coarse, rate, ray_ori, ray_dir, R,
                       n_max_hits_coarse, n_max_hits, th_early_stop, opt_num_intersected,
                       hit_idx_coarse, tmin_coarse, tmax_coarse, hit_idx, tmin, tmax, valid_len,
                       status);
    return sailor::check_launch("octree_traversal");
  });
}

extern "C" int sailor_octree_sampling(const int32_t* hit_idx, const float* tmin,
                                      const float* tmax, const float* noise,
                                      const float* valid_len, const float* node_pos,
                                      int n_nodes, const float* voxel_size, int B, int R,
                                      int n_max_hits, int max_hits, int S, int start_scale,
                                      int32_t* sampled_idx, float* sampled_t, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && S > 0 && n_max_hits > 0 && n_nodes >= 0,
                 "ray_voxels_points_sampling: bad sizes");
  SAILOR_REQUIRE(max_hits >= 0 && max_hits <= n_max_hits,
                 "ray_voxels_points_sampling: max_hits %d outside [0, %d]", max_hits, n_max_hits);
  if (R == 0) return SAILOR_OK;
  return sailor::in_parts((long long)B * R, [&](long long first, long long n) {
    hipLaunchKernelGGL(adaptive_sampling_kernel,
                       dim3(sailor::ceil_div(n, kWalkThreads / kGroup)),
                       dim3(kWalkThreads), 0, sailor::as_stream(stream), hit_idx, tmin, tmax,
                       noise, valid_len, reinterpret_cast<const float4*>(node_pos), n_nodes,
                       voxel_size, first, first + n, R, n_max_hits, max_hits, S, start_scale,
                       sampled_idx, sampled_t);
    return sailor::check_launch("ray_voxels_points_sampling");
  });
}

extern "C" int sailor_trilinear_aggregate(const float* node_pos, int n_nodes,
                                          const float* ray_ori, const float* ray_dir,
                                          const int32_t* sampled_idx, const float* sampled_t,
                                          const float* feats, int B, int R, int S, int C,
                                          float* out, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && S > 0 && C > 0 && n_nodes >= 0,
                 "trilinear_aggregate_features: bad sizes");
  SAILOR_REQUIRE(((uintptr_t)feats & 15) == 0, "trilinear_aggregate_features: feats must be "
                 "16-byte aligned");
  if (R == 0) return SAILOR_OK;
  hipLaunchKernelGGL(trilinear_fwd_kernel, dim3(grid_of((long long)B * R * S)), dim3(kThreads),
                     0, sailor::as_stream(stream), reinterpret_cast<const float4*>(node_pos),
                     n_nodes, ray_ori, ray_dir, sampled_idx, sampled_t,
                     reinterpret_cast<const float4*>(feats), B, R, S, C, out);
  return sailor::check_launch("trilinear_aggregate_features");
}

extern "C" int sailor_trilinear_aggregate_backward(const float* node_pos, int n_nodes,
                                                   const float* ray_ori, const float* ray_dir,
                                                   const int32_t* sampled_idx,
                                                   const float* sampled_t,
                                                   const float* grad_out, int B, int R, int S,
                                                   int C, float* grad_feats, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && S > 0 && C > 0 && n_nodes >= 0,
                 "trilinear_aggregate_features_backward: bad sizes");
  SAILOR_REQUIRE(((uintptr_t)grad_feats & 15) == 0, "trilinear_aggregate_features_backward: "
                 "grad_feats must be 16-byte aligned");
  if (R == 0) return SAILOR_OK;
  hipLaunchKernelGGL(trilinear_bwd_kernel, dim3(grid_of((long long)B * R * S)), dim3(kThreads),
                     0, sailor::as_stream(stream), reinterpret_cast<const float4*>(node_pos),
                     n_nodes, ray_ori, ray_dir, sampled_idx, sampled_t, grad_out, B, R, S, C,
                     reinterpret_cast<float4*>(grad_feats));
  return sailor::check_launch("trilinear_aggregate_features_backward");
}

extern "C" int sailor_project_sampled_xyz(const float* node_pos, int n_nodes, const float* ray_ori,
                                          const float* ray_dir, const int32_t* sampled_idx,
                                          const float* sampled_t, const float* Ks,
                                          const float* RTs, int B, int V, int R, int S,
                                          int ori_w, int ori_h, int record_corners,
                                          float* proj_xy, float* proj_z, void* stream) {
  SAILOR_REQUIRE(B > 0 && V > 0 && R >= 0 && S > 0 && n_nodes >= 0 && ori_w > 0 && ori_h > 0,
                 "project_sampled_xyz: bad sizes");
  if (R == 0) return SAILOR_OK;
  hipStream_t st = sailor::as_stream(stream);
  const long long n = (long long)B * V * R * S * (record_corners ? 9 : 1);
  hipLaunchKernelGGL(fill_value, dim3(grid_of(2 * n)), dim3(kThreads), 0, st, proj_xy, 2 * n,
                     -1.0f);
  hipLaunchKernelGGL(fill_value, dim3(grid_of(n)), dim3(kThreads), 0, st, proj_z, n, -1.0f);
  if (int e = sailor::check_launch("project_sampled_xyz (fill)")) return e;
  hipLaunchKernelGGL(project_kernel, dim3(grid_of((long long)B * V * R * S)), dim3(kThreads), 0,
                     st, reinterpret_cast<const float4*>(node_pos), n_nodes, ray_ori, ray_dir,
                     Ks, RTs, sampled_idx, sampled_t, B, V, R, S, ori_w, ori_h,
                     record_corners ? 1 : 0, proj_xy, proj_z);
  return sailor::check_launch("project_sampled_xyz");
}
