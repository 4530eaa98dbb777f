// Device-side building blocks shared by the ray/voxel traversal kernels: the
// slab test, the coarse-grid DDA with per-node child expansion, and the
// length-weighted sampler.  Every expression keeps the reference's operation
// order; callers compile with -ffp-contract=off.
#pragma once

#include "common.h"

namespace sailor {

constexpr float kNoHit = -1.0f;
constexpr float kDdaFar = 9999999.0f;  // DBL_MAX macro of intersection_kernel.cu:16

// RayVoxelIntersection (intersection_kernel.cu:36-71) with inv = 1/d
// precomputed (IEEE division; the reference uses __fdividef).
__device__ __forceinline__ float2 slab_test(float3 o, float3 inv, float3 c,
                                            float size) {
  float lo = 0.0f, hi = 100000.f;
  const float half = size / 2.0f;
#define SAILOR_SLAB_AXIS(OA, IA, CA)                                  \
  {                                                                   \
    float t0 = (CA - half - OA) * IA;                                 \
    float t1 = (CA + half - OA) * IA;                                 \
    if (t0 > t1) { float tmp = t0; t0 = t1; t1 = tmp; }               \
    if (t1 < lo) return make_float2(kNoHit, kNoHit);                  \
    if (t0 > hi) return make_float2(kNoHit, kNoHit);                  \
    lo = (t0 > lo) ? t0 : lo;                                         \
    hi = (t1 < hi) ? t1 : hi;                                         \
    if (lo > hi) return make_float2(kNoHit, kNoHit);                  \
  }
  SAILOR_SLAB_AXIS(o.x, inv.x, c.x)
  SAILOR_SLAB_AXIS(o.y, inv.y, c.y)
  SAILOR_SLAB_AXIS(o.z, inv.z, c.z)
#undef SAILOR_SLAB_AXIS
  return make_float2(lo, hi);
}

struct RayCtx {
  const int* vc;          // coarse volume of this batch (node gindex or -1)
  const float4* np;       // node centre + size
  const int4* ni;         // node batch / parent / first child / #children
  int n_nodes;            // entries >= n_nodes are treated as empty
  float3 o, d, inv;
  float3 center;          // centre of the volume bbox
  float3 bst;             // bbox min - half a fine voxel
  float vs_top;           // coarse voxel size
  int dc;
  float rate;

  __device__ __forceinline__ void init(const int* vol_coarse, const float4* node_pos,
                                       const int4* node_info, int num_nodes,
                                       const float* vol_bbox,
                                       const float* voxel_size, int b, int dim_fine,
                                       int dim_coarse, int rate_i, const float* ori,
                                       const float* dir) {
    dc = dim_coarse;
    vc = vol_coarse + (size_t)b * dc * dc * dc;
    np = node_pos;
    ni = node_info;
    n_nodes = num_nodes;
    rate = (float)rate_i;
    const float* bb = vol_bbox + b * 6;
    center = make_float3((bb[0] + bb[1]) / 2.0f, (bb[2] + bb[3]) / 2.0f,
                         (bb[4] + bb[5]) / 2.0f);
    const float vs = voxel_size[b];
    vs_top = vs * (float)(dim_fine / dim_coarse);
    bst = make_float3(bb[0] - vs / 2.0f, bb[2] - vs / 2.0f, bb[4] - vs / 2.0f);
    o = make_float3(ori[0], ori[1], ori[2]);
    d = make_float3(dir[0], dir[1], dir[2]);
    inv = make_float3(1.0f / d.x, 1.0f / d.y, 1.0f / d.z);
  }
};

// Coarse-grid DDA of a ray (intersection_kernel.cu:128-439): the cell
// (x, y, z) and the ray parameters of the next x / y / z boundaries.
struct Dda {
  int x, y, z, ix, iy, iz;
  float tx, ty, tz, dtx, dty, dtz;
  // entry cell at ray parameter t_in (the volume's slab-test entry)
  __device__ __forceinline__ void start(const RayCtx& c, float t_in) {
    const float spx = c.o.x + t_in * c.d.x;
    const float spy = c.o.y + t_in * c.d.y;
    const float spz = c.o.z + t_in * c.d.z;
    const float sox = spx - c.bst.x, soy = spy - c.bst.y, soz = spz - c.bst.z;
    x = sat_f2i(sox / c.vs_top);
    y = sat_f2i(soy / c.vs_top);
    z = sat_f2i(soz / c.vs_top);
    x = x < 0 ? 0 : x;
    y = y < 0 ? 0 : y;
    z = z < 0 ? 0 : z;
    x = x < c.dc ? x : c.dc - 1;
    y = y < c.dc ? y : c.dc - 1;
    z = z < c.dc ? z : c.dc - 1;
    const float stx = (c.d.x >= 0) ? 1.f : -1.f;
    const float sty = (c.d.y >= 0) ? 1.f : -1.f;
    const float stz = (c.d.z >= 0) ? 1.f : -1.f;
    const float nbx = (stx > 0) ? ((float)x + stx) * c.vs_top : (float)x * c.vs_top;
    const float nby = (sty > 0) ? ((float)y + sty) * c.vs_top : (float)y * c.vs_top;
    const float nbz = (stz > 0) ? ((float)z + stz) * c.vs_top : (float)z * c.vs_top;
    tx = (c.d.x != 0) ? (nbx - sox) / c.d.x : kDdaFar;
    ty = (c.d.y != 0) ? (nby - soy) / c.d.y : kDdaFar;
    tz = (c.d.z != 0) ? (nbz - soz) / c.d.z : kDdaFar;
    dtx = (c.d.x != 0) ? c.vs_top / c.d.x * stx : kDdaFar;
    dty = (c.d.y != 0) ? c.vs_top / c.d.y * sty : kDdaFar;
    dtz = (c.d.z != 0) ? c.vs_top / c.d.z * stz : kDdaFar;
    ix = (int)stx;
    iy = (int)sty;
    iz = (int)stz;
  }
  __device__ __forceinline__ int cell(int dc) const { return (x * dc + y) * dc + z; }
  // one step; false once the cell leaves the grid
  __device__ __forceinline__ bool advance(int dc) {
    if (tx < ty) {
      if (tx < tz) { x += ix; tx += dtx; }
      else { z += iz; tz += dtz; }
    } else {
      if (ty < tz) { y += iy; ty += dty; }
      else { z += iz; tz += dtz; }
    }
    return !(x < 0 || x >= dc || y < 0 || y >= dc || z < 0 || z >= dc);
  }
};

// ---- Lane groups -----------------------------------------------------------
// G lanes walk a ray together: all of them run the same DDA, and a coarse
// node's children (up to rate^3 records, contiguous in the node array) are
// tested G at a time, so a test is one coalesced load and one slab test instead
// of a serial chain of them.  8 lanes: a wave is as long as the longest of 8
// rays instead of 64, a launch has 8 times the waves to hide the chain's loads
// behind, and the DDA that all lanes repeat is still cheap (a wave per ray
// spends its time there).  Calls with more rays than the chip holds waves for,
// and few children per node to share, take fewer (rules at the entry points).
constexpr int kGroup = 8;
constexpr int kChildBatch = 2;   // children per lane loaded together (4: the same)

template <int G>
struct LaneGroup {
  static constexpr int size = G;
  int sub, base;   // lane within the group, first lane of the group in its wave
  __device__ __forceinline__ LaneGroup() {
    const int lane = threadIdx.x & 63;
    sub = lane % G;
    base = lane - sub;
  }
  // the group's lanes for which p holds, bit i = lane i
  __device__ __forceinline__ unsigned vote(bool p) const {
    return (unsigned)(__ballot(p) >> base) & ((1u << G) - 1);
  }
  __device__ __forceinline__ float from(float x, int i) const { return __shfl(x, i, G); }
  __device__ __forceinline__ int from(int x, int i) const { return __shfl(x, i, G); }
  __device__ __forceinline__ int before(unsigned votes) const {
    return __popc(votes & ((1u << sub) - 1));
  }
  __device__ __forceinline__ int inclusive_sum(int x) const {
#pragma unroll
    for (int o = 1; o < G; o <<= 1) {
      const int y = __shfl_up(x, o, G);
      if (sub >= o) x += y;
    }
    return x;
  }
};

// LDS written by some lanes of a wave and read by others of it: the LDS
// serves a wave in order, only the compiler has to keep it.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Words [from, n) of a row set to v by the whole wave, 16 bytes a lane where
// the row allows it.
__device__ __forceinline__ void fill_row(unsigned* row, int from, int n, unsigned v, int lane) {
  const int head = min(n, from + (int)(((16 - ((uintptr_t)(row + from) & 15)) & 15) / 4));
  if (from + lane < head) row[from + lane] = v;
  const int quads = (n - head) / 4;
  for (int q = lane; q < quads; q += 64)
    reinterpret_cast<uint4*>(row + head)[q] = make_uint4(v, v, v, v);
  const int tail = head + 4 * quads;
  if (tail + lane < n) row[tail + lane] = v;
}

// Sink interface (every lane of the group makes the same calls):
// put(pos, node, t0, t1) receives hit number `pos`; put_lanes(pos, node, t0,
// t1, hit, votes) the hits of up to G children, one per lane in order,
// the first of them number `pos`; stop() is polled after every coarse cell
// and may end the walk early (used once all samples are placed; never changes
// hits that were already emitted).
//
// Returns the number of hits; *vl_out receives the weighted valid length
// (children weighted by `rate`, the coarse interval by 1).
template <int G, class Sink>
__device__ __forceinline__ int traverse(const RayCtx& c, const LaneGroup<G>& grp,
                                        int th_early_stop, bool training, int opt_num,
                                        Sink& sink, float* vl_out) {
  float vl = 0.0f;
  int count = 0;
  float2 dep = slab_test(c.o, c.inv, c.center, c.vs_top * (float)c.dc);
  if (dep.x < 0.0f || dep.y < 0.0f) {
    *vl_out = vl;
    return 0;
  }
  Dda g;
  g.start(c, dep.x);
  const int J = 4 * c.dc;
  bool pre_empty = false, has_valid = false;
  int n_succ_empty = 0, n_inter = 0;
  // The DDA's path depends on the ray alone, so the coarse-volume entry of
  // the next cell is loaded while the current cell is visited.
  int node_next = c.vc[g.cell(c.dc)];
  for (int j = 0; j < J; ++j) {
    // ---- visit coarse cell (x, y, z): RayVoxelIntersectionNodeListNew
    int rid = -1;
    const int node = node_next;
    Dda nx = g;   // the cell after this one (the step below)
    const bool next_in = nx.advance(c.dc);
    if (next_in && j + 1 < J) node_next = c.vc[nx.cell(c.dc)];
    if (node > -1 && node < c.n_nodes) {
      // the node's record and its info are loaded together (the info is
      // used only when the slab test hits, which it nearly always does for
      // a cell the DDA visits)
      const float4 p = c.np[node];
      const int4 info = c.ni[node];
      const float2 vd = slab_test(c.o, c.inv, make_float3(p.x, p.y, p.z), p.w);
      if (!(vd.x < 0 || vd.y < 0)) {
        if (info.x >= 0) {
          int r = count;
          if (!training && info.z >= 0) {
            const int ch_end = min(info.z + info.w, c.n_nodes);
            // the records of up to kChildBatch children per lane are loaded
            // together: a round of loads tests 2 G children
            for (int ch0 = info.z; ch0 < ch_end; ch0 += G * kChildBatch) {
              float4 q[kChildBatch];
#pragma unroll
              for (int u = 0; u < kChildBatch; ++u) {
                const int ch = ch0 + u * G + grp.sub;
                q[u] = c.np[ch < ch_end ? ch : ch_end - 1];
              }
#pragma unroll
              for (int u = 0; u < kChildBatch; ++u) {
                const int ch = ch0 + u * G + grp.sub;
                const float2 cd =
                    slab_test(c.o, c.inv, make_float3(q[u].x, q[u].y, q[u].z), q[u].w);
                const bool hit = ch < ch_end && !(cd.x < 0 || cd.y < 0);
                unsigned votes = grp.vote(hit);
                if (votes == 0) continue;
                sink.put_lanes(r, ch, cd.x, cd.y, hit, votes);
                r += __popc(votes);
                // float += double in the reference (:252): one rounding of the
                // exact double sum, in hit order
                const float len = cd.y - cd.x;
                do {
                  const int i = __ffs(votes) - 1;
                  votes &= votes - 1;
                  vl = (float)((double)vl + (double)grp.from(len, i) * (double)c.rate);
                } while (votes);
              }
            }
          }
          sink.put(r, node, vd.x, vd.y);
          vl += vd.y - vd.x;
          ++r;
          count = r;
          rid = r - 1;
        }
      }
    }
    // ---- early termination options (intersection_kernel.cu:407-423)
    if (th_early_stop > -1) {
      if (rid == -1) {
        if (pre_empty && has_valid) n_succ_empty++;
        pre_empty = true;
      } else {
        n_succ_empty = 0;
        pre_empty = false;
        has_valid = true;
      }
      if ((n_succ_empty + 1) >= th_early_stop) break;
    }
    if (opt_num > -1) {
      if (rid + 1 > 0) n_inter++;
      if (n_inter >= opt_num) break;
    }
    if (sink.stop()) break;
    // ---- DDA step (computed above)
    g = nx;
    if (!next_in) break;
  }
  *vl_out = vl;
  return count;
}

// Length-weighted per-interval sampling (sampling_kernel.cu:1125-1174) of one
// row by a lane group: G hits at a time, one per lane in hit order.
struct SampleRow {
  float valid_len, start_vs;
  int S;
  const float* nz;   // the row's noise
  int* oi;           // the row's outputs
  float* ot;
  int has;           // slots used
  __device__ __forceinline__ void init(float vl, float svs, int s, const float* noise,
                                       int* out_idx, float* out_t) {
    valid_len = vl;
    start_vs = svs;
    S = s;
    nz = noise;
    oi = out_idx;
    ot = out_t;
    has = 0;
  }
  // Sample j (0-based) of an interval that receives n samples; r = noise.
  __device__ __forceinline__ static float sample_z(float mn, float mx, int n, int j,
                                                   float r) {
    const float off = (mx - mn) / (float)(n + 1);
    const float base = mn + off * (float)(j + 1);
    return (float)((double)base - (double)off / 2.0 + (double)(off * r));
  }
  __device__ __forceinline__ static float leftover_z(float mn, float mx, float r) {
    const float off = (float)((double)(mx - mn) / 2.0);
    const float base = mn + off;
    return (float)((double)base - (double)off / 2.0 + (double)(off * r));
  }
  // Places the samples of this lane's interval (mn, mx) of node v, size cvs:
  // as many as its share of the valid length, at least one, at most what the
  // intervals before it left.
  template <int G>
  __device__ __forceinline__ void intervals(const LaneGroup<G>& grp, bool on, int v, float mn,
                                            float mx, float cvs) {
    int want = 0;
    if (on) {
      const float rate = start_vs / cvs;
      want = sat_f2i((mx - mn) * rate * (float)S / valid_len);
      want = want >= 1 ? want : 1;
      want = want < S ? want : S;
    }
    const int end = grp.inclusive_sum(want);
    int slot = has + end - want;
    slot = slot < S ? slot : S;
    const int n = min(want, S - slot);
    // the noise of several samples is loaded before the first is stored (the
    // compiler cannot tell that the stores leave it alone)
    constexpr int kAhead = 4;
    for (int j0 = 0; j0 < n; j0 += kAhead) {
      float r[kAhead];
#pragma unroll
      for (int j = 0; j < kAhead; ++j) r[j] = nz[slot + min(j0 + j, n - 1)];
#pragma unroll
      for (int j = 0; j < kAhead; ++j)
        if (j0 + j < n) {
          ot[slot + j0 + j] = sample_z(mn, mx, n, j0 + j, r[j]);
          oi[slot + j0 + j] = v;
        }
    }
    has = min(S, has + grp.from(end, G - 1));
  }
  // One midpoint sample of a hit into `slot`.
  __device__ __forceinline__ void leftover(int slot, int v, float mn, float mx) {
    ot[slot] = leftover_z(mn, mx, nz[slot]);
    oi[slot] = v;
  }
};

}  // namespace sailor
