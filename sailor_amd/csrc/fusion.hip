// TSDF fusion: adaptive bounding box + projective TSDF integration.
//
// Follows c_lib/VoxelEncoding/src/fusion_kernel.cu (integrate_cuda :236-340,
// obtain_origin_bbox :137-184, obtain_resized_bbox :51-103, inverse_mat3x3
// :105-135).  Compiled with -ffp-contract=off: every arithmetic expression is
// evaluated as written (one rounding per operation), which is what makes the
// occupied-voxel list reproducible bit for bit by the CPU oracle.
//
// MI355X mapping
//  * bbox: one pass over the depth maps; each workgroup reduces its pixels in
//    registers / LDS and issues 6 integer atomics (order-preserving float keys)
//    instead of one CAS loop per pixel and bound.
//  * integrate: one lane per voxel, a wave per 4 x 4 x 16 brick, z fastest, so
//    the 16 B/voxel of output (tsdf, weight, colour, occupancy) is written in
//    64-byte runs; views that cannot observe a brick are skipped, by its
//    projection and a table of the views' deepest usable depth per 16^2 pixel
//    tile; the occupied count is aggregated with wave ballots and one atomic
//    per workgroup.
#include "common.h"

namespace {

constexpr int kThreads = 256;
constexpr int kMaxViews = 64;

// 3x3 inverse by adjugate / determinant, same expression order as the
// reference (fusion_kernel.cu:115-133).
__device__ __forceinline__ void inverse3x3(const float* M, float* out) {
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

__global__ void bbox_init_keys(int* keys, int B) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= B * 6) return;
  // [B,3,2]: (min, max) per axis; initial values of the reference (:655-656)
  keys[i] = (i & 1) ? sailor::fkey(-99999.0f) : sailor::fkey(99999.0f);
}

// Back-projects every valid pixel (0.1 m < d <= 5 m) and reduces min/max of
// (p - th) / (p + th) per batch.  grid = (blocks, B).
__global__ void __launch_bounds__(kThreads)
bbox_reduce(const float* __restrict__ depths, const float* __restrict__ K,
            const float* __restrict__ R, const float* __restrict__ T, int V,
            int H, int W, float thres, int* keys) {
  __shared__ float s_inv[kMaxViews * 18];
  __shared__ float s_red[6][kThreads / 64];
  const int b = blockIdx.y;
  for (int v = threadIdx.x; v < V; v += blockDim.x) {
    inverse3x3(K + ((size_t)b * V + v) * 9, s_inv + v * 18);
    inverse3x3(R + ((size_t)b * V + v) * 9, s_inv + v * 18 + 9);
  }
  __syncthreads();

  float lo[3] = {3.0e38f, 3.0e38f, 3.0e38f};
  float hi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
  const long long HW = (long long)H * W;
  const long long n = (long long)V * HW;
  const float* dep = depths + (size_t)b * n;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    float d = dep[i];
    if (d < 0.1f || d > 5.0f) continue;
    int v = (int)(i / HW);
    long long r = i - (long long)v * HW;
    int py = (int)(r / W);
    int px = (int)(r - (long long)py * W);
    const float* ki = s_inv + v * 18;
    const float* ri = ki + 9;
    const float* t = T + ((size_t)b * V + v) * 3;
    float fx = (float)px, fy = (float)py;
    float cx = (ki[0] * fx + ki[1] * fy + ki[2]) * d;
    float cy = (ki[3] * fx + ki[4] * fy + ki[5]) * d;
    float cz = (ki[6] * fx + ki[7] * fy + ki[8]) * d;
    cx -= t[0];
    cy -= t[1];
    cz -= t[2];
    float p[3];
    p[0] = ri[0] * cx + ri[1] * cy + ri[2] * cz;
    p[1] = ri[3] * cx + ri[4] * cy + ri[5] * cz;
    p[2] = ri[6] * cx + ri[7] * cy + ri[8] * cz;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      lo[a] = fminf(lo[a], p[a] - thres);
      hi[a] = fmaxf(hi[a], p[a] + thres);
    }
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    float l = sailor::wave_min_f(lo[a]);
    float h = sailor::wave_max_f(hi[a]);
    if (lane == 0) {
      s_red[2 * a][wid] = l;
      s_red[2 * a + 1][wid] = h;
    }
  }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int j = threadIdx.x;
    float acc = s_red[j][0];
    for (int w = 1; w < (int)(blockDim.x / 64); ++w)
      acc = (j & 1) ? fmaxf(acc, s_red[j][w]) : fminf(acc, s_red[j][w]);
    // Only contribute if this block saw a valid pixel.
    bool seen = (j & 1) ? (acc > -3.0e38f) : (acc < 3.0e38f);
    if (seen) {
      if (j & 1)
        atomicMax(keys + b * 6 + j, sailor::fkey(acc));
      else
        atomicMin(keys + b * 6 + j, sailor::fkey(acc));
    }
  }
}

// keys (stored in-place in vol_bbox) -> vol_origin, cubic vol_bbox, voxel_size
// (obtain_resized_bbox, fusion_kernel.cu:51-103).  One thread per batch.
__global__ void bbox_finalize(float* vol_bbox_keys, int B, int dim,
                              const float* fixed_bbox, float* vol_origin,
                              float* voxel_size) {
  int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  float o[6];
  if (fixed_bbox) {
    for (int j = 0; j < 6; ++j) o[j] = fixed_bbox[b * 6 + j];
  } else {
    const int* keys = reinterpret_cast<const int*>(vol_bbox_keys) + b * 6;
    for (int j = 0; j < 6; ++j) o[j] = sailor::fkey_inv(keys[j]);
  }
  for (int j = 0; j < 6; ++j) vol_origin[b * 6 + j] = o[j];
  if (fixed_bbox) {
    for (int j = 0; j < 6; ++j) vol_bbox_keys[b * 6 + j] = o[j];
    voxel_size[b] = (o[1] - o[0]) / (float)(dim - 1);
    return;
  }
  float x_min = o[0], x_max = o[1], y_min = o[2], y_max = o[3], z_min = o[4],
        z_max = o[5];
  float x_len = x_max - x_min, y_len = y_max - y_min, z_len = z_max - z_min;
  float max_len = fmaxf(x_len, fmaxf(y_len, z_len));
  // (a + b) / 2.0 in the reference is a double division of a float sum; the
  // halving is exact, so the float division below gives identical bits.
  float x_c = (x_min + x_max) / 2.0f, y_c = (y_min + y_max) / 2.0f,
        z_c = (z_min + z_max) / 2.0f;
  voxel_size[b] = max_len / (float)(dim - 1);
  float half = max_len / 2.0f;
  if (max_len == x_len) {
    y_min = y_c - half; y_max = y_c + half;
    z_min = z_c - half; z_max = z_c + half;
  } else if (max_len == y_len) {
    x_min = x_c - half; x_max = x_c + half;
    z_min = z_c - half; z_max = z_c + half;
  } else {
    x_min = x_c - half; x_max = x_c + half;
    y_min = y_c - half; y_max = y_c + half;
  }
  float* bb = vol_bbox_keys + b * 6;
  bb[0] = x_min; bb[1] = x_max; bb[2] = y_min;
  bb[3] = y_max; bb[4] = z_min; bb[5] = z_max;
}

__global__ void keys_to_float(float* buf, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  buf[i] = sailor::fkey_inv(reinterpret_cast<const int*>(buf)[i]);
}

// Largest depth of every kTile x kTile pixel tile that an integration may use
// (0.1 m <= d <= 4 m; a NaN, which passes those tests, as infinity), -1 where
// the tile has none.  grid = (ceil(tiles_x / 4), tiles_y, B * V): 4 tiles of a
// tile row per workgroup.
constexpr int kTile = 16;

__global__ void __launch_bounds__(kThreads)
depth_tiles_kernel(const float* __restrict__ depths, int H, int W, int tiles_x, int tiles_y,
                   float* __restrict__ tiles) {
  __shared__ float s_max[kThreads / 64][4];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const float* img = depths + (size_t)blockIdx.z * H * W;
  const int x = blockIdx.x * 64 + lane;
  float m = -1.0f;
  for (int r = wid; r < kTile; r += kThreads / 64) {
    const int y = blockIdx.y * kTile + r;
    if (x < W && y < H) {
      const float d = img[(size_t)y * W + x];
      if (!(d < 0.1f || d > 4.0f)) m = fmaxf(m, d != d ? __builtin_inff() : d);
    }
  }
#pragma unroll
  for (int o = 1; o < kTile; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if (lane % kTile == 0) s_max[wid][lane / kTile] = m;
  __syncthreads();
  if (threadIdx.x < 4) {
    for (int w = 0; w < kThreads / 64; ++w) m = w ? fmaxf(m, s_max[w][threadIdx.x])
                                                  : s_max[0][threadIdx.x];
    const int tx = blockIdx.x * 4 + threadIdx.x;
    if (tx < tiles_x) tiles[((size_t)blockIdx.z * tiles_y + blockIdx.y) * tiles_x + tx] = m;
  }
}

// Bricks of kBx x kBy x kBz voxels, z fastest: a wave integrates one, 64 voxels
// per pass.
constexpr int kBx = 4, kBy = 4, kBz = 16;
constexpr int kPassY = 64 / kBz;
constexpr int kPasses = kBx * kBy / kPassY;
static_assert(64 % kBz == 0 && kBy % kPassY == 0, "whole passes over the brick");

struct Bricks {
  unsigned ny, nz, n;
  __host__ __device__ Bricks(int X, int Y, int Z)
      : ny((Y + kBy - 1) / kBy), nz((Z + kBz - 1) / kBz),
        n((unsigned)((X + kBx - 1) / kBx) * ny * nz) {}
  __device__ void corner(unsigned brick, int& x, int& y, int& z) const {
    x = (int)(brick / (ny * nz)) * kBx;
    y = (int)(brick / nz % ny) * kBy;
    z = (int)(brick % nz) * kBz;
  }
};

// masks[b * bricks + i], bit k: view k may observe a voxel of brick i of volume
// b; every other view leaves all of the brick's voxels unchanged.  VP lanes (V
// rounded up to a power of two) per brick, a view each; grid = (.., B).  A lane
// projects the 8 corners of the brick's voxel centres: where all are in front
// of the camera, the brick's pixels lie within the corners' bounding box, taken
// 2 pixels wider than they can round, and an observation needs a depth of at
// least cz - trunc there (tiles).  Bounds that are not finite, and bricks that
// reach the camera plane, count as observed.
__global__ void __launch_bounds__(kThreads)
observing_views_kernel(const float* __restrict__ vol_bbox, const float* __restrict__ voxel_size,
                       const float* __restrict__ K, const float* __restrict__ RT,
                       const float* __restrict__ tiles, int tiles_x, int tiles_y, int V, int VP,
                       int H, int W, int X, int Y, int Z, float trunc_weight,
                       unsigned long long* __restrict__ masks) {
  const Bricks br(X, Y, Z);
  const int b = blockIdx.y, per = kThreads / VP;
  const int k = threadIdx.x & (VP - 1);
  const float vs = voxel_size[b], trunc = vs * trunc_weight;
  const float* bb = vol_bbox + b * 6;
  // whole groups of VP lanes stay together: the vote below is theirs
  for (unsigned brick = blockIdx.x * per + threadIdx.x / VP; brick < br.n;
       brick += gridDim.x * per) {
    bool seen = false;
    if (k < V) {
      int x0, y0, z0;
      br.corner(brick, x0, y0, z0);
      const float lo[3] = {bb[0] + (float)x0 * vs, bb[2] + (float)y0 * vs,
                           bb[4] + (float)z0 * vs};
      const float hi[3] = {bb[0] + (float)(min(x0 + kBx, X) - 1) * vs,
                           bb[2] + (float)(min(y0 + kBy, Y) - 1) * vs,
                           bb[4] + (float)(min(z0 + kBz, Z) - 1) * vs};
      const float* rt = RT + ((size_t)b * V + k) * 12;
      const float* kk = K + ((size_t)b * V + k) * 9;
      const float inf = __builtin_inff();
      float u0 = inf, u1 = -inf, v0 = inf, v1 = -inf, c0 = inf, c1 = -inf, p0 = inf;
      float ec = 0.0f, eu = 0.0f, ev = 0.0f;
      bool finite = true;
#pragma unroll
      for (int corner = 0; corner < 8; ++corner) {
        const float x = corner & 1 ? hi[0] : lo[0], y = corner & 2 ? hi[1] : lo[1],
                    z = corner & 4 ? hi[2] : lo[2];
        const float cx = rt[0] * x + rt[1] * y + rt[2] * z + rt[3];
        const float cy = rt[4] * x + rt[5] * y + rt[6] * z + rt[7];
        const float cz = rt[8] * x + rt[9] * y + rt[10] * z + rt[11];
        const float pz = kk[6] * cx + kk[7] * cy + kk[8] * cz;
        const float u = (kk[0] * cx + kk[1] * cy + kk[2] * cz) / pz;
        const float v = (kk[3] * cx + kk[4] * cy + kk[5] * cz) / pz;
        // 1e-6 of the sums of magnitudes bounds the rounding of 7 operations
        const float ax = fabsf(rt[0] * x) + fabsf(rt[1] * y) + fabsf(rt[2] * z) + fabsf(rt[3]);
        const float ay = fabsf(rt[4] * x) + fabsf(rt[5] * y) + fabsf(rt[6] * z) + fabsf(rt[7]);
        const float az = fabsf(rt[8] * x) + fabsf(rt[9] * y) + fabsf(rt[10] * z) + fabsf(rt[11]);
        const float ap = fabsf(kk[6]) * ax + fabsf(kk[7]) * ay + fabsf(kk[8]) * az;
        const float au = fabsf(kk[0]) * ax + fabsf(kk[1]) * ay + fabsf(kk[2]) * az;
        const float av = fabsf(kk[3]) * ax + fabsf(kk[4]) * ay + fabsf(kk[5]) * az;
        u0 = fminf(u0, u);
        u1 = fmaxf(u1, u);
        v0 = fminf(v0, v);
        v1 = fmaxf(v1, v);
        c0 = fminf(c0, cz);
        c1 = fmaxf(c1, cz);
        p0 = fminf(p0, pz - 1e-6f * ap);
        ec = fmaxf(ec, 1e-6f * az);
        eu = fmaxf(eu, 1e-6f * (au + fabsf(u) * ap));
        ev = fmaxf(ev, 1e-6f * (av + fabsf(v) * ap));
        finite = finite && fabsf(u) < 1e8f && fabsf(v) < 1e8f && au + av + ap + az < 1e12f;
      }
      if (!finite || !(p0 > 0.05f)) {
        seen = !(finite && c1 < -1e-3f - ec);   // cz < 0 throughout: never observed
      } else {
        const float ex = 2.0f + eu / p0, ey = 2.0f + ev / p0;
        u0 -= ex; u1 += ex; v0 -= ey; v1 += ey;
        if (u1 >= 0.0f && v1 >= 0.0f && u0 <= (float)W && v0 <= (float)H) {
          const int tx0 = (int)fmaxf(u0, 0.0f) / kTile, ty0 = (int)fmaxf(v0, 0.0f) / kTile;
          const int tx1 = min((int)fminf(u1, (float)W) / kTile, tiles_x - 1);
          const int ty1 = min((int)fminf(v1, (float)H) / kTile, tiles_y - 1);
          const float need = c0 - trunc - 1e-3f - ec;
          const float* tv = tiles + ((size_t)b * V + k) * tiles_x * tiles_y;
          seen = (tx1 - tx0 + 1) * (ty1 - ty0 + 1) > 512;   // wide: as observed
          for (int ty = ty0; ty <= ty1 && !seen; ++ty) {
            float m = -1.0f;
            for (int tx = tx0; tx <= tx1; ++tx) m = fmaxf(m, tv[(size_t)ty * tiles_x + tx]);
            seen = m >= 0.0f && !(m < need);
          }
        }
      }
    }
    unsigned long long m = __ballot(seen) >> ((threadIdx.x & 63) & ~(VP - 1));
    if (VP < 64) m &= (1ull << VP) - 1;
    if (k == 0) masks[(size_t)b * br.n + brick] = m;
  }
}

// One lane per voxel; a brick per wave, or SPLIT = 4 waves per brick with a
// pass each; grid = (ceil(bricks * SPLIT / 4), B).  masks: the views to evaluate
// for each brick (null: all of them).  Bound by vector issue where views remain
// (the reference's IEEE divisions, 7 per view and voxel) and by the 16 B written
// per voxel elsewhere: 256^3 voxels, 4 views of 1024^2 around one performer
// 290 us without the masks, 93 us with them and about 20 us to make them
// (0.27 GB written; bricks of 4 x 4 x 32 and 8^3 voxels -8 and +27 us, but at
// 128^3 the former costs 15 us more); masks made by one wave of each 512-voxel
// workgroup before its voxels: 156 us.  COMP (precision form): the TSDF is
// formed as the Kahan-compensated sum of obs_weight * dist over the observing
// views divided once by the weight sum, instead of the reference's running
// average (tsdf * w_old + obs_weight * dist) / w_new -- the same value in exact
// arithmetic, with one rounding of the sum instead of one per view.
template <bool COMP, int SPLIT>
__global__ void __launch_bounds__(kThreads)
integrate_kernel(float* __restrict__ tsdf_vol, float* __restrict__ weight_vol,
                 float* __restrict__ color_vol, int* __restrict__ occ_vol,
                 int* __restrict__ num_occ, const float* __restrict__ vol_bbox,
                 const float* __restrict__ K, const float* __restrict__ RT,
                 const float* __restrict__ colors,
                 const float* __restrict__ depths,
                 const float* __restrict__ voxel_size,
                 const unsigned long long* __restrict__ masks, float obs_weight, int H,
                 int W, int V, int X, int Y, int Z, float trunc_weight,
                 float th_low, float th_high) {
  static_assert(kPasses % SPLIT == 0, "whole passes per wave");
  constexpr int passes = kPasses / SPLIT;
  __shared__ int s_cnt[kThreads / 64];
  const Bricks br(X, Y, Z);
  const int b = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float vs = voxel_size[b];
  const float trunc = vs * trunc_weight;
  const float* bb = vol_bbox + b * 6;
  int count = 0;
  for (unsigned item = blockIdx.x * (kThreads / 64) + wid; item < br.n * SPLIT;
       item += gridDim.x * (kThreads / 64)) {
    const unsigned brick = item / SPLIT;
    const int pass0 = (int)(item % SPLIT) * passes;
    int x0, y0, z0;
    br.corner(brick, x0, y0, z0);
    unsigned long long views = V < 64 ? (1ull << V) - 1 : ~0ull;
    if (masks) views = masks[(size_t)b * br.n + brick];
    const int vz = z0 + lane % kBz;
#pragma unroll 1
    for (int pass = pass0; pass < pass0 + passes; ++pass) {
      const int vx = x0 + pass / (kBy / kPassY);
      const int vy = y0 + pass % (kBy / kPassY) * kPassY + lane / kBz;
      bool occupied = false;
      if (vx < X && vy < Y && vz < Z) {
        const int vid = (vx * Y + vy) * Z + vz;
        float pt_x = bb[0] + (float)vx * vs;
        float pt_y = bb[2] + (float)vy * vs;
        float pt_z = bb[4] + (float)vz * vs;
        float tsdf = 1.0f, w = 0.0f, col = 0.0f;
        float ksum = 0.0f, kcomp = 0.0f;  // COMP: sum of obs_weight * dist, lost low bits
        const size_t img = (size_t)H * W;
        for (unsigned long long left = views; left; left &= left - 1) {
          const int k = __ffsll((long long)left) - 1;
          const float* rt = RT + ((size_t)b * V + k) * 12;
          const float* kk = K + ((size_t)b * V + k) * 9;
          float cx = rt[0] * pt_x + rt[1] * pt_y + rt[2] * pt_z + rt[3];
          float cy = rt[4] * pt_x + rt[5] * pt_y + rt[6] * pt_z + rt[7];
          float cz = rt[8] * pt_x + rt[9] * pt_y + rt[10] * pt_z + rt[11];
          float px = kk[0] * cx + kk[1] * cy + kk[2] * cz;
          float py = kk[3] * cx + kk[4] * cy + kk[5] * cz;
          float pz = kk[6] * cx + kk[7] * cy + kk[8] * cz;
          px = px / pz;
          py = py / pz;
          int ix = sailor::sat_f2i(roundf(px));
          int iy = sailor::sat_f2i(roundf(py));
          if (ix < 0 || ix >= W || iy < 0 || iy >= H || cz < 0) continue;
          size_t pix = ((size_t)b * V + k) * img + (size_t)iy * W + ix;
          float d = depths[pix];
          if (d < 0.1f || d > 4.0f) continue;
          float diff = d - cz;
          if (diff < -trunc) continue;
          float dist = fminf(1.0f, diff / trunc);
          float w_old = w;
          float w_new = w_old + obs_weight;
          w = w_new;
          if constexpr (COMP) {
            const float y = obs_weight * dist - kcomp;
            const float t = ksum + y;
            kcomp = (t - ksum) - y;
            ksum = t;
          } else {
            tsdf = (tsdf * w_old + obs_weight * dist) / w_new;
          }
          // packed colour running average (fusion_kernel.cu:320-331)
          float old_b = floorf(col / 65536.0f);
          float old_g = floorf((col - old_b * 256.0f * 256.0f) / 256.0f);
          float old_r = col - old_b * 256.0f * 256.0f - old_g * 256.0f;
          float nc = colors[pix];
          float new_b = floorf(nc / 65536.0f);
          float new_g = floorf((nc - new_b * 256.0f * 256.0f) / 256.0f);
          float new_r = nc - new_b * 256.0f * 256.0f - new_g * 256.0f;
          new_b = fminf(roundf((old_b * w_old + obs_weight * new_b) / w_new), 255.0f);
          new_g = fminf(roundf((old_g * w_old + obs_weight * new_g) / w_new), 255.0f);
          new_r = fminf(roundf((old_r * w_old + obs_weight * new_r) / w_new), 255.0f);
          col = new_b * 256.0f * 256.0f + new_g * 256.0f + new_r;
        }
        if constexpr (COMP) {
          if (w > 0.0f) tsdf = (ksum - kcomp) / w;
        }
        occupied = tsdf < trunc * th_high && tsdf > -trunc * th_low;
        size_t o = (size_t)b * X * Y * Z + vid;
        tsdf_vol[o] = tsdf;
        weight_vol[o] = w;
        color_vol[o] = col;
        occ_vol[o] = occupied ? vid : -1;
      }
      count += __popcll(__ballot(occupied));
    }
  }
  // occupied count: ballots per wave, one atomic per workgroup
  if (lane == 0) s_cnt[wid] = count;
  __syncthreads();
  if (threadIdx.x == 0) {
    int c = 0;
    for (int i = 0; i < (int)(blockDim.x / 64); ++i) c += s_cnt[i];
    if (c) atomicAdd(num_occ + b, c);
  }
}

// Sum of the back-projected world points of the valid pixels (0.1 m <= d
// <= 4 m) and their count per batch (obtain_center_points,
// fusion_kernel.cu:186-233), with the same per-pixel arithmetic as the bbox
// pass.  The reference adds every point with float atomics (order-dependent
// low bits); here each workgroup sums its pixels in double and writes one
// partial [x, y, z, n]; center_finalize adds the partials in block order, so
// the result is reproducible and exact to float32 rounding of the double
// sum.  grid = (kCenterBlocks, B).
constexpr int kCenterBlocks = 256;

__global__ void __launch_bounds__(kThreads)
center_partials(const float* __restrict__ depths, const float* __restrict__ K,
                const float* __restrict__ R, const float* __restrict__ T, int V, int H, int W,
                double* __restrict__ partials) {
  __shared__ float s_inv[kMaxViews * 18];
  __shared__ double s_red[4][kThreads / 64];
  const int b = blockIdx.y;
  for (int v = threadIdx.x; v < V; v += blockDim.x) {
    inverse3x3(K + ((size_t)b * V + v) * 9, s_inv + v * 18);
    inverse3x3(R + ((size_t)b * V + v) * 9, s_inv + v * 18 + 9);
  }
  __syncthreads();
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  const long long HW = (long long)H * W;
  const long long n = (long long)V * HW;
  const float* dep = depths + (size_t)b * n;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (long long)gridDim.x * blockDim.x) {
    float d = dep[i];
    if (d < 0.1f || d > 4.0f) continue;
    int v = (int)(i / HW);
    long long r = i - (long long)v * HW;
    int py = (int)(r / W);
    int px = (int)(r - (long long)py * W);
    const float* ki = s_inv + v * 18;
    const float* ri = ki + 9;
    const float* t = T + ((size_t)b * V + v) * 3;
    float fx = (float)px, fy = (float)py;
    float cx = (ki[0] * fx + ki[1] * fy + ki[2]) * d;
    float cy = (ki[3] * fx + ki[4] * fy + ki[5]) * d;
    float cz = (ki[6] * fx + ki[7] * fy + ki[8]) * d;
    cx -= t[0];
    cy -= t[1];
    cz -= t[2];
    acc[0] += (double)(ri[0] * cx + ri[1] * cy + ri[2] * cz);
    acc[1] += (double)(ri[3] * cx + ri[4] * cy + ri[5] * cz);
    acc[2] += (double)(ri[6] * cx + ri[7] * cy + ri[8] * cz);
    acc[3] += 1.0;
  }
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    double x = acc[a];
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    if (lane == 0) s_red[a][wid] = x;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double x = 0.0;
    for (int w = 0; w < kThreads / 64; ++w) x += s_red[threadIdx.x][w];
    partials[((size_t)b * gridDim.x + blockIdx.x) * 4 + threadIdx.x] = x;
  }
}

__global__ void center_finalize(const double* __restrict__ partials, int B, int blocks,
                                float* __restrict__ center, float* __restrict__ num_pts) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= B) return;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < blocks; ++k)
    for (int a = 0; a < 4; ++a) acc[a] += partials[((size_t)b * blocks + k) * 4 + a];
  center[b * 3 + 0] = (float)acc[0];
  center[b * 3 + 1] = (float)acc[1];
  center[b * 3 + 2] = (float)acc[2];
  num_pts[b] = (float)acc[3];
}

int launch_bbox(const float* depths, const float* K, const float* R,
                const float* T, int B, int V, int H, int W, float th,
                int* keys, hipStream_t st) {
  hipLaunchKernelGGL(bbox_init_keys, dim3(sailor::ceil_div(B * 6, 64)),
                     dim3(64), 0, st, keys, B);
  long long n = (long long)V * H * W;
  int blocks = (int)std::min<long long>(2048, (n + kThreads - 1) / kThreads);
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(bbox_reduce, dim3(blocks, B), dim3(kThreads), 0, st,
                     depths, K, R, T, V, H, W, th, keys);
  return sailor::check_launch("bbox_reduce");
}

// Masks pay for their two kernels and a pass over the depth maps (about 10 us
// and the maps' bytes) where voxels x views are many: 4 views of 1024^2, with
// and without masks 74 and 69 us at 128^3, 79 and 90 us at 160^3, 143 and
// 229 us at 256^3; 8 of 512^2 82 and 80 us at 96^3, 87 and 91 us at 112^3; 1 of
// 512^2 59 and 61 us at 192^3; 4 of 1024^2 at 32^3 99 and 42 us (whole call).
bool use_masks(int V, int H, int W, int X, int Y, int Z) {
  return (double)X * Y * Z * V > (double)(1 << 23) + (double)V * H * W;
}
// Waves per brick: a wave's 4 passes one after another take V projections each,
// which a chip that is not full waits for; a full one gains from fewer, longer
// waves.  1 and 4 waves: 4 views of 1024^2 55 and 42 us at 32^3, 83 and 69 us at
// 128^3, 142 and 176 us at 256^3 (masks); 1 view of 64^2 14.7 and 12.9 us at
// 32^3, 14.8 and 16.1 us at 48^3, 30 and 36 us at 160^3; 20 of 256^2 122 and
// 81 us at 64^3, 425 and 481 us at 256^3.
unsigned brick_split(long long bricks, int V) {
  const long long few = V < 4 ? 256LL * V * V : std::min(4096LL * V, 32768LL);
  return bricks < few ? 4 : 1;
}

}  // namespace

// Workspace: a mask of views per brick, then the depth of each pixel tile.
extern "C" size_t sailor_integrate_workspace_bytes(int B, int V, int H, int W, int X, int Y,
                                                   int Z) {
  if (B <= 0 || V <= 0 || H <= 0 || W <= 0 || X <= 0 || Y <= 0 || Z <= 0) return 0;
  return (size_t)B * Bricks(X, Y, Z).n * sizeof(unsigned long long) +
         (size_t)B * V * ((H + kTile - 1) / kTile) * ((W + kTile - 1) / kTile) * sizeof(float);
}

namespace {

int integrate_impl(bool comp, int32_t* occ_vol, int32_t* num_occ, const float* K,
                   const float* RT, const float* R, const float* T, const float* colors,
                   const float* depths, int B, int V, int H, int W, int X, int Y, int Z,
                   float obs_weight, float th_bbox, float trunc_weight, float tsdf_th_low,
                   float tsdf_th_high, const float* fixed_bbox, float* tsdf, float* weight,
                   float* color, float* vol_origin, float* vol_bbox, float* voxel_size,
                   void* workspace, size_t workspace_bytes, void* stream) {
  SAILOR_REQUIRE(B > 0 && V > 0 && H > 0 && W > 0, "integrate: empty input");
  SAILOR_REQUIRE(V <= kMaxViews, "integrate: at most %d views", kMaxViews);
  SAILOR_REQUIRE(X > 1 && Y > 0 && Z > 0, "integrate: bad volume dims");
  SAILOR_REQUIRE((long long)X * Y * Z < (1LL << 31), "integrate: volume too large");
  hipStream_t st = sailor::as_stream(stream);
  int* keys = reinterpret_cast<int*>(vol_bbox);
  if (!fixed_bbox) {
    int rc = launch_bbox(depths, K, R, T, B, V, H, W, th_bbox, keys, st);
    if (rc) return rc;
  }
  hipLaunchKernelGGL(bbox_finalize, dim3(sailor::ceil_div(B, 64)), dim3(64), 0,
                     st, vol_bbox, B, X, fixed_bbox, vol_origin, voxel_size);
  const unsigned n = Bricks(X, Y, Z).n;
  const int tiles_x = sailor::ceil_div(W, kTile), tiles_y = sailor::ceil_div(H, kTile);
  // a launch holds fewer than 2^32 lanes: larger grids loop
  auto blocks = [](long long want) { return dim3((unsigned)std::min(want, 1LL << 23)); };
  unsigned long long* masks = nullptr;
  if (workspace != nullptr) {
    SAILOR_REQUIRE(workspace_bytes >= sailor_integrate_workspace_bytes(B, V, H, W, X, Y, Z),
                   "integrate: workspace of %zu bytes is smaller than the %zu required",
                   workspace_bytes, sailor_integrate_workspace_bytes(B, V, H, W, X, Y, Z));
    SAILOR_REQUIRE((reinterpret_cast<uintptr_t>(workspace) & 7) == 0,
                   "integrate: workspace must be 8-byte aligned");
    // the tiles' launch takes a grid plane per view and a row per tile row
    if (use_masks(V, H, W, X, Y, Z) && (long long)B * V <= 65535 && tiles_y <= 65535) {
      masks = static_cast<unsigned long long*>(workspace);
      float* tiles = reinterpret_cast<float*>(masks + (size_t)B * n);
      hipLaunchKernelGGL(depth_tiles_kernel, dim3(sailor::ceil_div(tiles_x, 4), tiles_y, B * V),
                         dim3(kThreads), 0, st, depths, H, W, tiles_x, tiles_y, tiles);
      int VP = 1;
      while (VP < V) VP *= 2;
      dim3 grid = blocks(((long long)n * VP + kThreads - 1) / kThreads);
      grid.y = B;
      hipLaunchKernelGGL(observing_views_kernel, grid, dim3(kThreads), 0, st, vol_bbox,
                         voxel_size, K, RT, tiles, tiles_x, tiles_y, V, VP, H, W, X, Y, Z,
                         trunc_weight, masks);
    }
  }
  const unsigned split = brick_split((long long)n * B, V);
  dim3 grid = blocks(((long long)n * split + kThreads / 64 - 1) / (kThreads / 64));
  grid.y = B;
  auto kern = integrate_kernel<false, 1>;
  if (split == 1 && comp) kern = integrate_kernel<true, 1>;
  if (split == 4) kern = integrate_kernel<false, 4>;
  if (split == 4 && comp) kern = integrate_kernel<true, 4>;
  hipLaunchKernelGGL(kern, grid, dim3(kThreads), 0, st, tsdf, weight, color, occ_vol, num_occ,
                     vol_bbox, K, RT, colors, depths, voxel_size, masks, obs_weight, H, W, V, X,
                     Y, Z, trunc_weight, tsdf_th_low, tsdf_th_high);
  return sailor::check_launch("integrate");
}

}  // namespace

extern "C" int sailor_integrate(
    int32_t* occ_vol, int32_t* num_occ, const float* K, const float* RT,
    const float* R, const float* T, const float* colors, const float* depths,
    const int32_t* masks, int B, int V, int H, int W, int X, int Y, int Z,
    float obs_weight, float th_bbox, float trunc_weight, float tsdf_th_low,
    float tsdf_th_high, const float* fixed_bbox, float* tsdf, float* weight,
    float* color, float* vol_origin, float* vol_bbox, float* voxel_size,
    void* stream) {
  (void)masks;  // read by nothing in the reference kernel either (:316-317)
  return integrate_impl(false, occ_vol, num_occ, K, RT, R, T, colors, depths, B, V, H, W, X, Y,
                        Z, obs_weight, th_bbox, trunc_weight, tsdf_th_low, tsdf_th_high,
                        fixed_bbox, tsdf, weight, color, vol_origin, vol_bbox, voxel_size,
                        nullptr, 0, stream);
}

extern "C" int sailor_integrate_compensated(
    int32_t* occ_vol, int32_t* num_occ, const float* K, const float* RT,
    const float* R, const float* T, const float* colors, const float* depths,
    const int32_t* masks, int B, int V, int H, int W, int X, int Y, int Z,
    float obs_weight, float th_bbox, float trunc_weight, float tsdf_th_low,
    float tsdf_th_high, const float* fixed_bbox, float* tsdf, float* weight,
    float* color, float* vol_origin, float* vol_bbox, float* voxel_size,
    void* stream) {
  (void)masks;
  return integrate_impl(true, occ_vol, num_occ, K, RT, R, T, colors, depths, B, V, H, W, X, Y,
                        Z, obs_weight, th_bbox, trunc_weight, tsdf_th_low, tsdf_th_high,
                        fixed_bbox, tsdf, weight, color, vol_origin, vol_bbox, voxel_size,
                        nullptr, 0, stream);
}

extern "C" int sailor_integrate_workspace(
    int compensated, int32_t* occ_vol, int32_t* num_occ, const float* K, const float* RT,
    const float* R, const float* T, const float* colors, const float* depths, int B, int V,
    int H, int W, int X, int Y, int Z, float obs_weight, float th_bbox, float trunc_weight,
    float tsdf_th_low, float tsdf_th_high, const float* fixed_bbox, float* tsdf, float* weight,
    float* color, float* vol_origin, float* vol_bbox, float* voxel_size, void* workspace,
    size_t workspace_bytes, void* stream) {
  SAILOR_REQUIRE(workspace != nullptr, "integrate: workspace missing");
  return integrate_impl(compensated != 0, occ_vol, num_occ, K, RT, R, T, colors, depths, B, V, H,
                        W, X, Y, Z, obs_weight, th_bbox, trunc_weight, tsdf_th_low,
                        tsdf_th_high, fixed_bbox, tsdf, weight, color, vol_origin, vol_bbox,
                        voxel_size, workspace, workspace_bytes, stream);
}

extern "C" int sailor_get_origin_bbox(const float* depths, const float* K,
                                      const float* R, const float* T, int B,
                                      int V, int H, int W, float th_bbox,
                                      float* vol_origin, void* stream) {
  SAILOR_REQUIRE(B > 0 && V > 0 && V <= kMaxViews, "get_origin_bbox: bad B/V");
  hipStream_t st = sailor::as_stream(stream);
  int rc = launch_bbox(depths, K, R, T, B, V, H, W, th_bbox,
                       reinterpret_cast<int*>(vol_origin), st);
  if (rc) return rc;
  hipLaunchKernelGGL(keys_to_float, dim3(sailor::ceil_div(B * 6, 64)), dim3(64),
                     0, st, vol_origin, B * 6);
  return sailor::check_launch("get_origin_bbox");
}

extern "C" int sailor_get_center_xyz(const float* depths, const float* K, const float* R,
                                     const float* T, int B, int V, int H, int W,
                                     float* vol_center, float* vol_num_pts, void* workspace,
                                     size_t workspace_bytes, void* stream) {
  SAILOR_REQUIRE(B > 0 && V > 0 && V <= kMaxViews && H > 0 && W > 0,
                 "get_center_xyz: bad sizes (B=%d, V=%d, H=%d, W=%d)", B, V, H, W);
  const size_t need = (size_t)B * kCenterBlocks * 4 * sizeof(double);
  SAILOR_REQUIRE(workspace_bytes >= need, "get_center_xyz: workspace too small (%zu < %zu)",
                 workspace_bytes, need);
  hipStream_t st = sailor::as_stream(stream);
  double* part = reinterpret_cast<double*>(workspace);
  hipLaunchKernelGGL(center_partials, dim3(kCenterBlocks, B), dim3(kThreads), 0, st, depths,
                     K, R, T, V, H, W, part);
  hipLaunchKernelGGL(center_finalize, dim3(sailor::ceil_div(B, 64)), dim3(64), 0, st, part, B,
                     kCenterBlocks, vol_center, vol_num_pts);
  return sailor::check_launch("get_center_xyz");
}
