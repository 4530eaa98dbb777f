// Per-view sample features for the FastNerf inference surface: the chain
// proj_persp -> z_normalizer -> 4 x grid_sample -> t-psdf that the reference
// runs as separate PyTorch ops before InferNerf.infer_nerf
// (gui/gui_render.py:713-751, SRONet/BasicRenNet.py:245-259,296-311,
// utils_render/utils_render.py:380-410,656-663), fused into one pass:
// channels-last maps so a bilinear tap of the 16 feature channels is one
// 64-byte read, outputs written in the
// (batch, view, ray, sample) order infer_nerf consumes.
#include "image_sample.h"

namespace {

constexpr int kGeoC = 16, kRgbC = 16;
using sailor::bilinear_cl;

struct GatherArgs {
  const float* rays;   // [B,R,6]
  const float* dists;  // [B,R,S]
  const float* K;      // [B,V,3,3]
  const float* RT;     // [B,V,3,4]
  const float* geo;    // [B,V,Hg,Wg,16]
  const float* depth;  // [B,V,Hd,Wd]
  const float* rgbf;   // [B,V,Hr,Wr,16]
  const float* rgb;    // [B,V,Hc,Wc,3]
  const float* mid;    // [B,V]
  const float* dist;   // [B,V]
  int B, R, S, V, Hg, Wg, Hd, Wd, Hr, Wr, Hc, Wc, res;
  float* out_z;        // [B,V,R,S]
  float* out_tpsdf;    // [B,V,R,S]
  float* out_geo;      // [B,V,R,S,16]
  float* out_rgbf;     // [B,V,R,S,16]
  float* out_rgb;      // [B,V,R,S,3]
  float* out_dir;      // [B,V,R,S,3]
};

__device__ const float4 kZeroTap = {0.0f, 0.0f, 0.0f, 0.0f};

// bilinear_cl's taps of a 16-channel map at (gx, gy), 4 channels of each from
// channel c0 on: the same sums, with taps outside the map read from a zero so
// that all loads are issued together.
__device__ __forceinline__ float4 bilinear_quarter(const float* __restrict__ map, int H, int W,
                                                   float gx, float gy, int c0) {
  const float ix = sailor::grid_to_pixel(gx, W);
  const float iy = sailor::grid_to_pixel(gy, H);
  const bool in = ix > -1.0f && ix < (float)W && iy > -1.0f && iy < (float)H;
  const float fx0 = floorf(ix), fy0 = floorf(iy);
  const int x0 = in ? (int)fx0 : -2, y0 = in ? (int)fy0 : -2;
  const float ax = ix - fx0, ay = iy - fy0;
  float4 v[4];
  float w[4];
#pragma unroll
  for (int tap = 0; tap < 4; ++tap) {
    const int xx = x0 + (tap & 1), yy = y0 + (tap >> 1);
    const bool ok = xx >= 0 && xx < W && yy >= 0 && yy < H;
    w[tap] = ok ? ((tap & 1) ? ax : 1.0f - ax) * ((tap >> 1) ? ay : 1.0f - ay) : 0.0f;
    v[tap] = *(ok ? reinterpret_cast<const float4*>(map + ((size_t)yy * W + xx) * 16 + c0)
                  : &kZeroTap);
  }
  float4 o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int tap = 0; tap < 4; ++tap) {
    o.x += w[tap] * v[tap].x;
    o.y += w[tap] * v[tap].y;
    o.z += w[tap] * v[tap].z;
    o.w += w[tap] * v[tap].w;
  }
  return o;
}

__device__ __forceinline__ void store_once(float* p, float4 q) {
  typedef float v4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(v4{q.x, q.y, q.z, q.w}, reinterpret_cast<v4*>(p));
}

// Orders a wave's LDS writes before its later reads.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A wave handles 64 consecutive (ray, sample) pairs of one (batch, view): a
// lane per pair projects it and samples the narrow maps, then in 4 rounds four
// lanes per pair take 4 channels each of the two 16-channel maps, so that a tap
// is one 64-byte row and a round stores 1 KB in a row; the 3-channel outputs go
// through LDS for the same reason.  grid = (.., B V), where the view's camera is
// uniform and the pair's index splits in 32 bits (2^32 pairs have no room for
// their outputs).  Bound by the 160 bytes written per pair, which do not fit a
// cache and are stored past it: 60000 rays x 48 samples x 4 views (1.9 GB)
// 567 us (3.4 TB/s); with ordinary stores 715 us, and 16 workgroups per compute
// unit instead of 64 cost 12 us.
__global__ void __launch_bounds__(256) sample_features_kernel(GatherArgs a) {
  __shared__ float s_out[4][6 * 64];   // a wave's rgb, directions
  const unsigned RS = (unsigned)a.R * (unsigned)a.S;
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int bv = blockIdx.y; bv < a.B * a.V; bv += gridDim.y) {
    const int b = bv / a.V;
    const float* Rm = a.RT + (size_t)bv * 12;
    const float* Km = a.K + (size_t)bv * 9;
    const float mid = a.mid[bv], half_dist = a.dist[bv] / 2.0f;
    const float* geo = a.geo + (size_t)bv * a.Hg * a.Wg * kGeoC;
    const float* rgbf = a.rgbf + (size_t)bv * a.Hr * a.Wr * kRgbC;
    const float half = (float)(a.res / 2);
    const size_t e0 = (size_t)bv * RS;
    for (unsigned long long i0 = (blockIdx.x * 4ull + wid) * 64; i0 < RS;
         i0 += gridDim.x * 256ull) {
      const unsigned i = (unsigned)i0 + lane;
      float gx = -2.0f, gy = -2.0f;
      float* out = s_out[wid];
      if (i0 + lane < RS) {
        const unsigned r = i / (unsigned)a.S;
        const size_t e = e0 + i;
        const float* ray = a.rays + ((size_t)b * a.R + r) * 6;
        const float t = a.dists[(size_t)b * RS + i];
        // rays_points = ray_ori + ray_dir * dist (gui_render.py:723)
        const float px = ray[0] + ray[3] * t, py = ray[1] + ray[4] * t, pz = ray[2] + ray[5] * t;
        // proj_persp (utils_render.py:380-410): pts = R p + T
        const float x = Rm[0] * px + Rm[1] * py + Rm[2] * pz + Rm[3];
        const float y = Rm[4] * px + Rm[5] * py + Rm[6] * pz + Rm[7];
        const float z = Rm[8] * px + Rm[9] * py + Rm[10] * pz + Rm[11];
        const bool invalid = z < 0.01f;
        const bool invalid_d = t < 0.1f || t > 4.0f;  // p_depths outside [min_d, max_d]
        const float zd = invalid ? 1.0f : z;
        const float xn = x / zd, yn = y / zd, zn = z / zd;
        gx = (Km[0] * xn + Km[1] * yn + Km[2] * zn - half) / half;
        gy = (Km[3] * xn + Km[4] * yn + Km[5] * zn - half) / half;
        if (invalid || invalid_d) gx = gy = -2.0f;
        const float proj_z = invalid_d ? -2.0f : z;
        // z_normalizer (utils_render.py:656-663)
        a.out_z[e] = (proj_z - mid) / half_dist;
        float dep[1];
        bilinear_cl<1>(a.depth + (size_t)bv * a.Hd * a.Wd, a.Hd, a.Wd, gx, gy, dep);
        // t-psdf (gui_render.py:737)
        a.out_tpsdf[e] = fminf(fmaxf(proj_z - dep[0], -0.01f), 0.01f) * (1.0f / 0.01f);
        float c3[3];
        bilinear_cl<3>(a.rgb + (size_t)bv * a.Hc * a.Wc * 3, a.Hc, a.Wc, gx, gy, c3);
        out[3 * lane + 0] = c3[0];
        out[3 * lane + 1] = c3[1];
        out[3 * lane + 2] = c3[2];
        // ray direction in camera v (R @ dir, BasicRenNet.py:118-131)
        out[192 + 3 * lane + 0] = Rm[0] * ray[3] + Rm[1] * ray[4] + Rm[2] * ray[5];
        out[192 + 3 * lane + 1] = Rm[4] * ray[3] + Rm[5] * ray[4] + Rm[6] * ray[5];
        out[192 + 3 * lane + 2] = Rm[8] * ray[3] + Rm[9] * ray[4] + Rm[10] * ray[5];
      }
      wave_lds_fence();
#pragma unroll
      for (int d = lane; d < 192; d += 64) {
        if (3 * i0 + d >= 3ull * RS) break;
        __builtin_nontemporal_store(out[d], a.out_rgb + (e0 + i0) * 3 + d);
        __builtin_nontemporal_store(out[192 + d], a.out_dir + (e0 + i0) * 3 + d);
      }
      wave_lds_fence();   // read before the next pairs' are written
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int from = 16 * k + (lane >> 2), c0 = 4 * (lane & 3);
        const float kx = __shfl(gx, from, 64), ky = __shfl(gy, from, 64);
        if (i0 + from >= RS) continue;
        const size_t e = e0 + i0 + from;
        store_once(a.out_geo + e * kGeoC + c0, bilinear_quarter(geo, a.Hg, a.Wg, kx, ky, c0));
        store_once(a.out_rgbf + e * kRgbC + c0, bilinear_quarter(rgbf, a.Hr, a.Wr, kx, ky, c0));
      }
    }
  }
}

// [N][C][H][W] -> [N][H][W][C]; one thread per pixel (coalesced plane reads
// and contiguous channel-block writes).
__global__ void __launch_bounds__(256) nchw_to_nhwc_kernel(const float* __restrict__ src, int N,
                                                           int C, int HW,
                                                           float* __restrict__ dst) {
  const long long total = (long long)N * HW;
  for (long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x; p < total;
       p += (long long)gridDim.x * blockDim.x) {
    const long long n = p / HW, i = p - n * HW;
    const float* s = src + n * C * HW + i;
    float* d = dst + p * C;
    for (int c = 0; c < C; ++c) d[c] = s[(long long)c * HW];
  }
}

unsigned grid_of(long long work) {
  return (unsigned)std::max<long long>(1, std::min<long long>((work + 255) / 256, 256 * 16));
}

}  // namespace

extern "C" int sailor_nchw_to_nhwc(const float* src, int N, int C, int H, int W, float* dst,
                                   void* stream) {
  SAILOR_REQUIRE(N >= 0 && C > 0 && H > 0 && W > 0, "nchw_to_nhwc: bad sizes");
  if (N == 0) return SAILOR_OK;
  hipLaunchKernelGGL(nchw_to_nhwc_kernel, dim3(grid_of((long long)N * H * W)), dim3(256), 0,
                     sailor::as_stream(stream), src, N, C, H * W, dst);
  return sailor::check_launch("nchw_to_nhwc");
}

extern "C" int sailor_sample_features(
    const float* rays, const float* dists, int B, int R, int S, const float* K, const float* RT,
    int V, const float* geo_cl, int Hg, int Wg, const float* depth, int Hd, int Wd,
    const float* rgbf_cl, int Hr, int Wr, const float* rgb_cl, int Hc, int Wc,
    const float* depth_mid, const float* depth_dist, int res, float* out_z, float* out_tpsdf,
    float* out_geo, float* out_rgbf, float* out_rgb, float* out_dir, void* stream) {
  SAILOR_REQUIRE(B > 0 && R >= 0 && S > 0 && V > 0, "sample_features: bad sizes");
  SAILOR_REQUIRE(Hg > 1 && Wg > 1 && Hd > 1 && Wd > 1 && Hr > 1 && Wr > 1 && Hc > 1 && Wc > 1,
                 "sample_features: maps must be at least 2 x 2");
  SAILOR_REQUIRE(res >= 2, "sample_features: res must be at least 2");
  if (R == 0) return SAILOR_OK;
  GatherArgs a{rays, dists, K, RT, geo_cl, depth, rgbf_cl, rgb_cl, depth_mid, depth_dist,
               B, R, S, V, Hg, Wg, Hd, Wd, Hr, Wr, Hc, Wc, res,
               out_z, out_tpsdf, out_geo, out_rgbf, out_rgb, out_dir};
  const unsigned gy = (unsigned)std::min<long long>((long long)B * V, 65535);
  // up to 64 workgroups per compute unit over all views
  const long long want = ((long long)R * S + 255) / 256;
  const unsigned gx = (unsigned)std::min<long long>(want, std::max(1u, 256 * 64 / gy));
  hipLaunchKernelGGL(sample_features_kernel, dim3(gx, gy), dim3(256), 0,
                     sailor::as_stream(stream), a);
  return sailor::check_launch("sample_features");
}
