// Differentiable compositing of samples taken in the order given (the
// PyTorch compositing the reference trains with), forward and gradient.
//
// Semantics of c_lib/VoxelEncoding/voxel_encoding_helper.py:
//  * _volume_render_torch.forward (:132-164), density form:
//      delta_i = t_{i+1} - t_i, delta_{S-1} = 0;  e_i = delta_i sigma_i
//      alpha_i = 1 - exp(-e_i);  T_i = exp(-sum_{j<i} e_j);  w_i = alpha_i T_i
//  * _volume_render_torch.forward_occ (:166-186), occupancy form:
//      alpha_i = sigma_i;  T_i = prod_{j<i} (1 - alpha_j + 1e-6);  w_i = alpha_i T_i
//  * outputs feats = sum w_i f_i, depth = sum w_i t_i, ws = sum w_i,
//    alphas = sum w_i alpha_i; rays whose `valid` byte is 0 get zeros (and
//    zero gradients), as the reference's masked assignment does.
// No sort index, no early termination and no skipping of negative depths:
// every sample of the row takes part, exactly as in the tensor formulation.
//
// Gradient: with G_i = dL/dw_i = g_f . f_i + g_d t_i + g_w + g_a alpha_i and
// the suffix sums S_k = sum_{i>k} G_i w_i (accumulated walking the row
// backwards),
//   density:   dL/dsigma_k = delta_k [ exp(-e_k) (G_k T_k + g_a w_k) - S_k ]
//   occupancy: dL/dalpha_k = G_k T_k + g_a w_k - S_k / (1 - alpha_k + 1e-6)
//   dL/df_k = w_k g_f.
//
// Work split: a segment of 16, 32 or 64 lanes (backward: 8 too; the power of two
// that holds the row, rows over 64 in pieces) owns a ray, a lane a sample, so
// rows are read and written whole lines at a time; transmittances are a product
// (sum) scan over the segment and the suffix sums a scan from its end (of a row
// in pieces the backward keeps the state before each piece in the gradient row
// that it overwrites later).  Feature rows
// are walked flat, 16 bytes a lane where F % 4 == 0.  What bounds it is HBM:
// 65,536 rays x 48 x 16 channels move 0.23 GB forward and 0.43 GB backward.
// One lane per ray, each load of a wave in 64 different lines, took 127.5 and
// 462.6 us there; this form takes 52.0 and 87.3 us (4.3 and 4.9 TB/s).  Short
// rows take a lane per ray (lane_forward_pays).
//
// With `compensated` the forward keeps Kahan-compensated running sums (the
// density form's exponent prefix sum and the four output sums), one lane per
// ray in sample order.  The lane forms' channels are processed in groups of up
// to FG per lane (grid.y = channel groups), each lane re-running the cheap
// scalar recurrence of its ray.
#include "common.h"

namespace {

constexpr int kThreads = 128;
constexpr float kOccEps = 1e-6f;

template <bool COMP>
struct Sum {
  float s = 0.0f, c = 0.0f;
  __device__ __forceinline__ void add(float x) {
    if constexpr (!COMP) {
      s += x;
      return;
    }
    const float y = x - c;
    const float t = s + y;
    c = (t - s) - y;
    s = t;
  }
  // the value of the sum (c holds the negated lost low bits)
  __device__ __forceinline__ float value() const { return s - c; }
};

template <int FG, bool COMP>
__global__ void __launch_bounds__(kThreads)
lane_forward(const float* __restrict__ t, const float* __restrict__ sigma,
             const float* __restrict__ feats, const unsigned char* __restrict__ valid,
             long long n_rays, int S, int F, int occ_mode, float* __restrict__ out_feats,
             float* __restrict__ out_depth, float* __restrict__ out_ws,
             float* __restrict__ out_alpha) {
  const long long ray = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (ray >= n_rays) return;
  const int f0 = blockIdx.y * FG;
  const int nf = min(FG, F - f0);
  const float* tr = t + ray * S;
  const float* sr = sigma + ray * S;
  const float* fr = feats + ray * (long long)S * F + f0;
  Sum<COMP> acc[FG], dep, ws, al, pre;
  if (valid == nullptr || valid[ray] != 0) {
    float Tprod = 1.0f;
    for (int i = 0; i < S; ++i) {
      const float z = tr[i];
      float alpha, T;
      if (occ_mode) {
        alpha = sr[i];
        T = Tprod;
        Tprod *= 1.0f - alpha + kOccEps;
      } else {
        const float delta = i + 1 < S ? tr[i + 1] - z : 0.0f;
        const float e = delta * sr[i];
        T = expf(-pre.value());
        alpha = 1.0f - expf(-e);
        pre.add(e);
      }
      const float w = alpha * T;
#pragma unroll
      for (int j = 0; j < FG; ++j)
        if (j < nf) acc[j].add(w * fr[(size_t)i * F + j]);
      if (f0 == 0) {
        dep.add(w * z);
        ws.add(w);
        al.add(w * alpha);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < FG; ++j)
    if (j < nf) out_feats[ray * F + f0 + j] = acc[j].value();
  if (f0 == 0) {
    out_depth[ray] = dep.value();
    out_ws[ray] = ws.value();
    out_alpha[ray] = al.value();
  }
}

// All channels in one lane: G_i needs the full dot product g_f . f_i.  The
// first walk parks T_k in the gradient row that the second overwrites.
template <int FMAX>
__global__ void __launch_bounds__(kThreads)
lane_backward(const float* __restrict__ g_feats, const float* __restrict__ g_depth,
              const float* __restrict__ g_ws, const float* __restrict__ g_alpha,
              const float* __restrict__ t, const float* __restrict__ sigma,
              const float* __restrict__ feats, const unsigned char* __restrict__ valid,
              long long n_rays, int S, int F, int occ_mode, float* __restrict__ grad_sigma,
              float* __restrict__ grad_feats) {
  const long long ray = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (ray >= n_rays) return;
  const float* tr = t + ray * S;
  const float* sr = sigma + ray * S;
  const float* fr = feats + ray * (long long)S * F;
  float* gs = grad_sigma + ray * S;
  float* gf = grad_feats + ray * (long long)S * F;
  if (valid != nullptr && valid[ray] == 0) {
    for (int i = 0; i < S; ++i) gs[i] = 0.0f;
    for (int i = 0; i < S * F; ++i) gf[i] = 0.0f;
    return;
  }
  float gF[FMAX];
#pragma unroll
  for (int j = 0; j < FMAX; ++j) gF[j] = j < F ? g_feats[ray * F + j] : 0.0f;
  const float gD = g_depth[ray], gW = g_ws[ray], gA = g_alpha[ray];
  float pre = 0.0f, Tprod = 1.0f;
  for (int i = 0; i < S; ++i) {
    float alpha, T;
    if (occ_mode) {
      alpha = sr[i];
      T = Tprod;
      Tprod *= 1.0f - alpha + kOccEps;
    } else {
      const float delta = i + 1 < S ? tr[i + 1] - tr[i] : 0.0f;
      const float e = delta * sr[i];
      T = expf(-pre);
      alpha = 1.0f - expf(-e);
      pre += e;
    }
    const float w = alpha * T;
    gs[i] = T;
#pragma unroll
    for (int j = 0; j < FMAX; ++j)
      if (j < F) gf[(size_t)i * F + j] = w * gF[j];
  }
  float suffix = 0.0f;   // last sample first
  for (int i = S - 1; i >= 0; --i) {
    const float T = gs[i];
    const float z = tr[i];
    float G = gD * z + gW;
#pragma unroll
    for (int j = 0; j < FMAX; ++j)
      if (j < F) G += gF[j] * fr[(size_t)i * F + j];
    float grad;
    float w;
    if (occ_mode) {
      const float alpha = sr[i];
      w = alpha * T;
      G += gA * alpha;
      grad = G * T + gA * w - suffix / (1.0f - alpha + kOccEps);
    } else {
      const float delta = i + 1 < S ? tr[i + 1] - z : 0.0f;
      const float e = delta * sr[i];
      const float keep = expf(-e);
      const float alpha = 1.0f - keep;
      w = alpha * T;
      G += gA * alpha;
      grad = delta * (keep * (G * T + gA * w) - suffix);
    }
    gs[i] = grad;
    suffix += G * w;
  }
}

constexpr int kWave = 64;
constexpr int kWavesPerBlock = kThreads / kWave;

// Inclusive scan over each SEG-lane segment: of products (MUL) or sums, from
// its first lane or, REV, from its last.
template <int SEG, bool MUL, bool REV>
__device__ __forceinline__ float seg_scan(float x, int pos) {
#pragma unroll
  for (int o = 1; o < SEG; o <<= 1) {
    const float y = REV ? __shfl_down(x, o, SEG) : __shfl_up(x, o, SEG);
    if (REV ? pos + o < SEG : pos >= o) x = MUL ? x * y : x + y;
  }
  return x;
}

template <int SEG>
__device__ __forceinline__ float seg_sum(float x) {
#pragma unroll
  for (int o = 1; o < SEG; o <<= 1) x += __shfl_xor(x, o, SEG);
  return x;
}

// A sample's alpha and transmittance, lane `pos` of a segment holding sample
// i0 + pos; carry is the transmittance (occupancy form) or the exponent sum
// (density form) before sample i0 and leaves as the one after the piece.
// Lanes past the row (!in) have alpha 0 and leave the recurrence unchanged.
struct Sample {
  float alpha, T, keep;   // keep: exp(-e), density form
};
template <int SEG>
__device__ __forceinline__ Sample seg_sample(float sg, float delta, bool in, bool occ_mode,
                                             int pos, float& carry) {
  Sample r;
  if (occ_mode) {
    r.alpha = in ? sg : 0.0f;
    r.keep = 0.0f;
    const float inc = seg_scan<SEG, true, false>(in ? 1.0f - sg + kOccEps : 1.0f, pos);
    const float before = __shfl_up(inc, 1, SEG);
    r.T = pos == 0 ? carry : carry * before;
    carry *= __shfl(inc, SEG - 1, SEG);
  } else {
    const float e = in ? delta * sg : 0.0f;
    r.keep = expf(-e);
    r.alpha = in ? 1.0f - r.keep : 0.0f;
    const float inc = seg_scan<SEG, false, false>(e, pos);
    const float before = __shfl_up(inc, 1, SEG);
    r.T = expf(-(pos == 0 ? carry : carry + before));
    carry += __shfl(inc, SEG - 1, SEG);
  }
  return r;
}

// Flat walk of feature rows: lane -> (sample `sub` of `spw` per step, VEC
// channels from `c`); lanes past spw * F / VEC idle.
template <int VEC>
struct FlatLane {
  int fv, spw, sub, c;
  bool on;
  __device__ __forceinline__ FlatLane(int F, int lane) {
    fv = F / VEC;                       // channel vectors of a row
    fv = fv < kWave ? fv : kWave;
    spw = kWave / fv;
    sub = lane / fv;
    c = (lane - sub * fv) * VEC;
    on = sub < spw;
  }
};

template <int VEC> struct VecOf;
template <> struct VecOf<1> { typedef float T; };
template <> struct VecOf<4> { typedef float T __attribute__((ext_vector_type(4))); };

// grid.x = waves / 2, grid.y = groups of 64 * VEC channels.
template <int SEG, int VEC>
__global__ void __launch_bounds__(kThreads)
scan_forward(const float* __restrict__ t, const float* __restrict__ sigma,
             const float* __restrict__ feats, const unsigned char* __restrict__ valid,
             long long n_rays, int S, int F, int occ_mode, float* __restrict__ out_feats,
             float* __restrict__ out_depth, float* __restrict__ out_ws,
             float* __restrict__ out_alpha) {
  typedef typename VecOf<VEC>::T V;
  constexpr int RPW = kWave / SEG;   // rays of a wave
  __shared__ float s_w[kWavesPerBlock][kWave];
  __shared__ float s_acc[kWavesPerBlock][kWave * VEC];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int seg = lane / SEG, pos = lane % SEG;
  const long long ray0 = ((long long)blockIdx.x * kWavesPerBlock + wave) * RPW;
  const long long ray = ray0 + seg;
  const bool live = ray < n_rays && (valid == nullptr || valid[ray] != 0);
  const int g0 = blockIdx.y * kWave * VEC;         // first channel of this group
  const int Fg = min(F - g0, kWave * VEC);
  const FlatLane<VEC> fl(Fg, lane);
  V acc[RPW];
#pragma unroll
  for (int r = 0; r < RPW; ++r) acc[r] = V(0.0f);
  float carry = occ_mode ? 1.0f : 0.0f, dep = 0.0f, ws = 0.0f, al = 0.0f;
  for (int i0 = 0; i0 < S; i0 += SEG) {
    const int i = i0 + pos;
    const bool in = live && i < S;
    float z = 0.0f, sg = 0.0f, delta = 0.0f;
    if (in) {
      z = t[ray * S + i];
      sg = sigma[ray * S + i];
      if (!occ_mode && i + 1 < S) delta = t[ray * S + i + 1] - z;
    }
    const Sample q = seg_sample<SEG>(sg, delta, in, occ_mode != 0, pos, carry);
    const float w = q.alpha * q.T;
    if (in) {
      dep += w * z;
      ws += w;
      al += w * q.alpha;
    }
    // the wave's LDS accesses are served in order; the fence only keeps the
    // compiler from moving them
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    s_w[wave][lane] = w;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int n = min(SEG, S - i0);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      if (!__shfl((int)live, r * SEG, kWave)) continue;
      const float* row = feats + ((ray0 + r) * S + i0) * F + g0 + fl.c;
      if (fl.on) {
#pragma unroll 4
        for (int k = fl.sub; k < n; k += fl.spw)
          acc[r] += s_w[wave][r * SEG + k] * *reinterpret_cast<const V*>(row + (size_t)k * F);
      }
    }
  }
  // lanes of the same channels: halve the samples' lanes while their number
  // is even, add what is left in order
#pragma unroll
  for (int r = 0; r < RPW; ++r) {
    if (ray0 + r >= n_rays) break;
    V v = fl.on ? acc[r] : V(0.0f);
    int spw = fl.spw;
    while ((spw & 1) == 0) {
      spw >>= 1;
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        float* e = reinterpret_cast<float*>(&v) + j;
        const float y = __shfl_down(*e, spw * fl.fv, kWave);
        *e += y;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    *reinterpret_cast<V*>(&s_acc[wave][lane * VEC]) = v;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    for (int c = lane; c < Fg; c += kWave) {
      float x = 0.0f;
      for (int k = 0; k < spw; ++k) x += s_acc[wave][k * fl.fv * VEC + c];
      out_feats[(ray0 + r) * F + g0 + c] = x;
    }
  }
  if (blockIdx.y == 0) {
    dep = seg_sum<SEG>(dep);
    ws = seg_sum<SEG>(ws);
    al = seg_sum<SEG>(al);
    if (pos == 0 && ray < n_rays) {
      out_depth[ray] = dep;
      out_ws[ray] = ws;
      out_alpha[ray] = al;
    }
  }
}

// F <= FMAX <= 64 channels: G_i needs the full dot product g_f . f_i, which a
// sample's lane forms from its own feature row (16 bytes at a time, the rows
// of a segment adjacent); dL/df is written flat.
template <int SEG, int VEC, int FMAX>
__global__ void __launch_bounds__(kThreads)
scan_backward(const float* __restrict__ g_feats, const float* __restrict__ g_depth,
              const float* __restrict__ g_ws, const float* __restrict__ g_alpha,
              const float* __restrict__ t, const float* __restrict__ sigma,
              const float* __restrict__ feats, const unsigned char* __restrict__ valid,
              long long n_rays, int S, int F, int occ_mode, float* __restrict__ grad_sigma,
              float* __restrict__ grad_feats) {
  typedef typename VecOf<VEC>::T V;
  constexpr int RPW = kWave / SEG;
  __shared__ float s_w[kWavesPerBlock][kWave];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int seg = lane / SEG, pos = lane % SEG;
  const long long ray0 = ((long long)blockIdx.x * kWavesPerBlock + wave) * RPW;
  const long long ray = ray0 + seg;
  const bool exists = ray < n_rays;
  const bool live = exists && (valid == nullptr || valid[ray] != 0);
  const FlatLane<VEC> fl(F, lane);
  const float gD = live ? g_depth[ray] : 0.0f, gW = live ? g_ws[ray] : 0.0f,
              gA = live ? g_alpha[ray] : 0.0f;
  const bool occ = occ_mode != 0;
  // rows longer than a segment: the state before each piece, kept in the
  // sigma-gradient row (overwritten below) at the piece's first sample
  const int pieces = (S + SEG - 1) / SEG;
  float carry = occ ? 1.0f : 0.0f;
  auto load = [&](int i, bool in, float& z, float& sg, float& delta) {
    z = sg = delta = 0.0f;
    if (in) {
      z = t[ray * S + i];
      sg = sigma[ray * S + i];
      if (!occ && i + 1 < S) delta = t[ray * S + i + 1] - z;
    }
  };
  for (int p = 0; p + 1 < pieces; ++p) {
    float z, sg, delta;
    const bool in = live;
    load(p * SEG + pos, in, z, sg, delta);
    if (in && pos == 0) grad_sigma[ray * S + p * SEG] = carry;
    seg_sample<SEG>(sg, delta, in, occ, pos, carry);
  }
  float suffix = 0.0f;   // sum of G w over the later pieces
  for (int p = pieces - 1; p >= 0; --p) {
    const int i = p * SEG + pos;
    const bool in = live && i < S;
    float z, sg, delta;
    load(i, in, z, sg, delta);
    if (p + 1 < pieces) {
      // written by lane 0 of this segment above
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      carry = live ? grad_sigma[ray * S + p * SEG] : 1.0f;
    }
    float G = gD * z + gW;
    if (in) {
      const float* row = feats + (ray * S + i) * F;
      const float* gf = g_feats + ray * F;
#pragma unroll
      for (int j = 0; j < FMAX; j += VEC)
        if (j < F) {
          const V f = *reinterpret_cast<const V*>(row + j);
          const V g = *reinterpret_cast<const V*>(gf + j);
          const float* fe = reinterpret_cast<const float*>(&f);
          const float* ge = reinterpret_cast<const float*>(&g);
#pragma unroll
          for (int k = 0; k < VEC; ++k) G += ge[k] * fe[k];
        }
    }
    const Sample q = seg_sample<SEG>(sg, delta, in, occ, pos, carry);
    const float w = q.alpha * q.T;
    G += gA * q.alpha;
    const float inc = seg_scan<SEG, false, true>(in ? G * w : 0.0f, pos);
    const float after = __shfl_down(inc, 1, SEG);
    const float behind = suffix + (pos == SEG - 1 ? 0.0f : after);
    suffix += __shfl(inc, 0, SEG);
    if (exists && i < S) {
      float grad = 0.0f;
      if (in)
        grad = occ ? G * q.T + gA * w - behind / (1.0f - q.alpha + kOccEps)
                   : delta * (q.keep * (G * q.T + gA * w) - behind);
      grad_sigma[ray * S + i] = grad;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    s_w[wave][lane] = in ? w : 0.0f;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    const int n = min(SEG, S - p * SEG);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
      if (ray0 + r >= n_rays) break;
      const bool on = __shfl((int)live, r * SEG, kWave) != 0;
      if (!fl.on) continue;
      V g = V(0.0f);
      if (on) g = *reinterpret_cast<const V*>(g_feats + (ray0 + r) * F + fl.c);
      float* row = grad_feats + ((ray0 + r) * S + p * SEG) * F + fl.c;
      for (int k = fl.sub; k < n; k += fl.spw)
        *reinterpret_cast<V*>(row + (size_t)k * F) = on ? s_w[wave][r * SEG + k] * g : V(0.0f);
    }
  }
}

// lanes of a ray's segment
int seg_of(int S) { return S <= 8 ? 8 : S <= 16 ? 16 : S <= 32 ? 32 : 64; }

// Calls a lane per ray is faster for: a segment spends most of a short row on
// its reduction and leaves lanes idle, while a lane per ray waits for its
// samples one after another (so rays have to be many for it) and loses its rows
// from the caches once they are much larger than those.  Forward, lane and
// segment, occupancies, us: 1,048,576 rays of 4 x 4 (samples x channels) 63 and
// 453, 65,536 of 8 x 8 14 and 33, of 16 x 8 27 and 35, of 16 x 16 41 and 31;
// 262,144 of 8 x 8 81 and 115, of 16 x 4 138 and 122; 4,096 of 16 x 4 12 and
// 8.5.  Backward: 524,288 of 1 x 4 6 and 47, of 4 x 4 53 and 70, of 6 x 4 124
// and 88.
bool lane_forward_pays(long long n_rays, int S, int F) {
  const bool four = F % 4 == 0;   // 16 bytes a lane in the segments
  const long long row = (long long)S * F;
  if (S <= 8 && row <= (four ? 32 : 24)) return true;
  return S <= std::min<long long>(20, 4 + n_rays / 3072) && row <= (four ? 128 : 80) &&
         n_rays * row <= (four ? 1 << 24 : 1 << 23) && n_rays * S <= 3 << 20;
}
bool lane_backward_pays(int S, int F) { return S <= 4 && F <= 16 && S * F <= 20; }

int check_args(long long n_rays, int S, int F) {
  SAILOR_REQUIRE(n_rays >= 0 && S >= 1 && F >= 1,
                 "volume_render_torch: need n_rays >= 0, S >= 1, F >= 1 (got %lld, %d, %d)",
                 n_rays, S, F);
  return SAILOR_OK;
}

int launch_forward(bool lane, const float* t, const float* sigma, const float* feats,
                   const unsigned char* valid, long long n_rays, int S, int F, int occ_mode,
                   int compensated, float* out_feats, float* out_depth, float* out_ws,
                   float* out_alpha, hipStream_t st) {
  if (lane) {
    constexpr int FG = 8;
    auto kern = lane_forward<FG, false>;
    if (compensated) kern = lane_forward<FG, true>;
    hipLaunchKernelGGL(kern, dim3(sailor::ceil_div(n_rays, kThreads), (F + FG - 1) / FG),
                       dim3(kThreads), 0, st, t, sigma, feats, valid, n_rays, S, F, occ_mode,
                       out_feats, out_depth, out_ws, out_alpha);
    return sailor::check_launch("volume_render_torch_forward");
  }
  // 16-byte feature accesses where every row starts on 16 bytes
  const bool vec = F % 4 == 0 && ((uintptr_t)feats & 15) == 0;
  const int groups = (F + kWave * (vec ? 4 : 1) - 1) / (kWave * (vec ? 4 : 1));
#define SAILOR_SCAN_FWD(SEG, VEC)                                                             \
  hipLaunchKernelGGL((scan_forward<SEG, VEC>),                                                \
                     dim3(sailor::ceil_div(n_rays, kWavesPerBlock * (kWave / SEG)), groups),  \
                     dim3(kThreads), 0, st, t, sigma, feats, valid, n_rays, S, F, occ_mode,   \
                     out_feats, out_depth, out_ws, out_alpha)
  switch (seg_of(S)) {
    case 8:    // 8 rays' accumulators in a lane leave one wave per SIMD
    case 16: if (vec) SAILOR_SCAN_FWD(16, 4); else SAILOR_SCAN_FWD(16, 1); break;
    case 32: if (vec) SAILOR_SCAN_FWD(32, 4); else SAILOR_SCAN_FWD(32, 1); break;
    default: if (vec) SAILOR_SCAN_FWD(64, 4); else SAILOR_SCAN_FWD(64, 1);
  }
#undef SAILOR_SCAN_FWD
  return sailor::check_launch("volume_render_torch_forward");
}

int launch_backward(const float* g_feats, const float* g_depth, const float* g_ws,
                    const float* g_alpha, const float* t, const float* sigma, const float* feats,
                    const unsigned char* valid, long long n_rays, int S, int F, int occ_mode,
                    float* grad_sigma, float* grad_feats, hipStream_t st) {
  if (lane_backward_pays(S, F)) {
    auto kern = lane_backward<16>;
    if (F <= 4) kern = lane_backward<4>;
    hipLaunchKernelGGL(kern, dim3(sailor::ceil_div(n_rays, kThreads)), dim3(kThreads), 0, st,
                       g_feats, g_depth, g_ws, g_alpha, t, sigma, feats, valid, n_rays, S, F,
                       occ_mode, grad_sigma, grad_feats);
    return sailor::check_launch("volume_render_torch_backward");
  }
  const bool vec = F % 4 == 0 &&
                   (((uintptr_t)feats | (uintptr_t)g_feats | (uintptr_t)grad_feats) & 15) == 0;
#define SAILOR_SCAN_BWD(SEG, VEC, FM)                                                         \
  hipLaunchKernelGGL((scan_backward<SEG, VEC, FM>),                                           \
                     dim3(sailor::ceil_div(n_rays, kWavesPerBlock * (kWave / SEG))),          \
                     dim3(kThreads), 0, st, g_feats, g_depth, g_ws, g_alpha, t, sigma, feats, \
                     valid, n_rays, S, F, occ_mode, grad_sigma, grad_feats)
#define SAILOR_SCAN_BWD_F(SEG, VEC)                                                           \
  do {                                                                                        \
    if (F <= 4) SAILOR_SCAN_BWD(SEG, VEC, 4);                                                 \
    else if (F <= 16) SAILOR_SCAN_BWD(SEG, VEC, 16);                                          \
    else SAILOR_SCAN_BWD(SEG, VEC, 64);                                                       \
  } while (0)
  switch (seg_of(S)) {
    case 8: if (vec) SAILOR_SCAN_BWD_F(8, 4); else SAILOR_SCAN_BWD_F(8, 1); break;
    case 16: if (vec) SAILOR_SCAN_BWD_F(16, 4); else SAILOR_SCAN_BWD_F(16, 1); break;
    case 32: if (vec) SAILOR_SCAN_BWD_F(32, 4); else SAILOR_SCAN_BWD_F(32, 1); break;
    default: if (vec) SAILOR_SCAN_BWD_F(64, 4); else SAILOR_SCAN_BWD_F(64, 1);
  }
#undef SAILOR_SCAN_BWD_F
#undef SAILOR_SCAN_BWD
  return sailor::check_launch("volume_render_torch_backward");
}

}  // namespace

extern "C" int sailor_volume_render_torch_forward(const float* t, const float* sigma,
                                                  const float* feats,
                                                  const unsigned char* valid, long long n_rays,
                                                  int S, int F, int occ_mode, int compensated,
                                                  float* out_feats, float* out_depth,
                                                  float* out_ws, float* out_alpha,
                                                  void* stream) {
  int rc = check_args(n_rays, S, F);
  if (rc) return rc;
  SAILOR_REQUIRE((F + 7) / 8 <= 65535, "volume_render_torch: F = %d too large", F);
  const bool lane = compensated || lane_forward_pays(n_rays, S, F);
  return sailor::in_parts(n_rays, [&](long long r, long long n) {
    return launch_forward(lane, t + r * S, sigma + r * S, feats + r * S * F,
                          valid ? valid + r : nullptr, n, S, F, occ_mode, compensated,
                          out_feats + r * F, out_depth + r, out_ws + r, out_alpha + r,
                          sailor::as_stream(stream));
  });
}

extern "C" int sailor_volume_render_torch_backward(
    const float* g_feats, const float* g_depth, const float* g_ws, const float* g_alpha,
    const float* t, const float* sigma, const float* feats, const unsigned char* valid,
    long long n_rays, int S, int F, int occ_mode, float* grad_sigma, float* grad_feats,
    void* stream) {
  int rc = check_args(n_rays, S, F);
  if (rc) return rc;
  SAILOR_REQUIRE(F <= 64, "volume_render_torch_backward: at most 64 channels (got %d)", F);
  return sailor::in_parts(n_rays, [&](long long r, long long n) {
    return launch_backward(g_feats + r * F, g_depth + r, g_ws + r, g_alpha + r, t + r * S,
                           sigma + r * S, feats + r * S * F, valid ? valid + r : nullptr, n, S,
                           F, occ_mode, grad_sigma + r * S, grad_feats + r * S * F,
                           sailor::as_stream(stream));
  });
}
