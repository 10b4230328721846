// Dense (unbinned) poly-splat + WSR: every gaussian against every pixel it may weigh on.
//
// Two forms of the reference's dense entry points:
//   quad  : spike/render.py:14-49 arm "A" -- Q = a dx^2 + 2b dx dy + c dy^2 with dx = px - mu_x
//           (spike/forward.py:13-21), w = o*keep*max(0, 1 - Q/k)^2, WSR blend
//           (spike/arms.py:22-31).  Operands are the projected records proj[G,12]; the backward
//           yields the per-gaussian (a, b, c, mu_x, mu_y, col_o rgb, o_col) gradients that the
//           geometry backward consumes.
//   theta : spike/backward.py:11-63 (wsr_polysplat) -- u = Phi[p] . theta_u[g] for an arbitrary
//           basis Phi[P,6], w = o*keep*max(u,0)^2; backward gives g_theta[G,6], g_o[G],
//           g_color[G,3], g_w_b.
//
// Quad forward: a block per tile of pixels, the gaussians whose support reaches it listed in LDS
// (DenseWalk below).  Quad backward: a pass over the pixels for their WSR gradients (gnum = gC/den,
// gden = -(gC.C)/den), then waves per gaussian over the pixels of its support box.
// theta forward: the waves of a block share its pixels and split the gaussians, staged in LDS.
// theta backward: a block owns 64 gaussians and a band of pixels, whose WSR gradients it stages in
// LDS; its waves split the pixels.  Band partials go to a workspace and are summed in band order
// by a second kernel.
// All results are deterministic and there are no floating-point atomics.
//
// The quad form also renders the two per-pixel occlusion arms of spike/arms.py (ARM template):
//   SZ (soft-Z, :50-68):  W0 = o w_geo, z* = sum W0 z / (sum W0 + 1e-6) per pixel (pass 1),
//        h = sigmoid(-beta (z - z*)), C = WSR(W0 h) (pass 2); z is a constant of the gradient,
//        z* is not: its gradient Z = sum_g dL/dh h (1 - h) beta is a pixel pre-pass of the
//        backward, and dL/dW0 += Z (z - z*) / den0.  beta (softz_beta) gets a gradient too.
//   RV (revealage, :71-83): C = C_avg (1 - R) + c_b R, C_avg = sum W color / (sum W + 1e-6),
//        R = exp(sum log(1 - min(W, 1 - 1e-4))) (no w_b); dL/dW gains -dL/dlogR / (1 - a).
// aux [P,4] carries the per-pixel forward state to the backward (SZ: z*, den0; RV: R, C_avg).

#include <type_traits>

#include "tts_common.h"

namespace tts {

constexpr int kArmA = 0, kArmSZ = 1, kArmRV = 2;   // TTS_ARM_* values
constexpr int kQuadComp = 9;    // a, b, c, mu_x, mu_y, col_o r, g, b, o_col
constexpr int kThetaComp = 10;  // theta 0..5, o, color r, g, b
constexpr int kDenseTargetBlocks = 2048;
constexpr size_t kDenseMaxWorkspace = size_t(1) << 30;

// Pixels per band of the theta form's backward (a multiple of 256, or P) for G gaussians over P
// pixels: up to 2048 (64 gaussians, band) blocks of 16 waves, but bands of whole 1024-pixel
// stagings where those still give each CU two blocks.  Measured, about 512 / 1024 / 2048 blocks
// (us, band sums included): G 2000, 128x128 26 / 28 / 34; G 6000, 100x100 45 / 43 / 45; 200x200 135
// / 131 / 122; G 2000, 600x600 360 / 350 / 346.
inline int dense_band_pixels(int G, int P) {
  const int gchunks = (G + 63) / 64;
  int nb = kDenseTargetBlocks / (gchunks > 0 ? gchunks : 1);
  if (nb < 1) nb = 1;
  int pb = (P + nb - 1) / nb;
  pb = ((pb + 255) / 256) * 256;
  if (pb < 256) pb = 256;
  if (pb < 1024 && (int64_t)gchunks * ((P + 1023) / 1024) >= 512) pb = 1024;
  // 512 blocks run at once: among 4 to 8 such rounds, the split whose rounds hold the fewest pixels
  // in all, if it saves 2 % (G 20000, P 40000 434 -> 419 us, P 160000 1700 -> 1643)
  auto pixels = [&](int64_t b) { return ((int64_t)gchunks * ((P + b - 1) / b) + 511) / 512 * b; };
  for (int r = 5; r <= 8 && pb > 1024; ++r) {
    const int n = 512 * r / gchunks;
    if (n < 1) continue;
    const int b = ((P + n - 1) / n + 255) / 256 * 256;
    if (b >= 1024 && pixels(b) < pixels(pb) - pixels(pb) / 50) pb = b;
  }
  // keep the partials within the workspace cap, down to one band (past the cap from G = 2^30 / 40)
  while (pb < P && (size_t)((P + pb - 1) / pb) * (size_t)G * kThetaComp * 4 > kDenseMaxWorkspace)
    pb = pb <= P / 2 ? 2 * pb : P;
  return pb;
}

// Workspace of the theta form: [align to 256][gwb partials, nb floats, padded to 256]
// [partials nb*G*kThetaComp].
inline size_t pad256(size_t n) { return (n + 255) & ~size_t(255); }
inline size_t theta_ws_bytes(int G, int P) {
  if (G <= 0 || P <= 0) return 0;
  const int pb = dense_band_pixels(G, P);
  const size_t nb = (size_t)((P + pb - 1) / pb);
  return 256 + pad256(nb * 4) + nb * (size_t)G * kThetaComp * 4;
}

constexpr int kPreBlocks = 256;

// The quad form's backward takes the image in runs of up to kRunPixels pixels (whole rows, or part
// of one), so that its 24 bytes a pixel stay under 1 GiB.
constexpr int kRunPixels = 1 << 25;

// Workspace of the quad form, n = min(P, kRunPixels): [align to 256][gwb partials, kPreBlocks
// floats] [wild flags, kPreBlocks + 1 ints, padded to 256][per-pixel gradients, n float4][arm
// extras, n float2, padded][the shares' gradients, shares*G*(kQuadComp + 1), when there is more
// than one].
//
// Shares of a gaussian's box in the backward: few gaussians over a large image would leave most of
// the GPU idle, and from 256 on the sum of the shares costs more than it gives.  Every box the
// whole image, shares as here / 16 below 64 gaussians and 4 below 256 (us): G 1, 800x800 44 / 65; G
// 100 62 / 216; G 255, 400x400 42 / 67.
inline int quad_shares(int G, int P) {
  if (G >= 256) return 1;
  const int by_g = 1024 / G, by_p = P / 1024, n = by_g < by_p ? by_g : by_p;
  return n < 1 ? 1 : (n > 16 ? 16 : n);
}

inline size_t quad_ws_bytes(int G, int P) {
  if (G <= 0 || P <= 0) return 0;
  const size_t sh = (size_t)quad_shares(G, P), n = P < kRunPixels ? P : kRunPixels;
  return 256 + kPreBlocks * 4 + pad256((kPreBlocks + 1) * 4) + pad256(n * 16) + pad256(n * 8) +
         (sh > 1 ? sh * (size_t)G * (kQuadComp + 1) * 4 : 0);
}

// A long 1-D grid: blocks past 2^21 go to the z dimension (a launch holds under 2^32 threads per
// dimension).  The kernels take block_id() and leave when it is past their work.
inline dim3 grid_split(int64_t blocks, int y = 1) {
  constexpr int64_t kRow = int64_t(1) << 21;
  return blocks <= kRow ? dim3((unsigned)blocks, y)
                        : dim3((unsigned)kRow, y, (unsigned)((blocks + kRow - 1) / kRow));
}
__device__ __forceinline__ int block_id() { return (int)(blockIdx.x + gridDim.x * blockIdx.z); }

// ---------------------------------------------------------------- support culling
//
// A gaussian weighs nothing where Q >= k, so a tile of pixels only needs the gaussians whose
// support may reach it.  support_half returns half-extents of a box around the mean that holds
// every point where the *computed* u = 1 - Q/k can be positive, or infinity when it cannot say.
// The computed Q is off by at most 12 eps (a dx^2 + c dy^2) (three rounded products and sums;
// |2b dx dy| <= a dx^2 + c dy^2), so the points lie in the ellipse of the form with a and c
// reduced by 1e-6; 3e-5 is taken from a*c below, which also covers the rounding of a*c - b^2, and
// 0.1 % is added to k.  No bound is given, and the gaussian is taken everywhere, when the form is
// not positive definite by that margin, or when a value is so large (or not a number) that a
// product it enters, times a zero weight, might not be zero.
__device__ __forceinline__ float2 support_half(float4 r0, float4 r1, float4 r2, float kk) {
  const float a = r0.z, b = r0.w, c = r1.x;
  const float det = a * c * (1.0f - 3e-5f) - b * b;
  const bool ok = fabsf(r0.x) < 1e12f && fabsf(r0.y) < 1e12f && a > 0.0f && a < 1e9f &&
                  c > 0.0f && c < 1e9f && det > 1e-30f &&
                  fabsf(r1.y) + fabsf(r1.z) + fabsf(r1.w) + fabsf(r2.x) + fabsf(r2.y) < 1e12f;
  const float s = kk / det;
  return ok ? make_float2(sqrtf(s * c), sqrtf(s * a)) : make_float2(INFINITY, INFINITY);
}
// The limits on the values alone: a calm record may be evaluated anywhere.
__device__ __forceinline__ bool calm_record(float4 r0, float4 r1, float4 r2) {
  return fabsf(r0.x) < 1e12f && fabsf(r0.y) < 1e12f && fabsf(r0.z) < 1e9f && fabsf(r0.w) < 1e9f &&
         fabsf(r1.x) < 1e9f &&
         fabsf(r1.y) + fabsf(r1.z) + fabsf(r1.w) + fabsf(r2.x) + fabsf(r2.y) < 1e12f;
}
// u = 1 - Q/k with its roundings spelled out: the same value wherever it is inlined.
__device__ __forceinline__ float quad_u(float dx, float dy, float a, float b2, float c,
                                        float inv_k) {
  const float Q = __builtin_fmaf(__builtin_fmaf(a, dx, b2 * dy), dx, (c * dy) * dy);
  return __builtin_fmaf(-Q, inv_k, 1.0f);
}
// The same with the row's b2 dy and (c dy) dy at hand.
__device__ __forceinline__ float quad_u_row(float dx, float a, float b2dy, float cdy2,
                                            float inv_k) {
  const float Q = __builtin_fmaf(__builtin_fmaf(a, dx, b2dy), dx, cdy2);
  return __builtin_fmaf(-Q, inv_k, 1.0f);
}
// k with the margin above
__device__ __forceinline__ float support_k(float inv_k) { return 1.001f / inv_k; }

// Magnitudes whose products stay finite, so that a zero weight makes them zero: the longest is
// soft-Z's o_col (Z/den0) (z - z*), three factors.
__device__ __forceinline__ bool tame(float v) { return fabsf(v) < 1e12f; }

// Does the box reach the pixel centres within `half` of `centre`?  (false only when it cannot:
// an infinite extent gives true, a NaN difference too; 0.01 covers the rounding of both sides)
__device__ __forceinline__ bool reaches(float centre, float half, float mu, float ext) {
  return !(fabsf(centre - mu) > ext + half + 0.01f);
}

// A block's walk over the gaussians that reach its TS x TS pixels.  All threads test NT
// gaussians at a time against the tile and append the hits, in order, to a list in LDS (one
// barrier a round: the waves' hit counts are exchanged through a double buffer); when the list
// could overflow in the next round, and at the end, it is evaluated.  For that the tile is cut
// into 8 x 8 patches, one pixel per lane, and each patch's gaussians are dealt to SPL waves:
// a wave tests 64 list entries at once against its patch and visits every SPL-th hit, two at a
// time.  The order of a pixel's additions depends on nothing but the inputs.
template <int TS, int NT>
struct DenseWalk {
  static constexpr int NW = NT / 64;
  static constexpr int PATCH = (TS / 8) * (TS / 8);
  static constexpr int SPL = NW / PATCH;
  static constexpr int CAP = NT + NT / 4;
  static_assert(SPL * PATCH == NW, "whole waves per patch");
  float4 a[CAP];  // mu_x, mu_y, a, 2b
  float4 b[CAP];  // c, col_o r, g, b
  float2 o[CAP];  // o_col, depth
  float2 h[TS > 8 ? CAP : 1];  // half-extents
  int cnt[2][NW];

  // pixel of this lane: its tile starts at (X0, Y0)
  __device__ __forceinline__ static int lane_x() {
    return ((threadIdx.x >> 6) / SPL) % (TS / 8) * 8 + (threadIdx.x & 7);
  }
  __device__ __forceinline__ static int lane_y() {
    return ((threadIdx.x >> 6) / SPL) / (TS / 8) * 8 + ((threadIdx.x & 63) >> 3);
  }
  __device__ __forceinline__ static int split() { return (threadIdx.x >> 6) % SPL; }

  // STRAIGHT: a list of all gaussians tested for it (so that nearly all reach every patch) is
  // walked without testing the patches.  Arm A, every box the whole image: G 2000, 400x400 157 ->
  // 125 us, 800x800 536 -> 466 (and 30.6 -> 31.0 at G 10000, 800x800 with small boxes); not for the
  // other arms, whose pairs cost several times as much.
  template <bool STRAIGHT, class F>
  __device__ __forceinline__ void evaluate(int n, int tested, int X0, int Y0, const F& f) {
    const int lane = threadIdx.x & 63, sp = split();
    if (TS == 8) {
      for (int j = sp; j < n; j += 2 * SPL) {
        const bool two = j + SPL < n;
        const int j1 = two ? j + SPL : j;
        const float4 A0 = a[j], B0 = b[j], A1 = a[j1], B1 = b[j1];
        const float2 O0 = o[j], O1 = o[j1];
        f(A0, B0, O0);
        if (two) f(A1, B1, O1);
      }
      return;
    }
    if (STRAIGHT && n == tested) {
#pragma unroll 2
      for (int i = sp; i < n; i += SPL) f(a[i], b[i], o[i]);
      n = 0;
    }
    const float cx = (float)(X0 + (lane_x() & ~7)) + 4.0f;
    const float cy = (float)(Y0 + (lane_y() & ~7)) + 4.0f;
    int seen = 0;
    for (int j0 = 0; j0 < n; j0 += 64) {
      const int j = min(j0 + lane, n - 1);
      const float4 A = a[j];
      const float2 e = h[j];
      const bool hit = j0 + lane < n && reaches(cx, 3.5f, A.x, e.x) && reaches(cy, 3.5f, A.y, e.y);
      uint64_t m = __ballot(hit);
      if (SPL > 1) {
        const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                   __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
        const int hits = __popcll(m);
        m = __ballot(hit && (seen + rank) % SPL == sp);
        seen += hits;
      }
      while (m) {
        const int i0 = j0 + __builtin_ctzll(m);
        m &= m - 1;
        const bool two = m != 0;
        const int i1 = two ? j0 + __builtin_ctzll(m) : i0;
        m &= m - 1;
        const float4 A0 = a[i0], B0 = b[i0], A1 = a[i1], B1 = b[i1];
        const float2 O0 = o[i0], O1 = o[i1];
        f(A0, B0, O0);
        if (two) f(A1, B1, O1);
      }
    }
  }

  // f(A, B, O) for every gaussian that may weigh on this lane's pixel (and some that do not).
  // cull = 0 takes every gaussian.  Ends with a barrier.
  template <bool STRAIGHT = false, class F>
  __device__ __forceinline__ void walk(const float* __restrict__ proj, int G, float inv_k, int cull,
                                       int X0, int Y0, const F& f) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const float kk = support_k(inv_k);
    const float half = 0.5f * (TS - 1);
    const float cx = (float)X0 + 0.5f * TS, cy = (float)Y0 + 0.5f * TS;
    const float4* rec = reinterpret_cast<const float4*>(proj);
    int n = 0, buf = 0, from = 0;   // from: the first gaussian that the list is of
    float4 n0, n1, n2;
    if (G > 0) {
      const int64_t g = min((int)threadIdx.x, G - 1);
      n0 = rec[g * 3]; n1 = rec[g * 3 + 1]; n2 = rec[g * 3 + 2];
    }
    for (int g0 = 0; g0 < G; g0 += NT) {
      const float4 r0 = n0, r1 = n1, r2 = n2;
      if (G - g0 > NT) {   // the next round's records, in flight during this one
        const int64_t g = min(g0 + NT + (int)threadIdx.x, G - 1);
        n0 = rec[g * 3]; n1 = rec[g * 3 + 1]; n2 = rec[g * 3 + 2];
      }
      const float2 e = cull ? support_half(r0, r1, r2, kk) : make_float2(INFINITY, INFINITY);
      const bool hit = (int)threadIdx.x < G - g0 && reaches(cx, half, r0.x, e.x) &&
                       reaches(cy, half, r0.y, e.y);
      const uint64_t m = __ballot(hit);
      if (lane == 0) cnt[buf][wave] = __popcll(m);
      __syncthreads();
      const int v = lane < NW ? cnt[buf][lane] : 0;
      const int incl = wave_incl_scan(v);
      const int base = __builtin_amdgcn_readlane(incl, wave) - __builtin_amdgcn_readlane(v, wave);
      const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                 __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
      if (hit) {
        const int at = n + base + rank;
        a[at] = make_float4(r0.x, r0.y, r0.z, 2.0f * r0.w);
        b[at] = make_float4(r1.x, r1.z, r1.w, r2.x);
        o[at] = make_float2(r2.y, r1.y);
        if (TS > 8) h[at] = e;
      }
      n += __builtin_amdgcn_readlane(incl, 63);
      buf ^= 1;
      if (n > CAP - NT || G - g0 <= NT) {
        __syncthreads();
        evaluate<STRAIGHT>(n, min(G, g0 + NT) - from, X0, Y0, f);
        n = 0;
        from = g0 + NT;
        __syncthreads();
      }
    }
  }

  // Sums v over the SPL waves of each patch, in wave order, through the list's storage; call it
  // after walk().  Ends with a barrier.
  template <int N>
  __device__ __forceinline__ void join(float (&v)[N]) {
    if (SPL == 1) return;
    static_assert(SPL == 1 || N * NT <= 8 * CAP, "fits the list");
    float* s = reinterpret_cast<float*>(this);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; ++i) s[(i * NW + wave) * 64 + lane] = v[i];
    __syncthreads();
    const int w0 = wave / SPL * SPL;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      float t = 0.0f;
#pragma unroll
      for (int j = 0; j < SPL; ++j) t += s[(i * NW + w0 + j) * 64 + lane];
      v[i] = t;
    }
    __syncthreads();
  }
};

// ---------------------------------------------------------------- forward

struct Gauss {
  float mx, my, a, b, c, z, cr, cg, cb, oc;
};
// (a uniform index: scalar loads)
__device__ __forceinline__ Gauss gauss(const float* __restrict__ proj, int64_t g) {
  const float* r = proj + g * 12;
  return {r[0], r[1], r[2], r[3], r[4], r[5], r[6], r[7], r[8], r[9]};
}

// One pair's terms of a pixel's sums: colour, density, and revealage's logarithm.
template <int ARM, int N>
__device__ __forceinline__ void add_pair(float (&v)[N], float w, float cr, float cg, float cb,
                                         float oc, float z, float zstar, float beta) {
  if (ARM == kArmSZ) w *= sigmoidf_(-beta * (z - zstar));
  if (ARM == kArmRV) v[N - 1] += log1pf(-fminf(w * oc, 1.0f - 1e-4f));
  v[0] += w * cr;
  v[1] += w * cg;
  v[2] += w * cb;
  v[3] += w * oc;
}
// The pixel of those sums, and what its backward needs.
template <int ARM, int N>
__device__ __forceinline__ void blend_pixel(int64_t p, const float (&v)[N], float zstar, float den0,
                                            const float* __restrict__ bg, float* __restrict__ image,
                                            float* __restrict__ den_out, float4* __restrict__ aux) {
  if (ARM == kArmRV) {
    const float d = v[3] + 1e-6f, R = expf(v[N - 1]);
    const float a0 = v[0] / d, a1 = v[1] / d, a2 = v[2] / d;
    image[p * 3 + 0] = a0 * (1.0f - R) + bg[1] * R;
    image[p * 3 + 1] = a1 * (1.0f - R) + bg[2] * R;
    image[p * 3 + 2] = a2 * (1.0f - R) + bg[3] * R;
    if (den_out) den_out[p] = d;
    aux[p] = make_float4(R, a0, a1, a2);
  } else {
    const float wb = bg[0];
    const float d = v[3] + wb;
    image[p * 3 + 0] = (v[0] + wb * bg[1]) / d;
    image[p * 3 + 1] = (v[1] + wb * bg[2]) / d;
    image[p * 3 + 2] = (v[2] + wb * bg[3]) / d;
    if (den_out) den_out[p] = d;
    if (ARM == kArmSZ) aux[p] = make_float4(zstar, den0, 0.0f, 0.0f);
  }
}

// Bound by the tile tests (48 bytes of L2 per gaussian and tile) and by the pairs inside the
// support.  Visiting every pair instead, one thread per pixel, took 91 us at G 2000, 128x128 (64
// blocks, a serial chain of 2000), 1840-2040 us at G 10000, 800x800, and 441 us for SZ at G 3001,
// 173x131; this walk takes under 13, 41 and 20 us.
template <int ARM, int TS, int NT>
__global__ __launch_bounds__(NT) void k_render_dense(const float* __restrict__ proj, int G, int W,
                                                     int H, float inv_k, int cull,
                                                     const float* __restrict__ bg,
                                                     const float* __restrict__ szb,
                                                     float* __restrict__ image,
                                                     float* __restrict__ den_out,
                                                     float4* __restrict__ aux) {
  using Walk = DenseWalk<TS, NT>;
  __shared__ Walk s;
  const int tx = (W + TS - 1) / TS, bid = block_id();
  const int X0 = bid % tx * TS, Y0 = bid / tx * TS;
  if (Y0 >= H) return;
  const int x = X0 + Walk::lane_x(), y = Y0 + Walk::lane_y();
  const float px = (float)x + 0.5f, py = (float)y + 0.5f;
  const float beta = ARM == kArmSZ ? szb[0] : 0.0f;
  float zstar = 0.0f, den0 = 0.0f;
  auto weight = [&](const float4& A, const float4& B) {
    const float r = relu_nan(quad_u(px - A.x, py - A.y, A.z, A.w, B.x, inv_k));
    return r * r;
  };
  if (ARM == kArmSZ) {   // z* first
    if (!tame(beta)) cull = 0;
    float v[2] = {0.f, 0.f};
    s.walk(proj, G, inv_k, cull, X0, Y0, [&](const float4& A, const float4& B, const float2& O) {
      const float w = weight(A, B);
      v[0] += w * O.x;
      v[1] += w * O.x * O.y;
    });
    s.join(v);
    den0 = v[0] + 1e-6f;
    zstar = v[1] / den0;
    if (__syncthreads_or(!tame(zstar))) cull = 0;
  }
  float v[ARM == kArmRV ? 5 : 4] = {};
  s.template walk<ARM == kArmA>(proj, G, inv_k, cull, X0, Y0, [&](const float4& A, const float4& B,
                                                                  const float2& O) {
    add_pair<ARM>(v, weight(A, B), B.y, B.z, B.w, O.x, O.y, zstar, beta);
  });
  s.join(v);
  if (Walk::split() != 0 || x >= W || y >= H) return;
  blend_pixel<ARM>((int64_t)y * W + x, v, zstar, den0, bg, image, den_out, aux);
}

// The same for up to kFew gaussians: one thread per pixel, every pair visited, no list to build.
constexpr int kFew = 32;
template <int ARM>
__global__ __launch_bounds__(256) void k_render_dense_few(const float* __restrict__ proj, int G,
                                                          int W, int P, float inv_k,
                                                          const float* __restrict__ bg,
                                                          const float* __restrict__ szb,
                                                          float* __restrict__ image,
                                                          float* __restrict__ den_out,
                                                          float4* __restrict__ aux) {
  __shared__ float4 s_a[kFew], s_b[kFew];
  __shared__ float2 s_o[kFew];
  const int p = blockIdx.x * 256 + threadIdx.x;
  const float px = (float)(p % W) + 0.5f, py = (float)(p / W) + 0.5f;
  if ((int)threadIdx.x < G) {
    const float4* r = reinterpret_cast<const float4*>(proj + (int64_t)threadIdx.x * 12);
    const float4 r0 = r[0], r1 = r[1], r2 = r[2];
    s_a[threadIdx.x] = make_float4(r0.x, r0.y, r0.z, 2.0f * r0.w);
    s_b[threadIdx.x] = make_float4(r1.x, r1.z, r1.w, r2.x);
    s_o[threadIdx.x] = make_float2(r2.y, r1.y);
  }
  __syncthreads();
  const float beta = ARM == kArmSZ ? szb[0] : 0.0f;
  float zstar = 0.0f, den0 = 0.0f;
  auto weight = [&](const float4& A, const float4& B) {
    const float r = relu_nan(quad_u(px - A.x, py - A.y, A.z, A.w, B.x, inv_k));
    return r * r;
  };
  if (ARM == kArmSZ) {   // z* first
    float n = 0.0f, d = 0.0f;
#pragma unroll 4
    for (int g = 0; g < G; ++g) {
      const float w = weight(s_a[g], s_b[g]);
      const float2 O = s_o[g];
      d += w * O.x;
      n += w * O.x * O.y;
    }
    den0 = d + 1e-6f;
    zstar = n / den0;
  }
  float v[ARM == kArmRV ? 5 : 4] = {};
#pragma unroll 4
  for (int g = 0; g < G; ++g) {
    const float4 A = s_a[g], B = s_b[g];
    const float2 O = s_o[g];
    add_pair<ARM>(v, weight(A, B), B.y, B.z, B.w, O.x, O.y, zstar, beta);
  }
  if (p < P) blend_pixel<ARM>(p, v, zstar, den0, bg, image, den_out, aux);
}

// theta form, forward: SPL waves of a block share 64 * PX pixels (PX per lane), the gaussians are
// dealt to them in runs and their sums joined in wave order.  Every pair counts (the basis is
// arbitrary, so there is no support box): bound by the 10 CU cycles of LDS a gaussian's 40 bytes
// take per wave and, with PX pixels sharing them, by the VALU (13 instructions a pair); the joins
// cost where there are few gaussians, a wave's own pixels (SPL = 1) where there are few pixels.
constexpr int kThetaThreads = 1024;
constexpr int kThetaWaves = kThetaThreads / 64;

template <int PX, int SPL, int NT>
__global__ __launch_bounds__(NT) void k_wsr_dense(
    const float* __restrict__ theta, const float* __restrict__ o, const float* __restrict__ color,
    const uint8_t* __restrict__ keep, const float* __restrict__ phi, int G, int P,
    const float* __restrict__ bg, float* __restrict__ C, float* __restrict__ den_out) {
  __shared__ float4 s_a[NT];  // theta 0..3
  __shared__ float4 s_c[NT];  // o*keep*color, o*keep
  __shared__ float2 s_b[NT];  // theta 4, 5
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = wave % SPL;
  const int64_t p0 = ((int64_t)block_id() * (NT / 64 / SPL) + wave / SPL) * 64 * PX + lane;
  if ((int64_t)block_id() * (NT / SPL) * PX >= P) return;
  float f[PX][6], n[PX][4];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
#pragma unroll
    for (int k = 0; k < 6; ++k) f[i][k] = p0 + i * 64 < P ? phi[(p0 + i * 64) * 6 + k] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) n[i][k] = 0.f;
  }
  for (int g0 = 0; g0 < G; g0 += NT) {
    const int cnt = min(NT, G - g0);
    __syncthreads();
    if ((int)threadIdx.x < cnt) {
      const int g = g0 + threadIdx.x;
      const float* th = theta + (int64_t)g * 6;
      const float ok = (keep && !keep[g]) ? 0.0f : o[g];
      s_a[threadIdx.x] = make_float4(th[0], th[1], th[2], th[3]);
      s_b[threadIdx.x] = make_float2(th[4], th[5]);
      s_c[threadIdx.x] = make_float4(ok * color[(int64_t)g * 3 + 0], ok * color[(int64_t)g * 3 + 1],
                                     ok * color[(int64_t)g * 3 + 2], ok);
    }
    __syncthreads();
    const int j1 = (sub + 1) * cnt / SPL;
#pragma unroll 4
    for (int j = sub * cnt / SPL; j < j1; ++j) {
      const float4 A = s_a[j], Cc = s_c[j];
      const float2 B = s_b[j];
#pragma unroll
      for (int i = 0; i < PX; ++i) {
        const float u = f[i][0] * A.x + f[i][1] * A.y + f[i][2] * A.z + f[i][3] * A.w +
                        f[i][4] * B.x + f[i][5] * B.y;
        const float r = relu_nan(u);
        const float w = r * r;
        n[i][0] += w * Cc.x;
        n[i][1] += w * Cc.y;
        n[i][2] += w * Cc.z;
        n[i][3] += w * Cc.w;
      }
    }
  }
  static_assert(SPL == 1 || PX <= SPL, "a finishing wave each");
  // a pixel's sums, joined over the waves that share it: [wave][4][64] floats fill s_a
  float* s = reinterpret_cast<float*>(s_a);
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    if (SPL > 1) {
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 4; ++k) s[(wave * 4 + k) * 64 + lane] = n[i][k];
      __syncthreads();
      if (sub != i) continue;   // wave i of the sharing ones finishes their i-th run of pixels
#pragma unroll
      for (int k = 0; k < 4; ++k) n[i][k] = 0.f;
#pragma unroll
      for (int w = 0; w < SPL; ++w) {
#pragma unroll
        for (int k = 0; k < 4; ++k) n[i][k] += s[((wave - i + w) * 4 + k) * 64 + lane];
      }
    }
    const int64_t p = p0 + i * 64;
    if (p < P) {
      const float wb = bg[0];
      const float d = n[i][3] + wb;
      C[p * 3 + 0] = (n[i][0] + wb * bg[1]) / d;
      C[p * 3 + 1] = (n[i][1] + wb * bg[2]) / d;
      C[p * 3 + 2] = (n[i][2] + wb * bg[3]) / d;
      if (den_out) den_out[p] = d;
    }
  }
}

// ---------------------------------------------------------------- backward

// Stage pixels [p0, p0+256) of a band: (gnum r,g,b, gden); returns this thread's share of
// dL/dw_b = sum(gnum . c_b) + sum(gden).
__device__ __forceinline__ float stage_pixel_grads(const float* __restrict__ image,
                                                   const float* __restrict__ den,
                                                   const float* __restrict__ gimage, int p,
                                                   bool in, const float* __restrict__ bg,
                                                   float4* s_px) {
  float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
  if (in) {
    const float inv = 1.0f / den[p];
    const float g0 = gimage[(int64_t)p * 3 + 0], g1 = gimage[(int64_t)p * 3 + 1],
                g2 = gimage[(int64_t)p * 3 + 2];
    const float c0 = image[(int64_t)p * 3 + 0], c1 = image[(int64_t)p * 3 + 1],
                c2 = image[(int64_t)p * 3 + 2];
    q = make_float4(g0 * inv, g1 * inv, g2 * inv, -(g0 * c0 + g1 * c1 + g2 * c2) * inv);
  }
  s_px[threadIdx.x] = q;
  return q.x * bg[1] + q.y * bg[2] + q.z * bg[3] + q.w;
}

// Quad backward, pass 1: each pixel's WSR gradients q = (gnum r,g,b, gden) and RV's dL/dlogR
// (ex.x), this block's share of dL/dw_b (RV has no w_b) and whether any of its values is wild:
// such a value times a zero weight need not be zero, so pass 2 then visits every pair.  Block 0
// clears the flag the soft-Z pass may raise.
template <int ARM>
__global__ __launch_bounds__(256) void k_dense_pre(const float* __restrict__ image,
                                                   const float* __restrict__ den,
                                                   const float4* __restrict__ aux,
                                                   const float* __restrict__ gimage, int P,
                                                   const float* __restrict__ bg,
                                                   float4* __restrict__ q_out,
                                                   float2* __restrict__ ex,
                                                   float* __restrict__ gwb_part,
                                                   int* __restrict__ wild) {
  __shared__ float s_ftmp[4];
  float wpart = 0.0f;
  bool bad = false;
  for (int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x; p < P; p += (int64_t)gridDim.x * 256) {
    const float inv = 1.0f / den[p];
    const float g0 = gimage[p * 3 + 0], g1 = gimage[p * 3 + 1], g2 = gimage[p * 3 + 2];
    float4 q;
    if (ARM == kArmRV) {
      const float4 x = aux[p];  // R, C_avg
      const float R = x.x, k = (1.0f - R) * inv;  // dC/dC_avg / den
      q = make_float4(g0 * k, g1 * k, g2 * k, -(g0 * x.y + g1 * x.z + g2 * x.w) * k);
      // dL/dR * R = dL/dlogR
      const float gs = (g0 * (bg[1] - x.y) + g1 * (bg[2] - x.z) + g2 * (bg[3] - x.w)) * R;
      ex[p] = make_float2(gs, 0.0f);
      bad |= !tame(gs);
    } else {
      const float c0 = image[p * 3 + 0], c1 = image[p * 3 + 1], c2 = image[p * 3 + 2];
      q = make_float4(g0 * inv, g1 * inv, g2 * inv, -(g0 * c0 + g1 * c1 + g2 * c2) * inv);
      wpart += q.x * bg[1] + q.y * bg[2] + q.z * bg[3] + q.w;
    }
    q_out[p] = q;
    bad |= !tame(fabsf(q.x) + fabsf(q.y) + fabsf(q.z) + fabsf(q.w));
  }
  const float tot = block_sum256(wpart, s_ftmp);
  const int any = __syncthreads_or(bad);
  if (threadIdx.x == 0) {
    gwb_part[blockIdx.x] = tot;
    wild[blockIdx.x] = any;
    if (blockIdx.x == 0) wild[gridDim.x] = 0;
  }
}

// Soft-Z backward, between the passes: Z/den0 of every pixel, Z = dL/dz* =
// beta sum_g w_geo (gnum . col_o + gden o_col) h (1 - h); ex = (z*, Z/den0).  The forward's walk,
// over the W x H pixels from (xo, yo) on.
template <int TS, int NT>
__global__ __launch_bounds__(NT) void k_softz_pre(const float* __restrict__ proj, int G, int W,
                                                  int H, int xo, int yo, float inv_k, int cull,
                                                  const float* __restrict__ szb,
                                                  const float4* __restrict__ aux,
                                                  const float4* __restrict__ qbuf,
                                                  float2* __restrict__ ex, int* __restrict__ wild) {
  using Walk = DenseWalk<TS, NT>;
  __shared__ Walk s;
  const int tx = (W + TS - 1) / TS, bid = block_id();
  const int X0 = bid % tx * TS, Y0 = bid / tx * TS;
  if (Y0 >= H) return;
  const int x = X0 + Walk::lane_x(), y = Y0 + Walk::lane_y();
  const bool in = x < W && y < H;
  const int64_t p = (int64_t)y * W + x;
  const float px = (float)x + ((float)xo + 0.5f), py = (float)y + ((float)yo + 0.5f);
  const float beta = szb[0];
  float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
  float zs = 0.f, d0 = 1.f;
  if (in) {
    q = qbuf[p];
    const float4 ax = aux[p];
    zs = ax.x;
    d0 = ax.y;
  }
  const bool bad = !tame(fabsf(q.x) + fabsf(q.y) + fabsf(q.z) + fabsf(q.w)) || !tame(zs) ||
                   !tame(beta);
  if (__syncthreads_or(bad)) cull = 0;
  float Z[1] = {0.0f};
  s.walk(proj, G, inv_k, cull, X0 + xo, Y0 + yo, [&](const float4& A, const float4& B,
                                                     const float2& O) {
    const float r = relu_nan(quad_u(px - A.x, py - A.y, A.z, A.w, B.x, inv_k));
    const float h = sigmoidf_(-beta * (O.y - zs));
    Z[0] += r * r * (q.x * B.y + q.y * B.z + q.z * B.w + q.w * O.x) * h * (1.0f - h);
  });
  s.join(Z);
  const float zk = beta * Z[0] / d0;
  if (in && Walk::split() == 0) {
    ex[p] = make_float2(zs, zk);
    if (!tame(zs) || !tame(zk) || !tame(beta)) atomicOr(wild, 1);
  }
}

// Quad backward, pass 2: the pixels of the gaussians' support boxes, one pixel per lane, sums over
// lanes, waves and blocks in a fixed order.  ncomp = 9 (a, b, c, mu_x, mu_y, col_o rgb, o_col), 10
// for SZ (+ this gaussian's dL/dbeta).
//
// A block serves GPB gaussians with WPG waves each.  Where every box is small each gaussian's waves
// walk its box: bound by the latency of a few dependent steps (record, box, two to ten rounds of
// pixel loads, lane sums).  Otherwise all the block's waves walk one box after another, or, where
// two gaussians' boxes fill most of their union, both jointly: the waves deal out its 8 x 8 pixel
// cells and evaluate the pair on each, a lane staying in its row.  The pixel's 16-byte load, its
// coordinates and the loop are then paid once for two gaussians and the row's terms once per row:
// 20 VALU instructions a pixel and gaussian, which bound it (a box by itself: about 40, and 16
// bytes of L2 reads).  Only for calm records (no value whose product with a zero weight might not
// be zero). gridDim.y > 1 (few gaussians): each row of blocks takes a share of every box, or of the
// cells, and writes its own gradients; k_dense_reduce adds them.
//
// Whole arm-A backward in us, against one thread per gaussian over every pixel (bands of pixels
// staged in LDS, band sums): small boxes, G 2000, 128x128 9.6 (that form 40), G 10000, 300x300 15
// (435), 800x800 34 (3000); every box the whole image, G 2000, 128x128 29 (41), 400x400 178 (226),
// 800x800 802 (711), G 10000, 300x300 487 (468); a whole-image box among 256 small ones, 800x800
// 222 (388), among 10000 445 (3014).  Each box by itself always, by its own waves: 43, 331, 1487,
// 863, 797, 807.  Soft-Z, every box the whole image: 116 (294), 1009 (1003), G 4000, 400x400 1947
// (1867).
template <int ARM>
struct PairSums {
  float r = 0.f, g = 0.f, b = 0.f, o = 0.f, beta = 0.f;   // dL/d col_o, o_col, softz_beta
};
// Adds one pair's colour, density (and soft-Z beta) terms; returns its dL/dw_geo.
template <int ARM>
__device__ __forceinline__ float pair_grad(PairSums<ARM>& s, float w, float4 q, float2 e,
                                           const Gauss& gs, float beta) {
  const float oc = gs.oc, zg = gs.z;
  const float gw = q.x * gs.cr + q.y * gs.cg + q.z * gs.cb + q.w * oc;  // dL/dw_geo of arm A
  if (ARM == kArmSZ) {   // e: z*, Z/den0
    const float h = sigmoidf_(-beta * (zg - e.x));
    const float t = e.y * (zg - e.x);  // dL/dW0 through z*
    s.r += w * h * q.x;
    s.g += w * h * q.y;
    s.b += w * h * q.z;
    s.o += w * (h * q.w + t);
    s.beta -= w * gw * h * (1.0f - h) * (zg - e.x);
    return h * gw + oc * t;
  }
  s.r += w * q.x;
  s.g += w * q.y;
  s.b += w * q.z;
  if (ARM == kArmRV) {   // e.x: dL/dlogR
    const float W0 = w * oc;
    const float t = W0 <= 1.0f - 1e-4f ? -e.x / (1.0f - W0) : 0.0f;  // clamp gate
    s.o += w * (q.w + t);
    return gw + oc * t;
  }
  s.o += w * q.w;
  return gw;
}

template <int ARM>
__device__ __forceinline__ float2 pixel_extra(const float2* __restrict__ ex, int64_t p) {
  return ARM == kArmRV ? make_float2(ex[p].x, 0.0f) : ex[p];
}

// Two gaussians are walked jointly where that visits 4 / 5 of the pixels of their boxes or less (a
// visit costs a pair half of what it does alone, but twice the sums at the end), from boxes of 8192
// pixels in all on.
__device__ __forceinline__ bool joint_pays(int cells, int64_t pix) {
  return pix > 8192 && (int64_t)cells * 80 <= pix;
}

// The 8 x 8 cells of the union of the boxes in lanes j and j + 1: from pixel (x0, y0), up to (x1,
// y1).
struct Cells {
  int x0, x1, y0, y1, cols, rows;
};
__device__ __forceinline__ Cells pair_cells(int x0, int x1, int y0, int y1, int j) {
  Cells u;
  u.x0 = min(__builtin_amdgcn_readlane(x0, j), __builtin_amdgcn_readlane(x0, j + 1)) & ~7;
  u.x1 = max(__builtin_amdgcn_readlane(x1, j), __builtin_amdgcn_readlane(x1, j + 1));
  u.y0 = min(__builtin_amdgcn_readlane(y0, j), __builtin_amdgcn_readlane(y0, j + 1));
  u.y1 = max(__builtin_amdgcn_readlane(y1, j), __builtin_amdgcn_readlane(y1, j + 1));
  u.cols = (u.x1 - u.x0 + 7) / 8;
  u.rows = (u.y1 - u.y0 + 7) / 8;
  return u;
}

template <int ARM, int GPB, int WPG>
__global__ __launch_bounds__(64 * GPB * WPG) void k_render_dense_bwd(
    const float* __restrict__ proj, int G, int W, int H, float xc, float yc, int acc, float inv_k,
    int cull, const float* __restrict__ szb, const float4* __restrict__ qbuf,
    const float2* __restrict__ ex,
    const int* __restrict__ wild, int n_pre, int n_wild, const float* __restrict__ gwb_part,
    float* __restrict__ out, float* __restrict__ gwb) {
  constexpr int NC = ARM == kArmSZ ? kQuadComp + 1 : kQuadComp;
  constexpr int NW = GPB * WPG, NV = GPB * NC;
  // not for soft-Z, whose exponential is most of a pair either way (5 % gained jointly, for 48
  // registers more)
  constexpr bool kShared = GPB > 1 && ARM != kArmSZ;
  static_assert(NV <= 64 && (GPB & (GPB - 1)) == 0, "one wave finishes");
  __shared__ float s_sum[NW][NV];
  __shared__ float s_tot[NV];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // a scalar to the compiler
  int share = blockIdx.y, shares = gridDim.y;
  const int64_t g0 = (int64_t)block_id() * GPB;
  if (g0 >= G) return;
  // lane GPB i + j holds gaussian j of the block
  const int64_t g = g0 + (lane & (GPB - 1));
  const bool act = g < G;
  const float4* rec = reinterpret_cast<const float4*>(proj + min(g, (int64_t)G - 1) * 12);
  const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
  const Gauss own = gauss(proj, min(g0 + wave / WPG, (int64_t)G - 1));
  int any = 0;
  for (int i = lane; i < n_wild; i += 64) any |= wild[i];
  if (__ballot(any != 0)) cull = 0;
  if (g0 == 0 && share == 0 && wave == 0 && gwb) {
    float t = 0.0f;
    for (int i = lane; i < n_pre; i += 64) t += gwb_part[i];
    t = wave_sum(t);
    if (lane == 0) gwb[0] = acc & 1 ? gwb[0] + t : t;
  }
  out += ((int64_t)share * G + g0) * NC;
  const float mx = r0.x, my = r0.y;
  const float beta = ARM == kArmSZ ? szb[0] : 0.0f;
  // pixels [x0, x1) x [y0, y1): centres within the box; fminf / fmaxf turn an infinite box (and
  // the NaN of an infinite mean less an infinite extent) into the whole image
  int x0 = 0, x1 = W, y0 = 0, y1 = H;
  if (cull) {
    const float2 e = support_half(r0, r1, r2, support_k(inv_k));
    x0 = (int)fminf(fmaxf(ceilf(mx - e.x - (xc + 0.01f)), 0.0f), (float)W);
    y0 = (int)fminf(fmaxf(ceilf(my - e.y - (yc + 0.01f)), 0.0f), (float)H);
    x1 = (int)fmaxf(fminf(floorf(mx + e.x - (xc - 0.01f)) + 1.0f, (float)W), (float)x0);
    y1 = (int)fmaxf(fminf(floorf(my + e.y - (yc - 0.01f)) + 1.0f, (float)H), (float)y0);
  }
  const int n_pix = act ? (x1 - x0) * (y1 - y0) : 0;
  if (n_pix == 0) x0 = x1 = y0 = y1 = 0;
  // the pairs to be walked jointly; boxes of 32 rounds of their own waves and more are for all
  // waves
  int joint = 0;
  if (kShared && __ballot(n_pix > 4096)) {
    const bool calm = calm_record(r0, r1, r2) && inv_k < INFINITY;
#pragma unroll
    for (int j = 0; j < GPB; j += 2) {
      const int n0 = __builtin_amdgcn_readlane(n_pix, j);
      const int n1 = __builtin_amdgcn_readlane(n_pix, j + 1);
      const Cells u = pair_cells(x0, x1, y0, y1, j);
      if (n0 > 0 && n1 > 0 && joint_pays(u.cols * u.rows, (int64_t)n0 + n1) &&
          __builtin_amdgcn_readlane((int)calm, j) && __builtin_amdgcn_readlane((int)calm, j + 1))
        joint |= 1 << j;
    }
  }
  const bool large = kShared && (joint || __ballot(n_pix > 8192));
  if (shares > 1 && !__ballot(n_pix > 1024)) {   // not worth sharing
    if (share > 0) {
      if (threadIdx.x < NV && g0 + threadIdx.x / NC < G) out[threadIdx.x] = 0.0f;
      return;
    }
    shares = 1;
  }

  // sums of gaussian j over every parts-th run of 64 pixels of its box, from run `part` on
  auto walk = [&](const Gauss& h, int j, int part, int parts, float (&v)[10]) {
    // (lanes are read while every one is active)
    const int bx = __builtin_amdgcn_readlane(x0, j), by = __builtin_amdgcn_readlane(y0, j);
    const int bw = __builtin_amdgcn_readlane(x1, j) - bx;
    const int jn = __builtin_amdgcn_readlane(n_pix, j);
    PairSums<ARM> ps;
    float sxx = 0.f, sxy = 0.f, syy = 0.f, sx = 0.f, sy = 0.f;
    int i = 64 * part + lane;
    if (i < jn) {
      // this lane's pixel, stepped by S pixels in box order without dividing again
      const int S = 64 * parts, dxs = S % bw, dys = S / bw;
      int x = i % bw, y = i / bw;
      int64_t p = (int64_t)(by + y) * W + bx + x;
      float4 q = qbuf[p];
      float2 e = ARM != kArmA ? pixel_extra<ARM>(ex, p) : make_float2(0.f, 0.f);
      while (true) {
        const float dx = (float)(bx + x) + xc - h.mx, dy = (float)(by + y) + yc - h.my;
        const float4 qc = q;
        const float2 ec = e;
        i += S;
        if (i < jn) {   // the next pixel's loads, in flight during this one
          x += dxs;
          y += dys;
          if (x >= bw) {
            x -= bw;
            ++y;
          }
          p = (int64_t)(by + y) * W + bx + x;
          q = qbuf[p];
          if (ARM != kArmA) e = pixel_extra<ARM>(ex, p);
        }
        const float r = relu_nan(quad_u(dx, dy, h.a, 2.0f * h.b, h.c, inv_k));
        const float gu = r * pair_grad<ARM>(ps, r * r, qc, ec, h, beta);
        const float tx = gu * dx, ty = gu * dy;
        sxx += tx * dx;
        sxy += tx * dy;
        syy += ty * dy;
        sx += tx;
        sy += ty;
        if (i >= jn) break;
      }
    }
    v[0] = sxx; v[1] = sxy; v[2] = syy; v[3] = sx; v[4] = sy;
    v[5] = ps.r; v[6] = ps.g; v[7] = ps.b; v[8] = ps.o; v[9] = ps.beta;
#pragma unroll
    for (int k = 0; k < NC; ++k) v[k] = wave_sum(v[k]);
  };
  // lane k < NC writes component k of gaussian j from its sums v (of all lanes)
  auto finish = [&](const Gauss& h, int j, const float (&v)[10]) {
    // dL/dQ = dL/du * (-1/k) = -2 gu / k
    const float s = -2.0f * inv_k;
    const float m_x = s * v[3], m_y = s * v[4];
    float o = s * v[0];                                           // dQ/da = dx^2
    o = lane == 1 ? 2.0f * (s * v[1]) : o;                        // dQ/db = 2 dx dy
    o = lane == 2 ? s * v[2] : o;                                 // dQ/dc = dy^2
    o = lane == 3 ? -2.0f * (h.a * m_x + h.b * m_y) : o;            // dQ/dmu_x = -2 (a dx + b dy)
    o = lane == 4 ? -2.0f * (h.b * m_x + h.c * m_y) : o;            // dQ/dmu_y = -2 (b dx + c dy)
#pragma unroll
    for (int k = 5; k < NC; ++k) o = lane == k ? v[k] : o;
    if (lane < NC && g0 + j < G) out[j * NC + lane] = acc & 2 ? out[j * NC + lane] + o : o;
  };

  float v[10];
  if (!large) {   // each gaussian's waves walk its box
    const int j = wave / WPG, sub = wave % WPG;
    walk(own, j, WPG * share + sub, WPG * shares, v);
    if (WPG > 1) {
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NC; ++k) s_sum[wave][k] = v[k];
      }
      __syncthreads();
      if (sub != 0) return;
#pragma unroll
      for (int k = 0; k < NC; ++k) {
        float t = s_sum[wave][k];
#pragma unroll
        for (int w = 1; w < WPG; ++w) t += s_sum[wave + w][k];
        v[k] = t;
      }
    }
    finish(own, j, v);
    return;
  }

  // all waves walk one pair, or one box, after another
  const int part = NW * share + wave, parts = NW * shares;
  for (int j0 = 0; j0 < GPB; j0 += 2) {
    if (joint >> j0 & 1) {
      const Cells u = pair_cells(x0, x1, y0, y1, j0);
      const Gauss h[2] = {gauss(proj, g0 + j0), gauss(proj, g0 + j0 + 1)};   // (both have pixels)
      PairSums<ARM> ps[2];
      float sxx[2] = {}, sxy[2] = {}, syy[2] = {}, sx[2] = {}, sy[2] = {};
      const int cells = u.cols * u.rows;
      int i = (int)((int64_t)cells * part / parts);
      const int i1 = (int)((int64_t)cells * (part + 1) / parts);
      int band = i / u.cols, col = i - band * u.cols;
      while (i < i1) {   // cells [i, i + m) of one band of 8 rows
        const int m = min(i1 - i, u.cols - col);
        const int y = u.y0 + band * 8 + (lane >> 3);
        const bool row = y < u.y1;
        int x = u.x0 + col * 8 + (lane & 7);
        const float yf = (float)y + yc;
        float dy[2], bd[2], cd[2], s0[2], s1[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          dy[j] = yf - h[j].my;
          bd[j] = (2.0f * h[j].b) * dy[j];
          cd[j] = (h[j].c * dy[j]) * dy[j];
          s0[j] = s1[j] = 0.0f;
        }
        int64_t p = (int64_t)y * W + x;
        float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
        float2 e = make_float2(0.f, 0.f);
        if (row && x < u.x1) {
          q = qbuf[p];
          if (ARM != kArmA) e = pixel_extra<ARM>(ex, p);
        }
        for (int k = 0; k < m; ++k) {
          const float4 qc = q;
          const float2 ec = e;
          const bool in = row && x < u.x1;
          const float xf = (float)x + xc;
          x += 8;
          p += 8;
          if (k + 1 < m && row && x < u.x1) {   // the next cell's loads, in flight during this one
            q = qbuf[p];
            if (ARM != kArmA) e = pixel_extra<ARM>(ex, p);
          }
          if (in) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
              const float dx = xf - h[j].mx;
              // calm: no NaN; gu is half of dL/du
              const float r = fmaxf(quad_u_row(dx, h[j].a, bd[j], cd[j], inv_k), 0.0f);
              const float gu = r * pair_grad<ARM>(ps[j], r * r, qc, ec, h[j], beta);
              const float tx = gu * dx;
              s0[j] += gu;
              s1[j] += tx;
              sxx[j] += tx * dx;
            }
          }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {   // the row's dy
          const float t = dy[j] * s0[j];
          sx[j] += s1[j];
          sy[j] += t;
          sxy[j] += dy[j] * s1[j];
          syy[j] += dy[j] * t;
        }
        i += m;
        col = 0;
        ++band;
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float sum[10] = {sxx[j], sxy[j], syy[j], sx[j], sy[j],
                             ps[j].r, ps[j].g, ps[j].b, ps[j].o, 0.f};
#pragma unroll
        for (int k = 0; k < NC; ++k) {
          const float t = wave_sum(sum[k]);
          if (lane == 0) s_sum[wave][(j0 + j) * NC + k] = t;
        }
      }
      continue;
    }
    for (int j = j0; j < min(j0 + 2, GPB); ++j) {
      walk(gauss(proj, min(g0 + j, (int64_t)G - 1)), j, part, parts, v);
      if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NC; ++k) s_sum[wave][j * NC + k] = v[k];
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    float t = s_sum[0][threadIdx.x];
#pragma unroll
    for (int w = 1; w < NW; ++w) t += s_sum[w][threadIdx.x];
    s_tot[threadIdx.x] = t;
  }
  __syncthreads();
  if (wave < GPB) {
#pragma unroll
    for (int k = 0; k < NC; ++k) v[k] = s_tot[wave * NC + k];
    finish(gauss(proj, min(g0 + wave, (int64_t)G - 1)), wave, v);
  }
}

// theta form, backward: a block owns 64 gaussians (one per lane) and a band of pixels, 1024 of
// which it stages at a time with their WSR gradients; the 16 waves take runs of them and their
// sums are joined in wave order into the band's partial.  Bound by the VALU (24 instructions a
// pair).  256-thread blocks of 256 gaussians over 64 bands, and their 64 partials a gaussian, took
// 44 us at G 2000, 128x128 (17 of it the band sums), 55 at G 6000, 100x100, 151 at 200x200; this
// takes 26, 43 and 122.
__global__ __launch_bounds__(kThetaThreads) void k_wsr_dense_bwd(
    const float* __restrict__ theta, const float* __restrict__ o, const float* __restrict__ color,
    const uint8_t* __restrict__ keep, const float* __restrict__ phi, int G, int P, int PB,
    const float* __restrict__ bg, const float* __restrict__ C, const float* __restrict__ den,
    const float* __restrict__ gC, float* __restrict__ part, float* __restrict__ gwb_part) {
  __shared__ float s_all[kThetaThreads * kThetaComp];
  __shared__ float s_wb[kThetaWaves];
  float4* s_px = reinterpret_cast<float4*>(s_all);
  float4* s_fa = s_px + kThetaThreads;                                // phi 0..3
  float2* s_fb = reinterpret_cast<float2*>(s_fa + kThetaThreads);     // phi 4..5
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int band = blockIdx.y, gblock = block_id();
  if ((int64_t)gblock * 64 >= G) return;
  const int64_t g = (int64_t)gblock * 64 + lane;
  const bool act = g < G;
  float th[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float og = 0.f, kp = 0.f, col[3] = {0.f, 0.f, 0.f};
  if (act) {
#pragma unroll
    for (int i = 0; i < 6; ++i) th[i] = theta[(int64_t)g * 6 + i];
    og = o[g];
    kp = (keep && !keep[g]) ? 0.0f : 1.0f;
#pragma unroll
    for (int i = 0; i < 3; ++i) col[i] = color[(int64_t)g * 3 + i];
  }
  const float ok = og * kp;
  const float cr = ok * col[0], cg = ok * col[1], cb = ok * col[2];
  float v[kThetaComp] = {};   // theta 0..5, then sums of w q: r, g, b, den
  float wpart = 0.f;
  const int pend = min(P, (band + 1) * PB);
  for (int p0 = band * PB; p0 < pend; p0 += kThetaThreads) {
    __syncthreads();
    const int pp = p0 + threadIdx.x;
    const bool in = pp < pend;
    wpart += stage_pixel_grads(C, den, gC, pp, in, bg, s_px);
    float4 fa = make_float4(0.f, 0.f, 0.f, 0.f);
    float2 fb = make_float2(0.f, 0.f);
    if (in) {
      const float* f = phi + (int64_t)pp * 6;
      fa = make_float4(f[0], f[1], f[2], f[3]);
      fb = make_float2(f[4], f[5]);
    }
    s_fa[threadIdx.x] = fa;
    s_fb[threadIdx.x] = fb;
    __syncthreads();
    const int n = min(kThetaThreads, pend - p0);
    const int j1 = (wave + 1) * n / kThetaWaves;
#pragma unroll 2
    for (int j = wave * n / kThetaWaves; j < j1; ++j) {
      const float4 q = s_px[j];
      const float4 fa2 = s_fa[j];
      const float2 fb2 = s_fb[j];
      const float u = fa2.x * th[0] + fa2.y * th[1] + fa2.z * th[2] + fa2.w * th[3] +
                      fb2.x * th[4] + fb2.y * th[5];
      const float r = relu_nan(u);
      const float w = r * r;
      v[6] += w * q.x;
      v[7] += w * q.y;
      v[8] += w * q.z;
      v[9] += w * q.w;
      const float gu = r * (q.x * cr + q.y * cg + q.z * cb + q.w * ok);  // half of dL/du
      v[0] += gu * fa2.x;
      v[1] += gu * fa2.y;
      v[2] += gu * fa2.z;
      v[3] += gu * fa2.w;
      v[4] += gu * fb2.x;
      v[5] += gu * fb2.y;
    }
  }
  if (gblock == 0) {
    const float t = wave_sum(wpart);
    if (lane == 0) s_wb[wave] = t;
  }
  __syncthreads();
  if (gblock == 0 && threadIdx.x == 0) {
    float t = 0.f;
#pragma unroll
    for (int w = 0; w < kThetaWaves; ++w) t += s_wb[w];
    gwb_part[band] = t;
  }
#pragma unroll
  for (int k = 0; k < kThetaComp; ++k) s_all[(wave * kThetaComp + k) * 64 + lane] = v[k];
  __syncthreads();
  float t = 0.f;
  if (wave < kThetaComp) {   // wave k sums component k
#pragma unroll
    for (int w = 0; w < kThetaWaves; ++w) t += s_all[(w * kThetaComp + wave) * 64 + lane];
  }
  __syncthreads();
  if (wave < kThetaComp) s_all[wave * 64 + lane] = t;
  __syncthreads();
  if (wave == 0 && act) {
    float* dst = part + ((int64_t)band * G + g) * kThetaComp;
#pragma unroll
    for (int i = 0; i < 6; ++i) dst[i] = 2.0f * s_all[i * 64 + lane];
    const float gr = s_all[6 * 64 + lane], gg = s_all[7 * 64 + lane], gbl = s_all[8 * 64 + lane],
                gd = s_all[9 * 64 + lane];
    // num = sum w_geo*o*keep*color, den = sum w_geo*o*keep + w_b
    dst[6] = kp * (col[0] * gr + col[1] * gg + col[2] * gbl + gd);  // dL/do
    dst[7] = ok * gr;                                              // dL/dcolor
    dst[8] = ok * gg;
    dst[9] = ok * gbl;
  }
}

template <int N>
__device__ __forceinline__ void add_bands(const float*& src, int64_t stride, int& left, float& s) {
  float v[N];
#pragma unroll
  for (int b = 0; b < N; ++b) v[b] = src[b * stride];
#pragma unroll
  for (int b = 0; b < N; ++b) s += v[b];
  src += N * stride;
  left -= N;
}

// out[g][c] = sum over bands of part[band][g][c], in band order (acc: added to out); gwb = sum of
// gwb_part.
__global__ __launch_bounds__(256) void k_dense_reduce(const float* __restrict__ part, int nb,
                                                      int G, int ncomp,
                                                      const float* __restrict__ gwb_part,
                                                      float* __restrict__ out,
                                                      float* __restrict__ gwb, int acc) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t n = (int64_t)G * ncomp;
  if (i < n) {
    float s = 0.f;
    const float* src = part + i;
    int left = nb;   // bands in order, 16 loads in flight, then 8, 4, 2, 1
    while (left >= 16) add_bands<16>(src, n, left, s);
    if (left >= 8) add_bands<8>(src, n, left, s);
    if (left >= 4) add_bands<4>(src, n, left, s);
    if (left >= 2) add_bands<2>(src, n, left, s);
    if (left) add_bands<1>(src, n, left, s);
    out[i] = acc ? out[i] + s : s;
  }
  if (blockIdx.x == 0 && threadIdx.x < 64 && gwb) {   // wave 0: lanes over the bands
    float s = 0.f;
    for (int b = threadIdx.x; b < nb; b += 64) s += gwb_part[b];
    s = wave_sum(s);
    if (threadIdx.x == 0) gwb[0] = s;
  }
}

// Does pass 2 of the backward take four waves per gaussian, or one?  A support box grows with the
// image.  Measured, whole arm-A backward, four / one (us): G 10000, 800x800 85 / 151; G 4000,
// 800x800 57 / 124; G 2000, 400x400 19 / 32; G 10000, 300x300 31 / 25; 100x60 21 / 17; below 4096
// gaussians on small images the same within 5 %.
inline bool dense_wide(int G, int P) { return G <= 4096 || P >= (1 << 17); }

inline int dense_tiles(int H, int W, int ts) { return ((H + ts - 1) / ts) * ((W + ts - 1) / ts); }

// The support boxes allow 0.01 for the rounding of pixel coordinates (2^-8 at 2^16), and a 1/k in
// range.
inline int dense_cull(int H, int W, float ik) {
  return H <= (1 << 16) && W <= (1 << 16) && ik < INFINITY;
}

// Tiles and threads of the forward's walk (and of the soft-Z pass): every block tests all gaussians
// against its tile, so large tiles test less and small ones make more blocks; where every box is
// the whole image the pairs bound it, and blocks that fill the GPU evenly count.  Measured, arm A,
// small boxes / whole-image boxes (us; soft-Z orders the same way):
//                        few       16/256      16/512      16/1024     32/1024     8/512
//   G 16, 128x128        3.0/3.0   3.3/4.0     3.6/3.8     4.4/4.5     4.1/5.1     3.3/3.5
//   G 32, 400x400        4.6/4.7   3.8/5.9     4.9/6.7     7.6/9.4     4.3/6.8     8.6/10
//   G 64, 800x800        16/17     6.8/19      9.9/21      18/31       7.9/22      25/37
//   G 256, 400x400       20/20     4.1/23      5.2/21      8.0/22      4.5/26      9.0/22
//   G 256, 800x800       50/53     7.0/56      10/55       19/64       8.1/63      25/72
//   G 600, 512x512                 6.3/58      7.4/54      9.8/53      4.8/55      17/62
//   G 2000, 128x128                15/123      8.8/60      7.3/48      12/170      6.1/26
//   G 2000, 256x256                9.9/124     7.0/62      6.3/50      7.3/168     10/58
//   G 2000, 400x400                10/149      9.3/123     11/122      6.3/169     20/118
//   G 2000, 800x800                19/403      21/387      27/389      11/458      59/436
// (one thread per pixel, every pair visited: 3.1, 4.8, 16, 20, 58, -, 88, 90, 125, 390)
template <class F>
void dense_tiling(int G, int H, int W, const F& f) {
  using std::integral_constant;
  auto go = [&](auto ts, auto nt) {
    f(grid_split(dense_tiles(H, W, decltype(ts)::value)), ts, nt);
  };
  if (dense_tiles(H, W, 16) < 256)
    go(integral_constant<int, 8>{}, integral_constant<int, 512>{});
  else if (G <= (dense_tiles(H, W, 32) >= 256 ? 256 : 128))
    go(integral_constant<int, 16>{}, integral_constant<int, 256>{});
  else if (dense_tiles(H, W, 32) >= 256)
    go(integral_constant<int, 32>{}, integral_constant<int, 1024>{});
  else if (dense_tiles(H, W, 16) >= 512 && G <= 8192)
    go(integral_constant<int, 16>{}, integral_constant<int, 512>{});
  else
    go(integral_constant<int, 16>{}, integral_constant<int, 1024>{});
}

// So few gaussians that the forward visits every pair (the table above; the other arms' pairs cost
// more).
inline bool dense_few(int arm, int G, int H, int W) {
  static_assert(kFew >= 32, "staged at once");
  if (arm != kArmA) return G <= (arm == kArmSZ ? 8 : 2);
  return G <= 16 || (G <= 32 && dense_tiles(H, W, 16) >= 256 && dense_tiles(H, W, 32) <= 256);
}

template <int ARM>
void launch_render_dense(const float* proj, int G, int H, int W, float ik, const float* bg,
                         const float* szb, float* image, float* den, float4* aux,
                         hipStream_t stream) {
  if (dense_few(ARM, G, H, W)) {
    k_render_dense_few<ARM><<<grid1d(H * W, 256), 256, 0, stream>>>(proj, G, W, H * W, ik, bg, szb,
                                                                   image, den, aux);
    return;
  }
  const int cull = dense_cull(H, W, ik);
  dense_tiling(G, H, W, [&](dim3 grid, auto ts, auto nt) {
    constexpr int TS = decltype(ts)::value, NT = decltype(nt)::value;
    k_render_dense<ARM, TS, NT><<<grid, NT, 0, stream>>>(proj, G, W, H, ik, cull, bg, szb, image,
                                                         den, aux);
  });
}

// The whole quad backward of an arm; grad has kQuadComp columns (SZ: one more).
template <int ARM>
int launch_dense_bwd(const float* proj, int G, int H, int W, float ik, const float* bg,
                     const float* szb, const float* image, const float* den, const float4* aux,
                     const float* gimage, float* grad, float* gwb, void* ws, size_t ws_bytes,
                     hipStream_t stream) {
  const int P = H * W;
  if (!ws || ws_bytes < quad_ws_bytes(G, P)) return TTS_EWORKSPACE;
  const int cap = P < kRunPixels ? P : kRunPixels;
  char* base = reinterpret_cast<char*>((reinterpret_cast<uintptr_t>(ws) + 255) & ~uintptr_t(255));
  float* gwbp = reinterpret_cast<float*>(base);
  int* wild = reinterpret_cast<int*>(base + kPreBlocks * 4);
  base += kPreBlocks * 4 + pad256((kPreBlocks + 1) * 4);
  float4* q = reinterpret_cast<float4*>(base);
  base += pad256((size_t)cap * 16);
  float2* ex = reinterpret_cast<float2*>(base);
  float* part = reinterpret_cast<float*>(base + pad256((size_t)cap * 8));
  const int cull = dense_cull(H, W, ik);
  const int sh = quad_shares(G, P), nc = ARM == kArmSZ ? kQuadComp + 1 : kQuadComp;
  float* dst = sh > 1 ? part : grad;
  // runs of whole rows, or of part of a row
  const int rw = W < cap ? W : cap, rh = W < cap ? cap / W : 1;
  for (int yo = 0; yo < H; yo += rh) {
    for (int xo = 0; xo < W; xo += rw) {
      const int w = W - xo < rw ? W - xo : rw, h = H - yo < rh ? H - yo : rh, n = w * h;
      const int64_t at = (int64_t)yo * W + xo;
      const float4* ax = ARM == kArmA ? nullptr : aux + at;
      const int npre = n / 256 + 1 < kPreBlocks ? n / 256 + 1 : kPreBlocks;
      k_dense_pre<ARM><<<npre, 256, 0, stream>>>(image + at * 3, den + at, ax, gimage + at * 3, n,
                                                 bg, q, ex, gwbp, wild);
      if constexpr (ARM == kArmSZ)
        dense_tiling(G, h, w, [&](dim3 grid, auto ts, auto nt) {
          constexpr int TS = decltype(ts)::value, NT = decltype(nt)::value;
          k_softz_pre<TS, NT><<<grid, NT, 0, stream>>>(proj, G, w, h, xo, yo, ik, cull, szb, ax, q,
                                                       ex, wild + npre);
        });
      const int nw = npre + (ARM == kArmSZ ? 1 : 0);
      const int more = at > 0, acc = more + (more && sh == 1 ? 2 : 0);
      auto launch = [&](auto gpb, auto wpg) {
        constexpr int GPB = decltype(gpb)::value, WPG = decltype(wpg)::value;
        const dim3 grid = grid_split(((int64_t)G + GPB - 1) / GPB, sh);
        k_render_dense_bwd<ARM, GPB, WPG><<<grid, 64 * GPB * WPG, 0, stream>>>(
            proj, G, w, h, (float)xo + 0.5f, (float)yo + 0.5f, acc, ik, cull, szb, q, ex, wild,
            npre, nw, gwbp, dst, gwb);
      };
      using std::integral_constant;
      if (G >= 256 && G < 512 && P >= (1 << 18))
        launch(integral_constant<int, 1>{}, integral_constant<int, 16>{});
      else if (!dense_wide(G, P))
        launch(integral_constant<int, 4>{}, integral_constant<int, 1>{});
      else
        launch(integral_constant<int, ARM == kArmSZ ? 1 : 2>{}, integral_constant<int, 4>{});
      if (sh > 1)
        k_dense_reduce<<<grid1d((int64_t)G * nc, 256), 256, 0, stream>>>(part, sh, G, nc, nullptr,
                                                                        grad, nullptr, more);
    }
  }
  return launch_status();
}

// Unpacks the theta form's workspace into (partials, gwb partials); returns the band count or an
// error.
inline int theta_ws(void* ws, size_t ws_bytes, int G, int P, float** part, float** gwbp, int* PB) {
  if (!ws || ws_bytes < theta_ws_bytes(G, P)) return TTS_EWORKSPACE;
  *PB = dense_band_pixels(G, P);
  const int nb = (P + *PB - 1) / *PB;
  uintptr_t base = (reinterpret_cast<uintptr_t>(ws) + 255) & ~uintptr_t(255);
  *gwbp = reinterpret_cast<float*>(base);
  *part = reinterpret_cast<float*>(base + pad256((size_t)nb * 4));
  return nb;
}

}  // namespace tts

using namespace tts;

extern "C" {

size_t tts_dense_workspace_bytes(int G, int P) {
  // serves both forms
  const size_t t = theta_ws_bytes(G, P), q = quad_ws_bytes(G, P);
  return t > q ? t : q;
}

int tts_render_dense(const float* proj, int G, int H, int W, float k, const float* bg,
                     float* image, float* den, hipStream_t stream) {
  if ((G > 0 && !proj) || !bg || !image || H <= 0 || W <= 0 || G < 0 || !(k > 0.0f))
    return TTS_EINVAL;
  if (G > (1 << 30)) return TTS_EG;
  if ((int64_t)H * W > (int64_t(1) << 30)) return TTS_EINVAL;
  launch_render_dense<kArmA>(proj, G, H, W, (float)(1.0 / (double)k), bg, nullptr, image, den,
                             nullptr, stream);
  return launch_status();
}

int tts_render_dense_arm(const float* proj, int G, int H, int W, float k, const float* bg,
                         int arm, const float* softz_beta, float* image, float* den, float* aux,
                         hipStream_t stream) {
  if ((G > 0 && !proj) || !bg || !image || H <= 0 || W <= 0 || G < 0 || !(k > 0.0f))
    return TTS_EINVAL;
  if (arm != kArmA && arm != kArmSZ && arm != kArmRV) return TTS_EINVAL;
  if (arm != kArmA && !aux) return TTS_EINVAL;
  if (arm == kArmSZ && !softz_beta) return TTS_EINVAL;
  if (G > (1 << 30)) return TTS_EG;
  if ((int64_t)H * W > (int64_t(1) << 30)) return TTS_EINVAL;
  const float ik = (float)(1.0 / (double)k);
  float4* ax = reinterpret_cast<float4*>(aux);
  if (arm == kArmSZ)
    launch_render_dense<kArmSZ>(proj, G, H, W, ik, bg, softz_beta, image, den, ax, stream);
  else if (arm == kArmRV)
    launch_render_dense<kArmRV>(proj, G, H, W, ik, bg, nullptr, image, den, ax, stream);
  else
    launch_render_dense<kArmA>(proj, G, H, W, ik, bg, nullptr, image, den, nullptr, stream);
  return launch_status();
}

int tts_render_dense_bwd(const float* proj, int G, int H, int W, float k, const float* bg,
                         const float* image, const float* den, const float* gimage, float* grad9,
                         float* gwb, void* workspace, size_t workspace_bytes,
                         hipStream_t stream) {
  if (!proj || !bg || !image || !den || !gimage || !grad9 || H <= 0 || W <= 0 || G <= 0 ||
      !(k > 0.0f))
    return TTS_EINVAL;
  if (G > (1 << 30)) return TTS_EG;
  if ((int64_t)H * W > (int64_t(1) << 30)) return TTS_EINVAL;
  return launch_dense_bwd<kArmA>(proj, G, H, W, (float)(1.0 / (double)k), bg, nullptr, image, den,
                                 nullptr, gimage, grad9, gwb, workspace, workspace_bytes, stream);
}

int tts_render_dense_arm_bwd(const float* proj, int G, int H, int W, float k, const float* bg,
                             int arm, const float* softz_beta, const float* image,
                             const float* den, const float* aux, const float* gimage,
                             float* grad10, float* gwb, void* workspace, size_t workspace_bytes,
                             hipStream_t stream) {
  if (!proj || !bg || !image || !den || !gimage || !grad10 || H <= 0 || W <= 0 || G <= 0 ||
      !(k > 0.0f))
    return TTS_EINVAL;
  if (arm != kArmA && arm != kArmSZ && arm != kArmRV) return TTS_EINVAL;
  if (arm != kArmA && !aux) return TTS_EINVAL;
  if (arm == kArmSZ && !softz_beta) return TTS_EINVAL;
  if (G > (1 << 30)) return TTS_EG;
  if ((int64_t)H * W > (int64_t(1) << 30)) return TTS_EINVAL;
  const float ik = (float)(1.0 / (double)k);
  const float4* ax = reinterpret_cast<const float4*>(aux);
  if (arm == kArmSZ)
    return launch_dense_bwd<kArmSZ>(proj, G, H, W, ik, bg, softz_beta, image, den, ax, gimage,
                                    grad10, gwb, workspace, workspace_bytes, stream);
  if (arm == kArmRV)
    return launch_dense_bwd<kArmRV>(proj, G, H, W, ik, bg, nullptr, image, den, ax, gimage, grad10,
                                    gwb, workspace, workspace_bytes, stream);
  return launch_dense_bwd<kArmA>(proj, G, H, W, ik, bg, nullptr, image, den, nullptr, gimage,
                                 grad10, gwb, workspace, workspace_bytes, stream);
}

int tts_wsr_dense(const float* theta, const float* o, const float* color, const uint8_t* keep,
                  const float* phi, int G, int P, const float* bg, float* C, float* den,
                  hipStream_t stream) {
  if ((G > 0 && (!theta || !o || !color)) || !phi || !bg || !C || P <= 0 || G < 0)
    return TTS_EINVAL;
  if (G > (1 << 30) || P > (1 << 30)) return TTS_EINVAL;
  // Pixels per lane / sharing waves / threads, measured (us):
  //                      1/1/256  4/4/256  1/16/1024  4/16/1024
  //   G 1, P 16384         2.5      4.0       3.7        7.4
  //   G 1, P 640000        5.9       13        46         56
  //   G 64, P 50000        5.0      5.8       7.6        8.5
  //   G 150, P 640000       33       30        62         78
  //   G 300, P 160000       23       20        25         32
  //   G 2000, P 16384       80       62        19         37
  //   G 2000, P 50000       81       62        54         39
  //   G 2000, P 640000     381      292       461        363
  //   G 6000, P 100000     253      206       240        193
  const bool few = G <= 32 || (G <= 100 && P > 32768);
  const bool four = P > 32768 && (G <= 300 || (G <= 4096 && P >= (1 << 16)) || P >= (1 << 18));
  if (few)
    k_wsr_dense<1, 1, 256><<<grid_split(grid1d(P, 256)), 256, 0, stream>>>(
        theta, o, color, keep, phi, G, P, bg, C, den);
  else if (four)
    k_wsr_dense<4, 4, 256><<<grid_split(grid1d(P, 256)), 256, 0, stream>>>(
        theta, o, color, keep, phi, G, P, bg, C, den);
  else if (P <= 32768)
    k_wsr_dense<1, 16, 1024><<<grid_split(grid1d(P, 64)), 1024, 0, stream>>>(
        theta, o, color, keep, phi, G, P, bg, C, den);
  else
    k_wsr_dense<4, 16, 1024><<<grid_split(grid1d(P, 256)), 1024, 0, stream>>>(
        theta, o, color, keep, phi, G, P, bg, C, den);
  return launch_status();
}

int tts_wsr_dense_bwd(const float* theta, const float* o, const float* color,
                      const uint8_t* keep, const float* phi, int G, int P, const float* bg,
                      const float* C, const float* den, const float* gC, float* gtheta10,
                      float* gwb, void* workspace, size_t workspace_bytes, hipStream_t stream) {
  if (!theta || !o || !color || !phi || !bg || !C || !den || !gC || !gtheta10 || P <= 0 ||
      G <= 0)
    return TTS_EINVAL;
  if (G > (1 << 30) || P > (1 << 30)) return TTS_EINVAL;
  float *part, *gwbp;
  int PB;
  const int nb = theta_ws(workspace, workspace_bytes, G, P, &part, &gwbp, &PB);
  if (nb < 0) return nb;
  const dim3 grid = grid_split(grid1d(G, 64), nb);
  k_wsr_dense_bwd<<<grid, kThetaThreads, 0, stream>>>(theta, o, color, keep, phi, G, P, PB, bg, C,
                                                      den, gC, part, gwbp);
  k_dense_reduce<<<grid1d((int64_t)G * kThetaComp, 256), 256, 0, stream>>>(
      part, nb, G, kThetaComp, gwbp, gtheta10, gwb, 0);
  return launch_status();
}

}  // extern "C"
