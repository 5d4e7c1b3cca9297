// The losses beside the photometric one (replaces src/gpu/loss.cu:197-293 and hollow_loss / normal_loss /
// eval_metrics, 317-338): the normal-map supervision of the feature lanes, the hollow-penalty sum and the
// eval metrics (squared error and SSIM of the 8-bit prediction). Each workgroup leaves its sums in a
// partials array that one final workgroup adds up in a fixed order in double precision, so every result is
// deterministic (the reference adds per-warp sums with float atomics).
#pragma clang fp contract(off)
#include "b2c_kernels.h"
#include "device_math.h"
#include "ssim_common.h"

#include <algorithm>

namespace b2c {
namespace dev {
namespace {

constexpr int AUX_BLOCK = 256;
constexpr int AUX_GRID_MAX = 2048;  // grid-stride kernels: at most this many workgroups (and partials)

// Sum of one value over a 256-thread workgroup: wave shuffles, then the four wave totals in LDS, added by
// thread 0 in wave order.
template <typename T>
__device__ __forceinline__ T block_sum(T v, T* s_red) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();  // s_red may still be read from a previous call
  if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = v;
  __syncthreads();
  return ((s_red[0] + s_red[1]) + s_red[2]) + s_red[3];
}

// Normal supervision (loss.cu:206-238) for the pixels whose normal map is opaque (alpha byte above 127):
// with the target decoded as n = (2 r - 1, 1 - 2 g, 1 - 2 b) (r, g, b in [0, 1]; the [+X, -Y, -Z]
// convention) and the rendered feature p, the loss is k (|p - n|_1 + 1 - cos(p, n)), k = scale * weight, with
// both lengths floored at 1e-6. Its gradient, times grad_scale, is
//   k (sign(p - n) - n / (|p| |n|) + p (p . n) / (|p|^3 |n|)).
// Other pixels get a zero gradient.
__global__ void __launch_bounds__(AUX_BLOCK) normal_loss_kernel(b2c_normal_loss_args a) {
  __shared__ float s_red[4];
  const int npix = a.W * a.H;
  float local = 0.f;
  for (int pix = blockIdx.x * AUX_BLOCK + threadIdx.x; pix < npix; pix += gridDim.x * AUX_BLOCK) {
    const uint32_t nm = a.normals[pix];
    float4 out = make_float4(0.f, 0.f, 0.f, 0.f);
    if (((nm >> 24) & 0xffu) > 127u) {
      const float wp = a.weights ? (float)a.weights[pix] * (1.f / 255.f) : 1.f;
      const float k = a.scale * wp;
      const float nx = (float)(nm & 0xffu) * (2.f / 255.f) - 1.f;
      const float ny = 1.f - (float)((nm >> 8) & 0xffu) * (2.f / 255.f);
      const float nz = 1.f - (float)((nm >> 16) & 0xffu) * (2.f / 255.f);
      const float4 f = reinterpret_cast<const float4*>(a.feat)[pix];
      const float pl = fmaxf(sqrtf((f.x * f.x + f.y * f.y) + f.z * f.z), 1e-6f);
      const float nl = fmaxf(sqrtf((nx * nx + ny * ny) + nz * nz), 1e-6f);
      const float dot = (f.x * nx + f.y * ny) + f.z * nz;
      const float plnl = pl * nl;
      const float dx = f.x - nx, dy = f.y - ny, dz = f.z - nz;
      local = local + k * ((((fabsf(dx) + fabsf(dy)) + fabsf(dz)) + 1.f) - dot / plnl);
      const float inv = 1.f / plnl, radial = dot / ((pl * pl) * plnl);
      const float kg = k * a.grad_scale;
      const float sx = dx > 0.f ? 1.f : (dx < 0.f ? -1.f : 0.f);
      const float sy = dy > 0.f ? 1.f : (dy < 0.f ? -1.f : 0.f);
      const float sz = dz > 0.f ? 1.f : (dz < 0.f ? -1.f : 0.f);
      out = make_float4(kg * ((sx - nx * inv) + f.x * radial), kg * ((sy - ny * inv) + f.y * radial),
                        kg * ((sz - nz * inv) + f.z * radial), 0.f);
    }
    reinterpret_cast<float4*>(a.v_feat)[pix] = out;
  }
  const float t = block_sum(local, s_red);
  if (threadIdx.x == 0) a.partials[blockIdx.x] = t;
}

// Per-workgroup sums of the hollow penalty (loss.cu:197-204).
__global__ void __launch_bounds__(AUX_BLOCK) hollow_sum_kernel(const float* __restrict__ pen, int npix,
                                                               float* __restrict__ partials) {
  __shared__ float s_red[4];
  float local = 0.f;
  for (int pix = blockIdx.x * AUX_BLOCK + threadIdx.x; pix < npix; pix += gridDim.x * AUX_BLOCK)
    local = local + pen[pix];
  const float t = block_sum(local, s_red);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}

// Eval metrics (loss.cu:240-286): the prediction clamped to [0, 1] and rounded to 8 bits against the target, per channel
// the squared error and the clamped SSIM (both weighted by the target alpha when mask_weighted; zero outside the
// image), summed in double. Large images take eval_kernel, small ones eval_tile_kernel.
constexpr int ESTATS = 5;  // E[x], E[x^2], E[y], E[y^2], E[xy]

__device__ __forceinline__ float eval_pred(float p) { return __builtin_rintf(fminf(fmaxf(p, 0.f), 1.f) * 255.f) / 255.f; }

// The blurred statistics of one row: 11 taps of (u, v), added to st.
__device__ __forceinline__ void eval_tap(float w, float u, float v, float (&st)[ESTATS]) {
  const float wu = w * u, wv = w * v;
  st[0] = st[0] + wu;
  st[1] = __builtin_fmaf(wu, u, st[1]);
  st[2] = st[2] + wv;
  st[3] = __builtin_fmaf(wv, v, st[3]);
  st[4] = __builtin_fmaf(wu, v, st[4]);
}

__device__ __forceinline__ float eval_ssim(const float (&st)[ESTATS]) {
  const float mu1 = st[0], mu2 = st[2];
  const float s1 = fmaxf(0.f, st[1] - mu1 * mu1), s2 = fmaxf(0.f, st[3] - mu2 * mu2), s12 = st[4] - mu1 * mu2;
  const float num = ((2.f * mu1) * mu2 + C1) * (2.f * s12 + C2);
  const float den = ((mu1 * mu1 + mu2 * mu2) + C1) * ((s1 + s2) + C2);
  return fminf(fmaxf(num / den, -1.f), 1.f);
}

// One 256-thread workgroup per 16x16 tile and channel: the 26x26 input footprint and the horizontally blurred
// statistics of its rows in LDS, a thread per output pixel. A tile's chain is short (load, two blurs) where a strip
// walks at least 33 rows of 0.6 us each, so it is the faster one while the tiles leave the chip room.
constexpr int ET = 16;              // output tile edge
constexpr int EIN = ET + 2 * HALO;  // 26: input footprint edge

__global__ void __launch_bounds__(AUX_BLOCK) eval_tile_kernel(b2c_eval_args a, int tiles_x) {
  __shared__ float s_p[EIN * EIN], s_g[EIN * EIN];
  __shared__ float s_h[EIN * ET][ESTATS];
  __shared__ double s_red[4];
  const int c = blockIdx.y, x0 = ((int)blockIdx.x % tiles_x) * ET, y0 = ((int)blockIdx.x / tiles_x) * ET;
  const int tid = threadIdx.x;
  for (int i = tid; i < EIN * EIN; i += AUX_BLOCK) {
    const int y = y0 - HALO + i / EIN, x = x0 - HALO + i % EIN;
    const bool in = x >= 0 && x < a.W && y >= 0 && y < a.H;
    const size_t pix = in ? (size_t)y * a.W + x : 0;
    s_p[i] = in ? eval_pred(a.pred[pix * 4 + c]) : 0.f;
    s_g[i] = in ? gt_channel(a.gt[pix], c) : 0.f;
  }
  __syncthreads();
  for (int i = tid; i < EIN * ET; i += AUX_BLOCK) {
    const int first = (i / ET) * EIN + i % ET;
    float st[ESTATS] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 11; d++) eval_tap(gw_tap(d), s_p[first + d], s_g[first + d], st);
#pragma unroll
    for (int k = 0; k < ESTATS; k++) s_h[i][k] = st[k];
  }
  __syncthreads();
  const int ly = tid / ET, lx = tid % ET, y = y0 + ly, x = x0 + lx;
  double se = 0.0, ss = 0.0;
  if (x < a.W && y < a.H) {
    float st[ESTATS] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 11; d++) {
#pragma unroll
      for (int k = 0; k < ESTATS; k++) st[k] = __builtin_fmaf(gw_tap(d), s_h[(ly + d) * ET + lx][k], st[k]);
    }
    const int i = (ly + HALO) * EIN + lx + HALO;
    const float m = a.mask_weighted ? gt_channel(a.gt[(size_t)y * a.W + x], 3) : 1.f;
    const float d = fabsf(s_p[i] - s_g[i]) * m;
    se = (double)(d * d);
    ss = (double)(eval_ssim(st) * m);
  }
  const double tse = block_sum(se, s_red);
  const double tss = block_sum(ss, s_red);
  if (tid == 0) {
    const size_t wg = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
    a.partials[2 * wg] = (float)tse;
    a.partials[2 * wg + 1] = (float)tss;
  }
}

// One wave per (strip, channel): a strip is EW = 54 output columns by `rows` output rows, lane l owns column
// x0 - 5 + l and walks down the rows. A step loads one row (a step ahead), blurs it horizontally through a one-row LDS
// buffer into an 11-row register ring of the five statistics, and blurs the ring vertically; unrolled by 11, so the
// ring slots are static registers. Each lane adds its rows' terms in double; the wave's two sums go to partials.
// Bound by the VALU: 16x16 tiles with both passes in LDS re-read 2.6 times the pixels, ran 1.6 times the horizontal blurs,
// kept the statistics in LDS and took 68.4 us at 1600x900; this takes 38.8 us.
constexpr int EW = 64 - 2 * HALO;

__global__ void __launch_bounds__(64) eval_kernel(b2c_eval_args a, int strips_x, int nstrips, int rows) {
  __shared__ float s_p[2][64], s_g[2][64];  // one input row (double buffered)
  // workgroup b runs on XCD b mod 8; a strip's three channels read the same lines there
  const int per = (nstrips * 3 + 7) / 8;
  const int item = (int)(blockIdx.x % 8u) * per + (int)(blockIdx.x / 8u);
  if (item >= nstrips * 3) return;
  const int strip = item / 3, c = item - strip * 3, lane = threadIdx.x;
  const int x0 = (strip % strips_x) * EW, y0 = (strip / strips_x) * rows;
  const int x = x0 - HALO + lane;
  const bool col_in = x >= 0 && x < a.W, out_lane = lane >= HALO && lane < HALO + EW && x < a.W;
  const int xc = min(max(x, 0), a.W - 1), first = min(max(lane - HALO, 0), EW - 1);
  float ring[11][ESTATS], dm[11], mm[11];
  double se = 0.0, ss = 0.0;
  const auto at = [&](int y) { return (size_t)min(max(y, 0), a.H - 1) * a.W + xc; };  // clamped: always in bounds
  size_t pix = at(y0 - HALO);
  float p_next = a.pred[pix * 4 + c];
  uint32_t g_next = a.gt[pix];
  const int steps = rows + 2 * HALO;  // a multiple of 11
  for (int base = 0; base < steps; base += 11) {
#pragma unroll
    for (int j = 0; j < 11; j++) {
      const int r = base + j, y = y0 - HALO + r, buf = r & 1;
      const float p_raw = p_next;
      const uint32_t g_raw = g_next;
      pix = at(y + 1);
      p_next = a.pred[pix * 4 + c];
      g_next = a.gt[pix];
      const bool in = col_in && y >= 0 && y < a.H;
      const float p = in ? eval_pred(p_raw) : 0.f;
      const float g = in ? gt_channel(g_raw, c) : 0.f;
      mm[j] = a.mask_weighted ? gt_channel(g_raw, 3) : 1.f;
      dm[j] = fabsf(p - g) * mm[j];
      s_p[buf][lane] = p;
      s_g[buf][lane] = g;
      __syncthreads();
      float st[ESTATS] = {0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 11; d++) eval_tap(gw_tap(d), s_p[buf][first + d], s_g[buf][first + d], st);
#pragma unroll
      for (int k = 0; k < ESTATS; k++) ring[j][k] = st[k];
      if (r < 2 * HALO) continue;
      const int yo = y - HALO;
      if (yo >= a.H) continue;
#pragma unroll
      for (int k = 0; k < ESTATS; k++) st[k] = 0.f;
#pragma unroll
      for (int d = 0; d < 11; d++) {
        const float w = gw_tap(d);
#pragma unroll
        for (int k = 0; k < ESTATS; k++) st[k] = __builtin_fmaf(w, ring[(j + 1 + d) % 11][k], st[k]);  // oldest row first
      }
      const int slot = (j + 6) % 11;  // row yo
      if (out_lane) {
        se += (double)(dm[slot] * dm[slot]);
        ss += (double)(eval_ssim(st) * mm[slot]);
      }
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    se += __shfl_xor(se, o);
    ss += __shfl_xor(ss, o);
  }
  if (lane == 0) {
    a.partials[2 * (size_t)item] = (float)se;
    a.partials[2 * (size_t)item + 1] = (float)ss;
  }
}

// The partials hold one entry per channel and tile.
int eval_tiles(int W, int H) { return ((W + ET - 1) / ET) * ((H + ET - 1) / ET); }

// Rows of a strip, so that with its halo it walks whole rings of 11: as few walked rows as possible
// while at most two waves a SIMD (2048 on the 1024 SIMDs) run, whose rows then cost their latency, beyond that the least
// waves times rows. 23 rows at least, so strips never outnumber the 16x16 tiles that size the partials. 0: the tile
// kernel, where a tile, as long as 50 of those waves times rows, makes it the faster one. Tiles against strips:
// 7.1 and 21.3 us at 64x64, 13.3 and 21.8 us at 400x400, 20.7 and 22.0 us at 768x432 (1296 tiles); 23.6 and 22.1 us at
// 640x640 (1600), 68.7 and 38.7 us at 1600x900; 27.3 and 36.5 us at 16x30000, whose strips are 16 of 54 columns wide.
int eval_strip_rows(int W, int H) {
  const long strips_x = (W + EW - 1) / EW, resident = 2048;
  int best = 0;
  long best_cost = 50L * eval_tiles(W, H);
  for (int rows = 23; rows <= 122; rows += 11) {
    const long cost = std::max(strips_x * ((H + rows - 1) / rows) * 3, resident) * (rows + 2 * HALO);
    if (cost < best_cost) {
      best_cost = cost;
      best = rows;
    }
  }
  return best;
}

// Fixed-order double-precision sums of `count` partials (every `stride`-th from `first`) times `factor`,
// added to accum[slot]; with two = 1 also the interleaved second value into accum[slot + 1].
__global__ void __launch_bounds__(1024) aux_reduce_kernel(const float* __restrict__ partials, int count, int two,
                                                          float factor, float* __restrict__ accum, int slot) {
  __shared__ double s_red[2][16];
  double acc0 = 0.0, acc1 = 0.0;
  const int stride = two ? 2 : 1;
  for (int i = threadIdx.x; i < count; i += 1024) {
    acc0 += (double)partials[(size_t)i * stride];
    if (two) acc1 += (double)partials[(size_t)i * stride + 1];
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    acc0 += __shfl_xor(acc0, o);
    acc1 += __shfl_xor(acc1, o);
  }
  if ((threadIdx.x & 63) == 0) {
    s_red[0][threadIdx.x >> 6] = acc0;
    s_red[1][threadIdx.x >> 6] = acc1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double t0 = 0.0, t1 = 0.0;
    for (int k = 0; k < 16; k++) {
      t0 += s_red[0][k];
      t1 += s_red[1][k];
    }
    accum[slot] = (float)((double)accum[slot] + (double)factor * t0);
    if (two) accum[slot + 1] = (float)((double)accum[slot + 1] + (double)factor * t1);
  }
}

int aux_grid(int npix) {
  const int blocks = (npix + AUX_BLOCK - 1) / AUX_BLOCK;
  return blocks < AUX_GRID_MAX ? blocks : AUX_GRID_MAX;
}

}  // namespace
}  // namespace dev
}  // namespace b2c

using namespace b2c::dev;

extern "C" size_t b2c_aux_partials(int W, int H) {
  if (W <= 0 || H <= 0) return 0;
  const size_t ev = (size_t)2 * 3 * (size_t)eval_tiles(W, H);
  return ev > (size_t)AUX_GRID_MAX ? ev : (size_t)AUX_GRID_MAX;
}

extern "C" int b2c_hip_normal_loss(const b2c_normal_loss_args* a, hipStream_t stream) {
  const int npix = a->W * a->H;
  if (npix <= 0) return 0;
  if (!a->feat || !a->normals || !a->v_feat || !a->loss_accum || !a->partials) return (int)hipErrorInvalidValue;
  const int grid = aux_grid(npix);
  normal_loss_kernel<<<grid, AUX_BLOCK, 0, stream>>>(*a);
  aux_reduce_kernel<<<1, 1024, 0, stream>>>(a->partials, grid, 0, 1.f, a->loss_accum, 1);
  return (int)hipGetLastError();
}

extern "C" int b2c_hip_hollow_loss(const float* hollow_pen, int W, int H, float lam, float* loss_accum,
                                   float* partials, hipStream_t stream) {
  const int npix = W * H;
  if (npix <= 0) return 0;
  if (!hollow_pen || !loss_accum || !partials) return (int)hipErrorInvalidValue;
  const int grid = aux_grid(npix);
  hollow_sum_kernel<<<grid, AUX_BLOCK, 0, stream>>>(hollow_pen, npix, partials);
  aux_reduce_kernel<<<1, 1024, 0, stream>>>(partials, grid, 0, lam, loss_accum, 0);
  return (int)hipGetLastError();
}

extern "C" int b2c_hip_eval_metrics(const b2c_eval_args* a, hipStream_t stream) {
  if (a->W <= 0 || a->H <= 0) return 0;
  if (!a->pred || !a->gt || !a->loss_accum || !a->partials) return (int)hipErrorInvalidValue;
  const int rows = eval_strip_rows(a->W, a->H);
  int count = eval_tiles(a->W, a->H) * 3;
  if (rows == 0) {
    eval_tile_kernel<<<dim3(count / 3, 3), AUX_BLOCK, 0, stream>>>(*a, (a->W + ET - 1) / ET);
  } else {
    const int strips_x = (a->W + EW - 1) / EW;
    count = strips_x * ((a->H + rows - 1) / rows) * 3;
    eval_kernel<<<8 * ((count + 7) / 8), 64, 0, stream>>>(*a, strips_x, count / 3, rows);
  }
  aux_reduce_kernel<<<1, 1024, 0, stream>>>(a->partials, count, 1, 1.f, a->loss_accum, 4);
  return (int)hipGetLastError();
}
