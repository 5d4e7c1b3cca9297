// Consumers of the tile lists (replaces src/train/evidence.cu:47-183 and src/gpu/probe.cu:7-53): per-view
// evidence (each splat's front-to-back weight on the view's pixels, split by the pixel's mask, residual and
// loss weight), the per-class label vote, and the per-pixel depth probe. They reuse the render's bit-exact
// lists and, for the evidence, the forward's last_idx: one wave64 per 8x8 tile, one lane per pixel, the
// list staged through LDS 64 splats at a time, the same sigma, cutoff and alpha as the forward kernel, so a
// replayed fragment carries exactly the blend weight the render gave it.
#include "b2c_kernels.h"
#include "raster_common.h"

namespace b2c {
namespace dev {
namespace {

constexpr int VSTRIDE = 68;  // row stride of the [splat][pixel] weight matrix in LDS (16-byte rows; a row's
                             // 16-byte reads by consecutive lanes start 4 banks apart)
constexpr uint32_t LABEL_NONE = 0xFFFFFFFFu;  // a pixel that takes no part in the label vote

__device__ __forceinline__ float byte_chan(uint32_t p, int c) { return (float)((p >> (8 * c)) & 0xffu) * (1.f / 255.f); }

// Evidence and label vote of one view. Per pixel: m = target alpha * weight (the in-mask mass), m * res with
// res the mean absolute colour residual of the render (plus the weighted normal residual with FEAT), and
// k = (target alpha if the view is masked with alpha, else 1) * weight. Each lane replays its pixel's list
// up to last_idx and writes every fragment's blend weight vis into a [16 splats][64 pixels] LDS matrix; after each
// group of 16 splats lane 16 q + j contracts pixels 16 q .. 16 q + 15 of splat j's row with the pixel vectors (m, m res,
// k), whose 16 entries it keeps in registers for the whole tile, the four quarters are added and the sums stored as the
// (tile, splat) row at the entry's emit position (the reference adds them to the splat with float atomics,
// which MI355X performs past the per-XCD L2; evidence_reduce_kernel sums each splat's rows instead). With
// LABELS the tile's distinct classes are found once (ballots: labels are spatially coherent, a tile usually
// holds one or two), each with a pixel vector k * [pixel in the class]; the same rows are contracted with
// those vectors and added to the splat's class bins with float atomics. Classes beyond the first MAXC of a
// tile take a sum masked by class each, over the same quarters (the classes of a lane's quarter of the pixels are four
// registers of bytes): a pass with labels over 200k splats at 800x800 takes 622 us with classes of 5x5 pixels and 1916 us
// with a class for every pixel, against 1206 and 5187 us where 16 lanes walk the pixels of a class one by one.
// With all 64 splats of a batch in the matrix (17 KB) a CU held 9 waves, and every
// lane read the three pixel vectors from LDS for each row: 125 -> 92 us a 960x720 view with labels.
constexpr int EG = 16;   // splats per group
constexpr int MAXC = 4;  // classes per tile with their own pixel vector

// The sum over the wave's four 16-lane rows, in every lane.
__device__ __forceinline__ float sum_quarters(float x) {
  x += __shfl_xor(x, 16);
  return x + __shfl_xor(x, 32);
}

template <bool FEAT, bool LABELS>
__global__ void __launch_bounds__(64) evidence_kernel(b2c_evidence_args a) {
  __shared__ float4 s_g0[64], s_g1[64];
  __shared__ uint32_t s_id[64];
  __shared__ __attribute__((aligned(16))) float s_vis[EG * VSTRIDE];
  __shared__ __attribute__((aligned(16))) float s_kc[LABELS ? MAXC : 1][64];  // k of the tile's c-th class's pixels, else 0
  __shared__ uint32_t s_slot[64];
  const TileAt here = xcd_tile(blockIdx.x, a.tiles_x, a.tiles_y);
  const int tile = here.tile;
  if (tile < 0) return;
  const uint2 range = reinterpret_cast<const uint2*>(a.tile_ranges)[tile];
  const int lane = threadIdx.x;
  float4* rows = reinterpret_cast<float4*>(a.rows);
  // entries past the shrunk end composited nowhere: they get no row (the sum reads a row without this
  // pass's tag as zero)
  if (range.y <= range.x) return;
  const int px = here.tx * RT_W + (lane & 7), py = here.ty * RT_W + (lane >> 3);
  const bool inside = px < a.W && py < a.H;
  const float pcx = px + 0.5f, pcy = py + 0.5f;
  const float tcx = here.tx * RT_W + RT_W * 0.5f, tcy = here.ty * RT_W + RT_W * 0.5f;
  const PixelPoly pp = pixel_poly(pcx - tcx, pcy - tcy);
  float m = 0.f, mres = 0.f, k = 0.f;
  uint32_t last = range.x, lab = LABEL_NONE;
  if (inside) {
    const int pix = py * a.W + px;
    const uint32_t g = a.gt[pix];
    const float ga = byte_chan(g, 3);
    const float wp = a.weights ? (float)a.weights[pix] * (1.f / 255.f) : 1.f;
    const float4 o = reinterpret_cast<const float4*>(a.out_rgba)[pix];
    float res = (fabsf(o.x - byte_chan(g, 0)) + fabsf(o.y - byte_chan(g, 1)) + fabsf(o.z - byte_chan(g, 2))) * (1.f / 3.f);
    if constexpr (FEAT) {
      const uint32_t gn = a.normals[pix];
      if (((gn >> 24) & 0xffu) > 127u) {  // the normal loss's residual (loss.cu:218-223), weighted
        const float nx = (float)(gn & 0xffu) * (2.f / 255.f) - 1.f;
        const float ny = 1.f - (float)((gn >> 8) & 0xffu) * (2.f / 255.f);
        const float nz = 1.f - (float)((gn >> 16) & 0xffu) * (2.f / 255.f);
        const float4 f = reinterpret_cast<const float4*>(a.out_feat)[pix];
        const float pl = fmaxf(sqrtf(f.x * f.x + f.y * f.y + f.z * f.z), 1e-6f);
        const float nl = fmaxf(sqrtf(nx * nx + ny * ny + nz * nz), 1e-6f);
        const float nres = fabsf(f.x - nx) + fabsf(f.y - ny) + fabsf(f.z - nz) + 1.f - (f.x * nx + f.y * ny + f.z * nz) / (pl * nl);
        res += a.normal_weight * nres;
      }
    }
    m = ga * wp;
    mres = m * res;
    k = (a.masked_has_alpha ? ga : 1.f) * wp;
    last = a.last_idx[pix];
    if constexpr (LABELS) {
      lab = a.labels[pix];
      if (lab >= (uint32_t)B2C_LABEL_BINS || !(k != 0.f)) lab = LABEL_NONE;
    }
  }
  // this lane's quarter of the pixel vectors, through the weight matrix as scratch
  const int ej = lane & (EG - 1), eq = lane >> 4;
  float pm[16], pr[16], pk[16];
  s_vis[lane] = m;
  s_vis[64 + lane] = mres;
  s_vis[128 + lane] = k;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; i++) {
    pm[i] = s_vis[eq * 16 + i];
    pr[i] = s_vis[64 + eq * 16 + i];
    pk[i] = s_vis[128 + eq * 16 + i];
  }
  uint32_t cls[MAXC] = {0u, 0u, 0u, 0u};  // wave-uniform: the tile's first classes, in pixel order
  int ncls = 0;
  uint32_t rest = 0;  // the classes past those, one bit each
  uint32_t pl[4] = {};  // and this lane's quarter of the pixels' class among them, a byte each (LABEL_BINS: none)
  if constexpr (LABELS) {
    uint64_t todo = ballot64(lab != LABEL_NONE);
    int my_c = -1;
    while (todo != 0ull && ncls < MAXC) {
      const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)lab, __builtin_ctzll(todo));
      const uint64_t hit = ballot64(lab == b);
      if (lab == b) my_c = ncls;
      cls[ncls++] = b;
      todo &= ~hit;
    }
#pragma unroll
    for (int c = 0; c < MAXC; c++) s_kc[c][lane] = my_c == c ? k : 0.f;
    const uint32_t mine = my_c < 0 ? min(lab, (uint32_t)B2C_LABEL_BINS) : (uint32_t)B2C_LABEL_BINS;
    while (todo != 0ull) {
      const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)mine, __builtin_ctzll(todo));
      rest |= 1u << b;
      todo &= ~ballot64(mine == b);
    }
    if (rest != 0u) {
      __syncthreads();  // the pixel vectors are read
      reinterpret_cast<uint8_t*>(s_vis)[lane] = (uint8_t)mine;
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 4; i++) pl[i] = reinterpret_cast<const uint32_t*>(s_vis)[eq * 4 + i];
    }
  }
  float T = 1.f;
  for (uint32_t start = range.x; start < range.y; start += 64) {
    const uint32_t count = min(64u, range.y - start);
    __syncthreads();  // the previous batch's LDS is consumed
    if ((uint32_t)lane < count) {
      const uint32_t gid = a.vals_sorted[start + lane];
      s_id[lane] = gid;
      s_slot[lane] = a.slot_sorted[start + lane];
      const float4* rec = reinterpret_cast<const float4*>(a.raster_rec) + (size_t)gid * 4;
      const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
      const float3 def = sigma_coefs(r0.x, r0.y, r0.z, r0.w, r1.x, tcx, tcy);
      s_g0[lane] = make_float4(def.x, def.y, def.z, r0.z);
      s_g1[lane] = make_float4(r0.w, r2.w, r1.z, r1.x);  // (c01, log2 opacity, power, c11 / 2)
    } else {  // null splats: power = 0 and sigma = F = 1 fails the cutoff
      s_g0[lane] = make_float4(0.f, 0.f, 1.f, 0.f);
      s_g1[lane] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
    for (uint32_t g = 0; g < count; g += EG) {
      // entries before this pixel's last composited one, relative to the group (outside the image: none)
      const int last_rel = (int)(last - start) - (int)g;
#pragma unroll
      for (int j = 0; j < EG; j++) {
        const float4 g0 = s_g0[g + j], g1 = s_g1[g + j];
        const float sigma = poly_sigma(g0.w, g1.x, g1.w, g0.x, g0.y, g0.z, pp);
        const bool valid = (j < last_rel) & (sigma <= g1.z);
        const float alpha = valid ? fminf(ALPHA_MAX, fragment_alpha(sigma, g1.y)) : 0.f;
        const float vis = alpha * T;
        T = __builtin_fmaf(-alpha, T, T);  // as the forward rounds it
        s_vis[j * VSTRIDE + lane] = vis;
      }
      __syncthreads();
      const float* row = s_vis + ej * VSTRIDE;
      const float4* part = reinterpret_cast<const float4*>(row + eq * 16);
      const uint32_t e = g + ej;  // this lane's entry of the batch
      float a0 = 0.f, a1 = 0.f, a2 = 0.f;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float4 v = part[i];
        const float x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int c = 0; c < 4; c++) {
          a0 += x[c] * pm[4 * i + c];
          a1 += x[c] * pr[4 * i + c];
          a2 += x[c] * pk[4 * i + c];
        }
      }
      a0 = sum_quarters(a0);
      a1 = sum_quarters(a1);
      a2 = sum_quarters(a2);
      if (eq == 0 && e < count) rows[s_slot[e]] = make_float4(a0, a1, a2, __uint_as_float(a.row_tag));
      if constexpr (LABELS) {
        float* bins = a.label_acc + (size_t)s_id[min(e, count - 1u)] * B2C_LABEL_BINS;
#pragma unroll
        for (int c = 0; c < MAXC; c++) {
          if (c >= ncls) break;  // wave-uniform
          float sum = 0.f;
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float4 v = part[i], k4 = reinterpret_cast<const float4*>(s_kc[c] + eq * 16)[i];
            sum += v.x * k4.x; sum += v.y * k4.y; sum += v.z * k4.z; sum += v.w * k4.w;
          }
          sum = sum_quarters(sum);
          if (eq == 0 && e < count && sum != 0.f) atomicAdd(bins + cls[c], sum);
        }
        for (uint32_t left = rest; left != 0u; left &= left - 1u) {  // wave-uniform
          const uint32_t b = (uint32_t)__builtin_ctz(left);
          float sum = 0.f;
#pragma unroll
          for (int i = 0; i < 16; i++) sum += ((pl[i / 4] >> (8 * (i % 4))) & 0xFFu) == b ? row[eq * 16 + i] * pk[i] : 0.f;
          sum = sum_quarters(sum);
          if (eq == 0 && e < count && sum != 0.f) atomicAdd(bins + b, sum);
        }
      }
      __syncthreads();  // the group's rows are consumed
    }
  }
}

// The view's per-splat sums: one lane per emit position, a segmented inclusive scan across the wave over
// the splat ids of the emit order (a splat's rows are contiguous), and the last lane of each run piece adds
// the piece's sums to the splat's view accumulator (one float atomic per piece and value: about one per
// splat instead of one per (tile, splat) pair).
__global__ void __launch_bounds__(256) evidence_reduce_kernel(b2c_evidence_sum_args a) {
  const uint32_t s = blockIdx.x * 256u + threadIdx.x;
  const bool valid = s < a.m;
  const uint32_t id = valid ? a.ids[s] : NO_RUN;
  float v[3] = {0.f, 0.f, 0.f};
  const float4 r = reinterpret_cast<const float4*>(a.rows)[valid ? s : 0u];
  if (valid && __float_as_uint(r.w) == a.row_tag) {  // another tag: past its tile's shrunk end, zero
    v[0] = r.x;
    v[1] = r.y;
    v[2] = r.z;
  }
  seg_scan(id, v);
  const uint32_t next = dpp_u32<0x130, 0xF>(id, NO_RUN);  // wave_shl:1: the next lane's id (lane 63: none)
  if (valid && next != id && id < (uint32_t)a.n) {
    float* dst = a.view_acc + (size_t)id * 3;
#pragma unroll
    for (int k = 0; k < 3; k++)
      if (v[k] != 0.f) atomicAdd(dst + k, v[k]);
  }
}

// fold_view_kernel (evidence.cu:114-126): the view's sums into the running evidence: w_in, w_all, err, the
// sum of w_in^2 (for the effective view count) and the w_in-weighted unit direction towards the camera.
__global__ void __launch_bounds__(256) fold_view_kernel(b2c_evidence_sum_args a) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n) return;
  const float w_in = a.view_acc[(size_t)i * 3], err = a.view_acc[(size_t)i * 3 + 1], w_all = a.view_acc[(size_t)i * 3 + 2];
  float* e = a.evidence + (size_t)i * B2C_EVIDENCE_STRIDE;
  e[0] += w_in;
  e[1] += w_all;
  e[2] += err;
  e[7] += w_in * w_in;
  if (w_in != 0.f) {
    const float4 p = reinterpret_cast<const float4*>(a.pos_op)[i];
    const float dx = a.cam_pos[0] - p.x, dy = a.cam_pos[1] - p.y, dz = a.cam_pos[2] - p.z;
    const float il = 1.f / fmaxf(sqrtf(dx * dx + dy * dy + dz * dz), 1e-12f);
    e[4] += w_in * dx * il;
    e[5] += w_in * dy * il;
    e[6] += w_in * dz * il;
  }
}

// The rows download_evidence hands out ([n][7]: w_in, w_all, err, the participation ratio w_in^2 / sum w_in^2 of the
// views' in-mask mass, direction xyz), from the accumulator's 8 floats per splat. Formed here rather than on the
// host: 28 of 32 bytes per splat cross the link and no host loop follows. A thread owns one splat (two 16-byte
// loads); the workgroup's rows go out through LDS as one contiguous stretch.
constexpr int EXPORT_BLOCK = 256;
__global__ void __launch_bounds__(EXPORT_BLOCK) evidence_export_kernel(int n, const float* __restrict__ acc,
                                                                       float* __restrict__ out) {
#pragma clang fp contract(off)
  __shared__ float s_row[EXPORT_BLOCK * 7];
  const int i0 = blockIdx.x * EXPORT_BLOCK, i = i0 + threadIdx.x;
  if (i < n) {
    const float4 a = reinterpret_cast<const float4*>(acc)[(size_t)i * 2], b = reinterpret_cast<const float4*>(acc)[(size_t)i * 2 + 1];
    float* e = s_row + threadIdx.x * 7;
    e[0] = a.x;
    e[1] = a.y;
    e[2] = a.z;
    e[3] = b.w > 0.f ? (a.x * a.x) / b.w : 0.f;
    e[4] = b.x;
    e[5] = b.y;
    e[6] = b.z;
  }
  __syncthreads();
  const int count = min(EXPORT_BLOCK, n - i0) * 7;
  for (int j = threadIdx.x; j < count; j += EXPORT_BLOCK) out[(size_t)i0 * 7 + j] = s_row[j];
}

// The label vote download_labels hands out ([n][2]: the first class with the largest vote, and its share of the
// votes; zeros without votes), so 8 instead of 128 bytes per splat cross the link (200k splats: 25.6 MB and a
// host loop took 5.4 ms, this 0.2 ms). The votes are summed in class order, as a serial walk would.
__global__ void __launch_bounds__(EXPORT_BLOCK) label_export_kernel(int n, const float* __restrict__ acc,
                                                                    float* __restrict__ out) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * EXPORT_BLOCK + threadIdx.x;
  if (i >= n) return;
  const float4* a = reinterpret_cast<const float4*>(acc) + (size_t)i * (B2C_LABEL_BINS / 4);
  float4 v[B2C_LABEL_BINS / 4];
#pragma unroll
  for (int q = 0; q < B2C_LABEL_BINS / 4; q++) v[q] = a[q];
  float total = 0.f, best = 0.f;
  int win = 0;
#pragma unroll
  for (int k = 0; k < B2C_LABEL_BINS; k++) {
    const float4 q = v[k / 4];
    const float x = k % 4 == 0 ? q.x : (k % 4 == 1 ? q.y : (k % 4 == 2 ? q.z : q.w));
    total = total + x;
    if (x > best) {
      best = x;
      win = k;
    }
  }
  reinterpret_cast<float2*>(out)[i] = total > 0.f ? make_float2((float)win, best / total) : make_float2(0.f, 0.f);
}

// Depth probe (probe.cu:7-53) over the full lists of a projected and binned view: per pixel the accumulated
// alpha, the depth at which it first reaches tau (tau <= 0: the alpha-weighted mean depth, when the pixel is
// more than 5% covered), the weight arriving from more than delta behind that first surface, and the weight
// from more than margin behind the reference depth (if given). The transmittance stop ends a pixel as in the
// forward, and the walk is the forward's: per 4x4 quadrant lists of each batch (a splat whose ellipse cannot
// reach a quadrant composites nothing there), two list entries per step, no branch per fragment.
__global__ void __launch_bounds__(64) probe_kernel(b2c_probe_args a) {
  // lanes by quadrant as in the forward: lane 16 q + p is pixel p (row-major 4x4) of quadrant q; slot 64
  // is a null splat that pads the shorter quadrant lists
  __shared__ float4 s_g0[65], s_g1[65];
  __shared__ float s_z[65];  // camera depth
  __shared__ uint32_t s_list[4][66];  // per quadrant: LDS byte offsets of its splats, in depth order
  const TileAt here = xcd_tile(blockIdx.x, a.tiles_x, a.tiles_y);
  const int tile = here.tile;
  if (tile < 0) return;
  const uint2 range = reinterpret_cast<const uint2*>(a.tile_ranges)[tile];
  const int lane = threadIdx.x;
  const int q = lane >> 4, p = lane & 15;
  const int tx = here.tx, ty = here.ty;
  const int px = tx * RT_W + (q & 1) * 4 + (p & 3), py = ty * RT_W + (q >> 1) * 4 + (p >> 2);
  const float x0 = tx * RT_W + 0.5f, y0 = ty * RT_W + 0.5f;  // the tile's first pixel centre
  const bool inside = px < a.W && py < a.H;
  const float pcx = px + 0.5f, pcy = py + 0.5f;
  const float tcx = tx * RT_W + RT_W * 0.5f, tcy = ty * RT_W + RT_W * 0.5f;  // the tile centre
  const PixelPoly pp = pixel_poly(pcx - tcx, pcy - tcy);
  const bool mean_mode = a.tau <= 0.f;
  float T = 1.f, z_first = __builtin_inff(), deep = 0.f, behind = 0.f, zsum = 0.f;
  const float zr = (inside && a.ref_z) ? a.ref_z[py * a.W + px] : __builtin_inff();
  bool live = inside;
  if (lane < 8) s_list[lane >> 1][64 + (lane & 1)] = 64u * 16u;  // read by the last pair's prefetch
  if (lane == 0) {  // power = 0 and sigma = F = 1: fails the cutoff
    s_g0[64] = make_float4(0.f, 0.f, 1.f, 0.f);
    s_g1[64] = make_float4(0.f, 0.f, 0.f, 0.f);
    s_z[64] = 0.f;
  }
  const char* lds_g0 = reinterpret_cast<const char*>(s_g0);
  const char* lds_g1 = reinterpret_cast<const char*>(s_g1);
  const char* lds_z = reinterpret_cast<const char*>(s_z);
  for (uint32_t start = range.x; start < range.y; start += 64) {
    if (ballot64(live) == 0ull) break;
    const uint32_t remaining = min(64u, range.y - start);
    __syncthreads();
    Quadrants reach{};
    if ((uint32_t)lane < remaining) {
      const uint32_t gid = a.vals_sorted[start + lane];
      const float4* rec = reinterpret_cast<const float4*>(a.raster_rec) + (size_t)gid * 4;
      const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2], r3 = rec[3];
      const float3 def = sigma_coefs(r0.x, r0.y, r0.z, r0.w, r1.x, tcx, tcy);
      s_g0[lane] = make_float4(def.x, def.y, def.z, r0.z);
      s_g1[lane] = make_float4(r0.w, r2.w, r1.z, r1.x);  // (c01, log2 opacity, power, c11 / 2)
      s_z[lane] = r3.w;
      reach = quadrant_reach(r0.x, r0.y, r0.z, r0.w, r1.x, r1.z, x0, y0);
    }
    const uint32_t n_iter = quadrant_lists(reach, lane, s_list);
    __syncthreads();
    const uint32_t* my_list = s_list[q];
    uint32_t off0 = my_list[0], off1 = my_list[1];
    // One step, straight-line as in the forward: an invalid fragment, a stopped lane or a null splat
    // contributes alpha = 0 and leaves every sum unchanged. A composited fragment (valid and not stopping the
    // lane) adds its weight to the depth sums and may set z_first.
#define B2C_PROBE_STEP(off, next)                                                                       \
  do {                                                                                                  \
    const float4 g0 = *reinterpret_cast<const float4*>(lds_g0 + (off));                                 \
    const float4 g1 = *reinterpret_cast<const float4*>(lds_g1 + (off));                                 \
    const float sigma = poly_sigma(g0.w, g1.x, g1.w, g0.x, g0.y, g0.z, pp);                             \
    const bool valid = live & (sigma <= g1.z);                                                          \
    float a_cl = fminf(ALPHA_MAX, fragment_alpha(sigma, g1.y));                                         \
    asm volatile("" : "+v"(a_cl));                                                                      \
    const float alpha = valid ? a_cl : 0.f;                                                             \
    const float next_T = __builtin_fmaf(-alpha, T, T);                                                       \
    const bool stop = next_T <= T_CUTOFF;                                                               \
    live = live & !stop;                                                                                \
    const bool comp = valid & !stop;                                                                    \
    const float vis = comp ? alpha * T : 0.f;                                                           \
    const float z = *reinterpret_cast<const float*>(lds_z + ((off) >> 2));                              \
    deep += (__builtin_isfinite(z_first) & (z > z_first + a.delta)) ? vis : 0.f;                        \
    behind += (z > zr + a.margin) ? vis : 0.f;                                                          \
    zsum = comp ? fmaf(vis, z, zsum) : zsum;                                                            \
    T = comp ? next_T : T;                                                                              \
    z_first = (comp & !__builtin_isfinite(z_first) & (1.f - T >= a.tau)) ? z : z_first;                \
    (off) = my_list[next];                                                                              \
  } while (0)
    for (uint32_t i = 0; i < n_iter; i += 2) {
      B2C_PROBE_STEP(off0, i + 2);
      B2C_PROBE_STEP(off1, i + 3);
    }
#undef B2C_PROBE_STEP
  }
  if (mean_mode) z_first = (1.f - T) > 0.05f ? zsum / (1.f - T) : __builtin_inff();
  if (inside) reinterpret_cast<float4*>(a.out)[py * a.W + px] = make_float4(1.f - T, z_first, deep, behind);
}

}  // namespace
}  // namespace dev
}  // namespace b2c

using namespace b2c::dev;

extern "C" int b2c_hip_evidence_view(const b2c_evidence_args* a, hipStream_t stream) {
  const int n_tiles = a->tiles_x * a->tiles_y;
  if (n_tiles <= 0) return 0;
  if (!a->raster_rec || !a->rows || !a->slot_sorted || !a->gt || !a->out_rgba || !a->last_idx || a->row_tag == 0u)
    return (int)hipErrorInvalidValue;
  const bool feat = a->normals && a->normal_weight > 0.f;
  const bool labels = a->labels && a->label_acc;
  if (feat && !a->out_feat) return (int)hipErrorInvalidValue;
  const dim3 grid(xcd_grid(a->tiles_x, a->tiles_y)), block(64);
  if (feat) {
    if (labels) evidence_kernel<true, true><<<grid, block, 0, stream>>>(*a);
    else evidence_kernel<true, false><<<grid, block, 0, stream>>>(*a);
  } else {
    if (labels) evidence_kernel<false, true><<<grid, block, 0, stream>>>(*a);
    else evidence_kernel<false, false><<<grid, block, 0, stream>>>(*a);
  }
  return (int)hipGetLastError();
}

extern "C" int b2c_hip_evidence_sum(const b2c_evidence_sum_args* a, hipStream_t stream) {
  if (a->n <= 0) return 0;
  if (!a->ids || !a->rows || !a->view_acc || !a->pos_op || !a->evidence || a->row_tag == 0u)
    return (int)hipErrorInvalidValue;
  const int fill = b2c_hip_fill_u32(reinterpret_cast<uint32_t*>(a->view_acc), 0u, (size_t)a->n * 3, stream);
  if (fill) return fill;
  if (a->m) evidence_reduce_kernel<<<(a->m + 255) / 256, 256, 0, stream>>>(*a);
  fold_view_kernel<<<(a->n + 255) / 256, 256, 0, stream>>>(*a);
  return (int)hipGetLastError();
}

extern "C" int b2c_hip_evidence_export(int n, const float* evidence, float* out, hipStream_t stream) {
  if (n <= 0) return 0;
  if (!evidence || !out || (reinterpret_cast<uintptr_t>(evidence) & 15u)) return (int)hipErrorInvalidValue;
  evidence_export_kernel<<<(n + EXPORT_BLOCK - 1) / EXPORT_BLOCK, EXPORT_BLOCK, 0, stream>>>(n, evidence, out);
  return (int)hipGetLastError();
}

extern "C" int b2c_hip_label_export(int n, const float* label_acc, float* out, hipStream_t stream) {
  if (n <= 0) return 0;
  if (!label_acc || !out || (reinterpret_cast<uintptr_t>(label_acc) & 15u) || (reinterpret_cast<uintptr_t>(out) & 7u))
    return (int)hipErrorInvalidValue;
  label_export_kernel<<<(n + EXPORT_BLOCK - 1) / EXPORT_BLOCK, EXPORT_BLOCK, 0, stream>>>(n, label_acc, out);
  return (int)hipGetLastError();
}

extern "C" int b2c_hip_probe_depth(const b2c_probe_args* a, hipStream_t stream) {
  const int n_tiles = a->tiles_x * a->tiles_y;
  if (n_tiles <= 0) return 0;
  if (!a->raster_rec || !a->out) return (int)hipErrorInvalidValue;
  probe_kernel<<<dim3(xcd_grid(a->tiles_x, a->tiles_y)), dim3(64), 0, stream>>>(*a);
  return (int)hipGetLastError();
}
