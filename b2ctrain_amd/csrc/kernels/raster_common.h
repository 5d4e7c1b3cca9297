// Helpers shared by the forward and backward raster kernels.
#pragma once
#include "device_math.h"

namespace b2c {
namespace dev {

// Tile of a workgroup. Workgroups are dispatched round-robin over the 8 XCDs of an MI355X (workgroup b runs on
// XCD b % 8), and each XCD has its own L2. The image is cut into blocks of 4x4 tiles that go to the XCDs in
// turn: a block's tiles share splats through one L2, and every XCD gets its part of the image's dense and empty
// regions. One contiguous band of rows per XCD instead leaves the XCDs of the border rows idle while the
// middle ones work: the raster kernels measured 66 -> 43 us (forward) and 133 -> 96 us (backward) on 100k splats in
// front of an empty background at 800x800, 193 -> 178 and 402 -> 369 us on a full 1M-splat frame at 1080p, 531 ->
// 460 and 803 -> 747 us at 4K with large splats. Single tiles in turn lose some of the L2's sharing (backward 766 us
// in the last), 8x8 blocks balance less well on small images (160 against 153 us at 980x545). Images of fewer
// than 16 blocks per XCD take smaller blocks, down to single tiles. The grid covers whole blocks, a
// multiple of 8 of them; workgroups that land outside the image get tile -1 and return.
constexpr int NUM_XCD = 8;
struct XcdBlocks {
  int log2;     // block edge, log2 of tiles
  int bx, num;  // blocks per row, blocks
};
__host__ __device__ inline XcdBlocks xcd_blocks(int tiles_x, int tiles_y) {
  XcdBlocks b{2, 0, 0};
  while (true) {
    const int r = (1 << b.log2) - 1;
    b.bx = (tiles_x + r) >> b.log2;
    b.num = b.bx * ((tiles_y + r) >> b.log2);
    if (b.log2 == 0 || b.num >= 16 * NUM_XCD) return b;
    b.log2--;
  }
}
__host__ __device__ inline int xcd_grid(int tiles_x, int tiles_y) {
  const XcdBlocks b = xcd_blocks(tiles_x, tiles_y);
  return ((b.num + NUM_XCD - 1) / NUM_XCD * NUM_XCD) << (2 * b.log2);
}
struct TileAt {
  int tile, tx, ty;  // tile = ty tiles_x + tx, or -1 outside the image
};
__host__ __device__ inline TileAt xcd_tile(int workgroup, int tiles_x, int tiles_y) {
  const XcdBlocks b = xcd_blocks(tiles_x, tiles_y);
  const int k = workgroup / NUM_XCD;  // the k-th workgroup of its XCD: tile `in` of the XCD's block k >> 2 log2
  const int blk = (k >> (2 * b.log2)) * NUM_XCD + workgroup % NUM_XCD, in = k & ((1 << (2 * b.log2)) - 1);
  const int by = blk / b.bx;
  TileAt t;
  t.tx = ((blk - by * b.bx) << b.log2) + (in & ((1 << b.log2) - 1));
  t.ty = (by << b.log2) + (in >> b.log2);
  t.tile = t.tx < tiles_x && t.ty < tiles_y ? t.ty * tiles_x + t.tx : -1;
  return t;
}

constexpr float LOG2E = 1.44269504088896341f;

// A fragment's Mahalanobis half-distance sigma = a dx^2 + b dx dy + c dy^2 (a = c00 / 2, b = c01,
// c = c11 / 2; d = pixel centre - splat centre), evaluated as dx (a dx + b dy) + (c dy) dy with two fused
// multiply-adds. The forward, both backward modes and the CPU restatement (oracle/b2c_oracle.c) evaluate
// exactly this sequence, so every fragment's cutoff decision 0 <= sigma <= power agrees everywhere. lin =
// a dx + b dy and cdy = c dy are kept for the backward: d sigma / d dx = lin + a dx, d sigma / d dy =
// b dx + 2 cdy.
struct FragGeom {
  float dx, dy, lin, cdy, sigma;
};

__device__ __forceinline__ FragGeom frag_geom(float mx, float my, float a, float b, float c, float pcx, float pcy) {
#pragma clang fp contract(off)
  FragGeom f;
  f.dx = pcx - mx;
  f.dy = pcy - my;
  f.lin = __builtin_fmaf(a, f.dx, b * f.dy);
  f.cdy = c * f.dy;
  f.sigma = __builtin_fmaf(f.dx, f.lin, f.cdy * f.dy);
  return f;
}

// A fragment's sigma as a quadratic in the pixel centre's offset (u, v) from its tile's centre: with
// (mxr, myr) the splat centre relative to the tile centre and a = c00 / 2, b = c01, c = c11 / 2,
//   sigma = a (u - mxr)^2 + b (u - mxr)(v - myr) + c (v - myr)^2 = a uu + b uv + c vv + D u + E v + F,
// D = -(2a mxr + b myr), E = -(b mxr + 2c myr) and F the sigma at the tile centre (frag_geom's arithmetic at
// dx = -mxr, dy = -myr). D, E and F are formed once per (splat, tile); a pixel then costs five fused
// multiply-adds (u, v, uu, uv, vv are exact: u, v are +-0.5 .. +-3.5). Every kernel that tests or replays a
// fragment (forward, both backward modes, evidence, depth probe) and the CPU restatement evaluate exactly
// these operations, so all of them agree on which fragments pass. Rounding can leave sigma slightly
// negative where the exact value is 0 (a pixel centre on the splat centre): a fragment passes when
// sigma <= power, which keeps it, as the exact value would.
struct PixelPoly {
  float u, v, uu, uv, vv;
};

__device__ __forceinline__ PixelPoly pixel_poly(float u, float v) { return PixelPoly{u, v, u * u, u * v, v * v}; }

__device__ __forceinline__ float3 sigma_coefs(float mx, float my, float a, float b, float c, float tcx, float tcy) {
#pragma clang fp contract(off)
  const float mxr = mx - tcx, myr = my - tcy;
  const float D = -__builtin_fmaf(a + a, mxr, b * myr);
  const float E = -__builtin_fmaf(b, mxr, (c + c) * myr);
  const float F = __builtin_fmaf(mxr, __builtin_fmaf(a, mxr, b * myr), (c * myr) * myr);
  return make_float3(D, E, F);
}

__device__ __forceinline__ float poly_sigma(float a, float b, float c, float D, float E, float F, const PixelPoly& pp) {
  return __builtin_fmaf(a, pp.uu, __builtin_fmaf(b, pp.uv, __builtin_fmaf(c, pp.vv,
                                                 __builtin_fmaf(D, pp.u, __builtin_fmaf(E, pp.v, F)))));
}

// e^-sigma on the hardware exponential (v_exp_f32 is 2^x): the Gaussian factor of the opacity gradient.
__device__ __forceinline__ float gauss_weight(float sigma) { return __builtin_amdgcn_exp2f(sigma * -LOG2E); }

// log2 of a splat's opacity, precomputed once per splat for fragment_alpha.
__device__ __forceinline__ float log2_opacity(float opacity) { return __builtin_amdgcn_logf(opacity); }

// Unclamped alpha of a fragment, opacity * e^-sigma, as 2^(log2(opacity) - sigma log2 e): one fma and one
// v_exp_f32. Forward and backward must use this same expression: the backward recovers the forward's
// transmittance by dividing by (1 - alpha).
__device__ __forceinline__ float fragment_alpha(float sigma, float log2_op) {
  return __builtin_amdgcn_exp2f(__builtin_fmaf(sigma, -LOG2E, log2_op));
}

// Hollow loss (splat_math.cuh:14-17): a fragment at camera depth z behind a pixel's reference surface
// z_ref is penalised by h = clamp((z - z_ref - margin) / margin, 0, 1) (margin floored at 1e-4), and 0 when
// that quotient is not finite (no surface: z_ref = +inf). Evaluated as (z - (z_ref + margin)) / margin with
// the reciprocal taken once per pixel: the same value up to rounding, and the same bits in the forward,
// both backward modes and the CPU restatement.
struct HollowRef {
  float zm, inv_m;  // z_ref + margin, 1 / max(margin, 1e-4)
};
__device__ __forceinline__ HollowRef hollow_ref(float z_ref, float margin) {
  return HollowRef{z_ref + margin, 1.f / fmaxf(margin, 1e-4f)};
}
__device__ __forceinline__ float hollow_h(float z, HollowRef h) {
  const float d = (z - h.zm) * h.inv_m;
  return __builtin_isfinite(d) ? fminf(fmaxf(d, 0.f), 1.f) : 0.f;
}

// Sum of the magnitudes of the terms of poly_sigma, an upper bound over the tile's pixels (F, 3.5 |D|, 3.5 |E| and
// 12.25 (a + |b| + c), with F, D, E bounded term by term; mxr, myr: distance of the splat centre from the tile's).
// 1e-5 of it is far above the rounding of sigma.
__device__ __forceinline__ float sigma_scale(float mxr, float myr, float ah, float b, float ch) {
  const float bb = fabsf(b);
  return ((ah * mxr + bb * myr) * mxr + ch * myr * myr) + 3.5f * ((2.f * ah + bb) * mxr + (bb + 2.f * ch) * myr) +
         12.25f * (ah + bb + ch);
}

// Quadrant culling. A raster wave covers an 8x8 tile as four 4x4 quadrants of 16 lanes; q[2 qy + qx] is set when
// the splat's ellipse {sigma <= power} can reach a pixel centre of quadrant (qx, qy).
// sigma = ah dx^2 + ch dy^2 + b dx dy (ah = c00 / 2, ch = c11 / 2) is convex, so its minimum over the box
// spanned by the quadrant's pixel centres is 0 when the splat's centre lies inside and is otherwise attained on an
// edge that the centre lies beyond (sigma falls along the segment from the minimising point to the centre, so that
// segment leaves the box there). So the box is reached exactly if its vertical line nearest to the centre is, or
// its horizontal one; a line that passes through the centre lies inside the box and only adds a true answer.
// On the vertical line dx = xe, sigma = ch (dy - ky xe)^2 + qv xe^2 with ky = -b / 2 ch, qv = ah - b^2 / 4 ch: the
// ellipse meets it in |dy - ky xe| <= r = sqrt((power - qv xe^2) / ch), and the box's stretch of it, 3 long, if its
// middle is within r + 1.5. A negative radicand gives NaN, and the comparison no. Both quadrants on a line share r,
// so a splat takes 4 square roots and 8 comparisons. The clamped minimum on each quadrant's edges took about twice
// the operations, and the test was a quarter of the forward's arithmetic: 174 -> 162 us on 1M splats at 1080p, 457 ->
// 432 us at 4K with large splats, 122 -> 116 us with normals at 1237x822, 42.6 -> 39.9 us at 800x800.
// Rounding: power is raised by 2e-5 of the sum of the term magnitudes over the tile (sigma_scale). Half of it covers
// poly_sigma's own rounding. The rest raises r by 1e-5 scale / (ch r) or more; scale / ch is at least
// y^2 + (ky xe)^2 (y: the stretch's farther end), so next to the boundary that is 5e-6 (y + |ky xe|), against at most
// 1e-6 (y + |ky xe|) of rounding in the middle, ky xe, r and their difference. So a quadrant is dropped only when no
// pixel of it can pass the cutoff. A fragment in a dropped quadrant would have had alpha = 0, so culling changes no
// result. Degenerate conics and a non-finite centre keep every quadrant. (x0, y0) is the tile's first
// pixel centre.
struct Quadrants {
  bool q[4];
};

__device__ __forceinline__ Quadrants quadrant_reach(float mx, float my, float ah, float b, float ch, float power,
                                                    float x0, float y0) {
  const float ra = __builtin_amdgcn_rcpf(ah + ah), rc = __builtin_amdgcn_rcpf(ch + ch);
  const float ky = -b * rc, kx = -b * ra;  // minimising dy for a given dx, and dx for dy
  const float qv = __builtin_fmaf(0.5f * b, ky, ah), qh = __builtin_fmaf(0.5f * b, kx, ch);
  const float dx0 = x0 - mx, dy0 = y0 - my;
  const float scale = sigma_scale(fabsf(dx0 + 3.5f), fabsf(dy0 + 3.5f), ah, b, ch);
  const float pw = __builtin_fmaf(2e-5f, scale, power);
  const bool all = !(ah > 0.f && ch > 0.f) || !(fabsf(scale + (qv + qh)) < __builtin_inff());
  Quadrants m;
#pragma unroll
  for (int k = 0; k < 4; k++) m.q[k] = all;
#pragma unroll
  for (int k = 0; k < 2; k++) {
    const float xlo = dx0 + 4.f * k, ylo = dy0 + 4.f * k;
    const float xe = __builtin_amdgcn_fmed3f(xlo, xlo + 3.f, 0.f), ye = __builtin_amdgcn_fmed3f(ylo, ylo + 3.f, 0.f);
    const float rv = __builtin_amdgcn_sqrtf(__builtin_fmaf(-qv * xe, xe, pw) * (rc + rc)) + 1.5f;
    const float rh = __builtin_amdgcn_sqrtf(__builtin_fmaf(-qh * ye, ye, pw) * (ra + ra)) + 1.5f;
    const float cv = __builtin_fmaf(ky, xe, -1.5f - dy0), chz = __builtin_fmaf(kx, ye, -1.5f - dx0);
#pragma unroll
    for (int o = 0; o < 2; o++) {
      m.q[2 * o + k] |= fabsf(cv - 4.f * o) <= rv;   // column k, rows of quadrant o
      m.q[2 * k + o] |= fabsf(chz - 4.f * o) <= rh;  // row k, columns of quadrant o
    }
  }
  return m;
}

// The lanes of `m` below this one.
__device__ __forceinline__ uint32_t lanes_before(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Per-quadrant lists of a batch: the byte offsets (16 lane) of the lanes whose splat reaches the quadrant, in lane
// (depth) order, padded with the null splat 64. Returns the longest list's length.
template <typename List>
__device__ __forceinline__ uint32_t quadrant_lists(const Quadrants& reach, int lane, List& s_list) {
  uint32_t longest = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const uint64_t m = ballot64(reach.q[q]);
    const uint32_t c = popc64(m);
    if (reach.q[q]) s_list[q][lanes_before(m)] = (uint32_t)lane * 16u;
    if ((uint32_t)lane >= c) s_list[q][lane] = 64u * 16u;
    longest = max(longest, c);
  }
  return __builtin_amdgcn_readfirstlane(longest);
}

// Whether a fragment of this splat in the tile could reach the alpha cap: log2 alpha is log2 opacity - sigma
// log2 e, and sigma, 0 or more exactly, rounds no further below 0 than 1e-5 of the quadratic's term magnitudes
// over the tile (sigma_scale). -0.0015 lies below log2 0.999 by 30 roundings of the exponent. Anything
// not finite counts as possible.
__device__ __forceinline__ bool clamp_possible(float mx, float my, float ah, float b, float ch, float log2_op, float tcx,
                                               float tcy) {
  return !(log2_op + (1e-5f * LOG2E) * sigma_scale(fabsf(mx - tcx), fabsf(my - tcy), ah, b, ch) < -0.0015f);
}

// DPP controls (GCN/CDNA): row_shr:n = 0x110 + n, row_ror:n = 0x120 + n, row_bcast:15 = 0x142,
// row_bcast:31 = 0x143, wave_shl:1 = 0x130, wave_shr:1 = 0x138. Lanes whose source is outside the row mask or
// the wave get `fill`.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t x, uint32_t fill) {
  return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)x, CTRL, ROW_MASK, 0xF, false);
}

constexpr uint32_t NO_RUN = 0xFFFFFFFFu;  // the run id of a lane outside every run

// One Hillis-Steele step of a segmented inclusive scan across the wave: add the partial of the DPP source
// lane when it lies in the same run (runs are contiguous, so equal ids at both ends mean no run boundary in
// between). Each value takes one v_fmac_f32 whose first operand is read through the DPP shift: v += m * v[src],
// with m = 1 when the source lane lies in the same run (and, for the row broadcasts, in a row the step
// feeds) and 0 otherwise; a lane whose source is outside its row or the wave reads 0 (bound_ctrl). Adding
// m * t with m in {0, 1} rounds exactly as the plain sum does. One asm block holds the step's values in a
// fixed order, so a value's DPP read comes at least NV - 1 instructions after the previous step wrote it;
// the leading s_nop gives the two wait states a DPP read needs after a VALU write of its source for the
// first step.
#define B2C_FD(i, C) "v_fmac_f32_dpp %" #i ", %" #i ", %[m] " C " row_mask:0xf bank_mask:0xf bound_ctrl:1\n\t"
#define B2C_FD3(C) B2C_FD(0, C) B2C_FD(1, C) B2C_FD(2, C)
#define B2C_FD11(C) \
  B2C_FD3(C) B2C_FD(3, C) B2C_FD(4, C) B2C_FD(5, C) B2C_FD(6, C) B2C_FD(7, C) B2C_FD(8, C) B2C_FD(9, C) B2C_FD(10, C)
#define B2C_FD14(C) B2C_FD11(C) B2C_FD(11, C) B2C_FD(12, C) B2C_FD(13, C)
#define B2C_OP3(v) "+v"(v[0]), "+v"(v[1]), "+v"(v[2])
#define B2C_OP11(v) \
  B2C_OP3(v), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]), "+v"(v[8]), "+v"(v[9]), "+v"(v[10])
#define B2C_OP14(v) B2C_OP11(v), "+v"(v[11]), "+v"(v[12]), "+v"(v[13])
#define B2C_SEG_STEP(C)                                                                      \
  do {                                                                                       \
    if constexpr (NV == 3)                                                                   \
      asm("s_nop 1\n\t" B2C_FD3(C) : B2C_OP3(v) : [m] "v"(m));                               \
    else if constexpr (NV == 11)                                                             \
      asm("s_nop 1\n\t" B2C_FD11(C) : B2C_OP11(v) : [m] "v"(m));                             \
    else                                                                                     \
      asm("s_nop 1\n\t" B2C_FD14(C) : B2C_OP14(v) : [m] "v"(m));                             \
  } while (0)

// m for one step: 1 where the DPP source lane holds the same run id (and the lane lies in a row the step
// feeds), else 0.
template <int CTRL>
__device__ __forceinline__ float seg_scan_m(uint32_t id, bool row_ok) {
  const uint32_t src = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)id, CTRL, 0xF, 0xF, true);
  return (row_ok && src == id) ? 1.f : 0.f;
}

template <int NV>
__device__ __forceinline__ void seg_scan(uint32_t id, float (&v)[NV]) {
  static_assert(NV == 3 || NV == 11 || NV == 14, "the scan's asm steps cover 3, 11 and 14 values");
  const int lane = (int)__lane_id();
  float m;
  m = seg_scan_m<0x111>(id, true);  // row_shr:1
  B2C_SEG_STEP("row_shr:1");
  m = seg_scan_m<0x112>(id, true);  // row_shr:2
  B2C_SEG_STEP("row_shr:2");
  m = seg_scan_m<0x114>(id, true);  // row_shr:4
  B2C_SEG_STEP("row_shr:4");
  m = seg_scan_m<0x118>(id, true);  // row_shr:8
  B2C_SEG_STEP("row_shr:8");
  m = seg_scan_m<0x142>(id, (lane & 16) != 0);  // row_bcast:15 into rows 1 and 3
  B2C_SEG_STEP("row_bcast:15");
  m = seg_scan_m<0x143>(id, (lane & 32) != 0);  // row_bcast:31 into rows 2 and 3
  B2C_SEG_STEP("row_bcast:31");
}
#undef B2C_SEG_STEP
#undef B2C_OP14
#undef B2C_OP11
#undef B2C_OP3
#undef B2C_FD14
#undef B2C_FD11
#undef B2C_FD3
#undef B2C_FD

}  // namespace dev
}  // namespace b2c
