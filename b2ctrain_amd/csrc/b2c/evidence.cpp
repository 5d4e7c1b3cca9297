// Evidence pass and depth probe (replaces src/train/evidence.cu:185-266 and src/gpu/probe.cu:47-53): the
// host loop over views and the downloads; the replays are kernels/replay.hip.
#include "evidence.h"

#include <algorithm>

namespace b2c {

namespace {
// Module-level accumulators, as the reference keeps them (evidence.cu:22-23, 38-39).
DevBuf<float> g_evidence;  // [n][B2C_EVIDENCE_STRIDE]
DevBuf<float> g_view_acc;  // [n][3] the current view's (w_in, err, w_all)
DevBuf<float> g_labels;    // [n][B2C_LABEL_BINS]
// The downloads' rows, formed on the device from the accumulators (every download of one pass writes the same
// values). They are reserved before their accumulators, so an accumulator that holds n splats has n rows beside it
// also after a reserve has thrown.
DevBuf<float> g_evidence_rows;  // [n][7]
DevBuf<float> g_label_rows;     // [n][2]
bool g_labels_valid = false;
}  // namespace

void compute_evidence(RenderCtx& ctx, const Model& m, const std::vector<ViewGPU>& views, const std::vector<Camera>& cams,
                      const EvidenceParams& cfg, hipStream_t stream) {
  if (views.size() != cams.size()) throw std::runtime_error("compute_evidence: one camera per view");
  const size_t n = (size_t)(m.n > 0 ? m.n : 1);
  g_evidence_rows.reserve(n * 7);
  g_evidence.reserve(n * B2C_EVIDENCE_STRIDE);
  g_evidence.zero(stream);
  g_view_acc.reserve(n * 3);
  g_labels_valid = cfg.export_labels;
  if (g_labels_valid) {
    g_label_rows.reserve(n * 2);
    g_labels.reserve(n * B2C_LABEL_BINS);
    g_labels.zero(stream);
  }
  const bool use_normals = cfg.evidence_normal_weight > 0.f;
  for (size_t v = 0; v < views.size(); v++) {
    const ViewGPU& view = views[v];
    if (view.W != ctx.W || view.H != ctx.H) ctx.setup(view.W, view.H, m.cap, stream);
    RenderParams rp;
    rp.cam = CameraGPU::from(cams[v], view.W, view.H);
    rp.sh_degree = m.degree;
    rp.bwd_info = true;
    rp.feat = (use_normals && view.normals) ? FeatureMode::Normals : FeatureMode::None;
    render_forward(ctx, m, rp, stream);
    if (m.n == 0) continue;
    b2c_evidence_args a{};
    a.tile_ranges = reinterpret_cast<const uint32_t*>(ctx.tile_ranges.ptr);
    a.vals_sorted = ctx.vals_sorted;
    a.raster_rec = reinterpret_cast<const float*>(ctx.raster_rec.ptr);
    a.out_rgba = reinterpret_cast<const float*>(ctx.out_rgba.ptr);
    a.out_feat = reinterpret_cast<const float*>(ctx.out_feat.ptr);
    a.last_idx = ctx.last_idx;
    a.gt = view.rgba;
    a.normals = rp.feat == FeatureMode::Normals ? view.normals : nullptr;
    a.weights = view.weights;
    a.labels = g_labels_valid ? view.labels : nullptr;
    a.W = ctx.W; a.H = ctx.H; a.tiles_x = ctx.tiles_x; a.tiles_y = ctx.tiles_y;
    a.masked_has_alpha = (view.masked && view.has_alpha) ? 1 : 0;
    a.normal_weight = cfg.evidence_normal_weight;
    a.slot_sorted = ctx.slot_sorted;
    a.num_isect = ctx.num_isect;
    a.row_tag = ctx.next_row_tag(4, stream);
    a.rows = reinterpret_cast<float*>(ctx.isect_rows.ptr);  // the backward's row buffer, free between passes
    a.label_acc = g_labels_valid ? g_labels.ptr : nullptr;
    LAUNCH_CHECK(b2c_hip_evidence_view(&a, stream));
    b2c_evidence_sum_args sa{};
    sa.n = m.n;
    sa.m = ctx.num_isect;
    sa.ids = ctx.vals;
    sa.rows = a.rows;
    sa.row_tag = a.row_tag;
    sa.view_acc = g_view_acc.ptr;
    sa.pos_op = reinterpret_cast<const float*>(m.pos_op.ptr);
    for (int k = 0; k < 3; k++) sa.cam_pos[k] = cams[v].pos[k];
    sa.evidence = g_evidence.ptr;
    LAUNCH_CHECK(b2c_hip_evidence_sum(&sa, stream));
  }
  HIP_CHECK(hipStreamSynchronize(stream));
}

const float* evidence_device(int* stride) {
  *stride = B2C_EVIDENCE_STRIDE;
  return g_evidence.ptr;
}

void download_evidence(const Model& m, float* out, hipStream_t stream) {
  const size_t n = (size_t)m.n;
  if (g_evidence.count < n * B2C_EVIDENCE_STRIDE || n == 0) {
    std::fill(out, out + n * 7, 0.f);
    return;
  }
  LAUNCH_CHECK(b2c_hip_evidence_export(m.n, g_evidence.ptr, g_evidence_rows.ptr, stream));
  HIP_CHECK(hipMemcpyAsync(out, g_evidence_rows.ptr, n * 7 * sizeof(float), hipMemcpyDeviceToHost, stream));
  HIP_CHECK(hipStreamSynchronize(stream));
}

void download_labels(const Model& m, float* out, hipStream_t stream) {
  const size_t n = (size_t)m.n;
  if (!g_labels_valid || g_labels.count < n * B2C_LABEL_BINS || n == 0) {
    std::fill(out, out + n * 2, 0.f);
    return;
  }
  LAUNCH_CHECK(b2c_hip_label_export(m.n, g_labels.ptr, g_label_rows.ptr, stream));
  HIP_CHECK(hipMemcpyAsync(out, g_label_rows.ptr, n * 2 * sizeof(float), hipMemcpyDeviceToHost, stream));
  HIP_CHECK(hipStreamSynchronize(stream));
}

std::vector<float> download_evidence(const Model& m, hipStream_t stream) {
  std::vector<float> out((size_t)m.n * 7);
  download_evidence(m, out.data(), stream);
  return out;
}

std::vector<float> download_labels(const Model& m, hipStream_t stream) {
  std::vector<float> out((size_t)m.n * 2);
  download_labels(m, out.data(), stream);
  return out;
}

void probe_depth(RenderCtx& ctx, float tau, float delta, const float* ref_z, float margin, float4* out, hipStream_t stream) {
  b2c_probe_args a{};
  a.tile_ranges = reinterpret_cast<const uint32_t*>(ctx.tile_ranges.ptr);
  a.vals_sorted = ctx.vals_sorted;
  a.raster_rec = reinterpret_cast<const float*>(ctx.raster_rec.ptr);
  a.W = ctx.W; a.H = ctx.H; a.tiles_x = ctx.tiles_x; a.tiles_y = ctx.tiles_y;
  a.tau = tau; a.delta = delta; a.margin = margin;
  a.ref_z = ref_z;
  a.out = reinterpret_cast<float*>(out);
  LAUNCH_CHECK(b2c_hip_probe_depth(&a, stream));
}

}  // namespace b2c
