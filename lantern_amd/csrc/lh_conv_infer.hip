// Forward convolution with a batch norm on running statistics, the residual join and relu in its epilogue: what the deferred work
// (lh_defer.hip) makes of conv2D_batch -> batchNormInference [-> + shortcut] [-> relu in place], the calls of a network that is
// served (the reference's readONNX inference_func, src/main/scala/lantern/ONNXLib.scala:597-830).
#include "lh_conv_fwd.h"
#include "lh_infer.h"
using namespace lh;

namespace {
// y = act((v - mean) * (gamma / sqrt(var + eps)) + beta [+ shortcut]) with v = sum + bias: k_bn_infer's formula, operation by
// operation, so that the chain gives the bits of its parts.  Complete sums only (no stream-K).
struct EpiConvBn : EpiConvOut {
  static constexpr bool ROWS = true;
  const float* gamma; const float* shift; const float* mean; const float* var; float eps;
  const float* shortcut;
  // a row's values as they lie in memory (0 past the last row), and what the epilogue makes of them
  __device__ __forceinline__ float row_load(const float* p, int row, int M) const {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, M * 4, LH_RSRC_FLAGS);
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, row * 4, 0, 0));
  }
  __device__ __forceinline__ void row_fetch(int row, int M, float4& v, float& b) const {
    v = make_float4(row_load(mean, row, M), row_load(gamma, row, M), row_load(shift, row, M), row_load(var, row, M));
    if (bias) b = row_load(bias, row, M);
  }
  __device__ __forceinline__ float4 row_params(const float4 v, float b) const { return make_float4(v.x, v.y / sqrtf(v.w + eps), v.z, b); }
  __device__ __forceinline__ float row_value(float v, const float4 p, float other, bool join) const {
    if (bias) v += p.w;
    float r = fmaf(v - p.x, p.y, p.z);
    if (join) r += other;
    if (relu) r = r < 0.f ? 0.f : r;
    return r;
  }
  __device__ __forceinline__ int lean_mode() const { return shortcut ? 3 : 0; }
  __device__ __forceinline__ const float* lean_other() const { return shortcut; }
  __device__ __forceinline__ void store_row(const Col& c, int i, int M, float v, const float4 p) const {
    if (!c.valid || i >= M) return;
    const int64_t at = (int64_t)c.off + (int64_t)i * PIX;
    out[at] = row_value(v, p, shortcut ? shortcut[at] : 0.f, shortcut != nullptr);
  }
};

// Launch forms: 1-3 whole tiles 128x128, 64x128, 64x64; 5-7 the last tiles of 64x64 / 64x128 / 128x128 sliced along the reduction
// (igemm_launch_shared_tail); 8-11 64x64 tiles on blocks of two groups of wavefronts, whole and sliced, and of four, whole and sliced;
// 4 the convolution by itself (any of its launch plans, stream-K among them), then the pass over it.  Channel counts that are no multiple of
// the slab's depth: 2, 3 and 4.
template <class AL, class BL>
bool launch_form(int form, const AL& al, const BL& bl, const EpiConvBn& ep, int M, int N, int K) {
  if (form == 1) return igemm_launch<128, 128, CONV_BK>(al, bl, ep, M, N, K, 1);
  if (form == 2) return igemm_launch<64, 128, CONV_BK>(al, bl, ep, M, N, K, 1);
  if (form == 5) return igemm_launch_shared_tail<64, 64, CONV_BK>(al, bl, ep, M, N, K);
  if (form == 8) return igemm_launch_shared_tail<64, 64, CONV_BK, 2, 1>(al, bl, ep, M, N, K);
  if (form == 9) return igemm_launch_shared_tail<64, 64, CONV_BK, 2>(al, bl, ep, M, N, K);
  if (form == 10) return igemm_launch_shared_tail<64, 64, CONV_BK, 4, 1>(al, bl, ep, M, N, K);
  if (form == 11) return igemm_launch_shared_tail<64, 64, CONV_BK, 4>(al, bl, ep, M, N, K);
  if (form == 6) return igemm_launch_shared_tail<64, 128, CONV_BK>(al, bl, ep, M, N, K);
  if (form == 7) return igemm_launch_shared_tail<128, 128, CONV_BK>(al, bl, ep, M, N, K);
  return igemm_launch<64, 64, CONV_BK>(al, bl, ep, M, N, K, 1);
}
int form_of_rule(int M, int N, int K) {
  const TilePick tp = pick_tile_conv(M, N, K);
  return tp.bm == 128 ? 1 : (tp.bn == 128 ? 2 : 3);
}
}  // namespace

namespace lh {
// ResNet-50 at 224x224 on one card in turn, 53 such chains (before: 53 convolutions, 53 batch norms, 33 relus and 16 joins, each a pass
// over memory): batch 32 4.28 -> 2.90 ms, batch 1 1.006 -> 0.797 ms; with forms 8-11 and the rows' parameters asked for ahead of the
// operands (a round trip less per launch: batch 1 742 -> 728 us) 2.92 -> 2.74 ms and 0.794 -> 0.728 ms.  What bounds it now is the
// convolutions themselves; at batch 1 a launch of the smallest takes 8.4 us for 4 slabs, 5 of them fixed.
void conv2d_bn_infer_now(const float* x, const float* w, const float* bias, int N, int C, int H, int W, int K, int R, int S, int sH, int sW, int pH, int pW,
                         const float* gamma, const float* beta, const float* mean, const float* var, float eps, const float* shortcut, float* out, int relu) {
  KernelCat kc_(CAT_CONV_FWD);
  ConvDims d;
  LH_REQUIRE(make_dims(d, N, C, H, W, K, R, S, sH, sW, pH, pW), "lh_conv2d_fwd: bad shape N%d C%d H%d W%d K%d R%d S%d s(%d,%d) p(%d,%d)", N, C, H, W, K, R, S, sH, sW, pH, pW);
  const int RS = R * S, CRS = C * RS, PQ = d.P * d.Q, cols = N * PQ;
  const uint32_t wbytes = (uint32_t)((size_t)K * CRS * 4), xbytes = (uint32_t)((size_t)N * C * H * W * 4);
  EpiConvBn ep;
  static_cast<EpiConvOut&>(ep) = make_epi(out, bias, K, d.P, d.Q, 0.f);
  ep.relu = relu; ep.gamma = gamma; ep.shift = beta; ep.mean = mean; ep.var = var; ep.eps = eps; ep.shortcut = shortcut;
  // Form 4: the convolution by itself, then the pass over it.  (`form` below: the rule's, where nothing is measured)
  auto parts = [&]() {
    lh_conv2d_fwd(x, w, bias, out, N, C, H, W, K, R, S, sH, sW, pH, pW);
    if (!failed()) bn_infer_now(out, gamma, beta, mean, var, eps, shortcut, out, relu, N, K, PQ);
    return !failed();
  };
  // The form is measured once per shape (the launch overwrites `out` and nothing else, so repeating it is harmless) and remembered.
  // false: reported.
  auto run_measured = [&](int loader, int form, auto valid, auto run) {
    static std::map<PlanKey, int> chosen;
    const PlanKey key = {{K, cols, CRS, H, W, sH, R | (shortcut ? 1 << 16 : 0) | (g_deterministic ? 1 << 17 : 0) | loader << 18}};
    const int forced = force_plan() >= 13 && force_plan() <= 19 ? force_plan() - 8 : force_plan();
    auto it = chosen.find(key);
    if (forced >= 1 && forced <= 11 && valid(forced)) form = forced;
    else if (it != chosen.end() && g_tune_enabled) { form = it->second; g_plans_remembered++; }
    else if (g_tune_enabled && !g_capturing && 2.0 * K * CRS * (double)cols >= g_tune_min_flop) {
      LaunchTimer timer;
      if (timer.ok) {
        float best_ms = 3.0e38f;
        const int order[11] = {3, 2, 1, 5, 6, 7, 4, 8, 9, 10, 11};
        for (int f : order) {
          if (!valid(f)) continue;
          const float ms = timer.ms([&]() { return run(f); });
          if (ms < 0.f || failed()) return false;
          if (ms < best_ms * 0.98f) { best_ms = ms; form = f; }
        }
        chosen[key] = form; g_plans_measured++;
        if (getenv("LH_TUNE_VERBOSE")) fprintf(stderr, "conv + bn (running) K%d N%d CRS%d H%d: form %d, %.4f ms\n", K, cols, CRS, H, form, best_ms);
      }
    }
    return run(form);
  };
  bool ok;
  if (C % CONV_BK == 0 && ((uintptr_t)w & 15) == 0) {
    // tap-major reduction order; a 1x1 filter already has that layout
    FilterCopy fc;
    fc.p = const_cast<float*>(w);
    const int prm[LAYOUT_PRM] = {K, C, RS};
    bool copied = RS == 1;
    LoadPlainK<true> al; al.base = fc.p; al.nbytes = wbytes; al.ld = CRS;
    LoadConvFwdTapB bl; bl.base = x; bl.nbytes = xbytes; bl.C = C; bl.H = H; bl.W = W; bl.sH = sH; bl.sW = sW; bl.pH = pH; bl.pW = pW; bl.HW = H * W;
    bl.dPQ.init(PQ); bl.dQ.init(d.Q); bl.dC.init(C); bl.dS.init(S);
    auto valid = [&](int form) {
      if ((form == 1 || form == 7) && K <= 64) return false;
      if (form >= 8) return !g_deterministic && (form == 8 || form == 10 || g_stream_cur == g_stream_raw) && cdiv(CRS, CONV_BK) >= (form >= 10 ? 16 : 8) && cdiv(K, 64) * cdiv(cols, 64) <= 8 * (int64_t)g_num_cu;
      if (form >= 5) return !g_deterministic && g_stream_cur == g_stream_raw && CRS >= 8 * CONV_BK;
      // the convolution by itself, where stream-K may win more than the pass behind it costs: fewer tiles than compute units, or a long
      // reduction (512 -> 512 channels 3x3 over 14x14, batch 32: 231 -> 219 us; without measuring, 7x7 over 7x7 to 4096 1798 -> 1091)
      if (form == 4) return !g_deterministic && (CRS >= 64 * CONV_BK || (cdiv(K, 64) * cdiv(cols, 64) < g_num_cu && CRS >= 16 * CONV_BK));
      return true;
    };
    ok = run_measured(0, stream_k_rule(K, cols, CRS) ? 4 : form_of_rule(K, cols, CRS), valid, [&](int form) {
      if (form == 4) return parts();
      if (!copied && !filter_copy(fc, w, wbytes, LAYOUT_KRSC, prm, wbytes)) return false;
      copied = true; al.base = fc.p;
      return launch_form(form, al, bl, ep, K, cols, CRS);
    });
    if (fc.scratch) lh_free_top(fc.scratch);
  } else {
    // Any other channel count: whole 64x64 and 64x128 tiles, or the parts with the convolution's own choice of plans (stream-K, tiles of
    // 32 rows, groups of wavefronts).  A whole tile by rule, its filter loaded 4 bytes at a time -> the measured form | the parts:
    // 100 -> 100 channels 3x3 over 7x7, batch 64 80.6 -> 27.8 | 29.8 us, 20 -> 50 channels 5x5 over 28x28, batch 1 31.3 -> 15.7 | 17.9.
    LoadConvFwdB bl; bl.base = x; bl.nbytes = xbytes; bl.C = C; bl.H = H; bl.W = W; bl.sH = sH; bl.sW = sW; bl.pH = pH; bl.pW = pW; bl.HW = H * W;
    bl.dPQ.init(PQ); bl.dQ.init(d.Q); bl.dRS.init(RS); bl.dS.init(S);
    auto valid = [&](int form) { return form == 2 || form == 3 || (form == 4 && !g_deterministic); };
    auto with = [&](const auto& al, int loader) {
      return run_measured(loader, form_of_rule(K, cols, CRS), valid, [&](int form) {
        if (form == 4) return parts();
        return form == 3 ? igemm_launch<64, 64, CONV_BK>(al, bl, ep, K, cols, CRS, 1) : igemm_launch<64, 128, CONV_BK>(al, bl, ep, K, cols, CRS, 1);
      });
    };
    if (CRS % 4 == 0 && ((uintptr_t)w & 15) == 0) { LoadPlainK<true> al; al.base = w; al.nbytes = wbytes; al.ld = CRS; ok = with(al, 1); }
    else { LoadPlainK<false> al; al.base = w; al.nbytes = wbytes; al.ld = CRS; ok = with(al, 2); }
  }
  if (!ok) return;
  LH_CHECK_LAUNCH();
}
}  // namespace lh
