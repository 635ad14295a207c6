// What the forward convolution's launches share (lh_conv.hip; lh_conv_infer.hip): shapes, operand loaders, the NCHW epilogue, the
// filter's copies.
#pragma once
#include "lh_igemm.h"
#include <map>

namespace lh {
namespace {
struct ConvDims { int N, C, H, W, K, R, S, sH, sW, pH, pW, P, Q; };

static inline bool make_dims(ConvDims& d, int N, int C, int H, int W, int K, int R, int S, int sH, int sW, int pH, int pW) {
  if (N < 1 || C < 1 || H < 1 || W < 1 || K < 1 || R < 1 || S < 1 || sH < 1 || sW < 1 || pH < 0 || pW < 0) return false;
  if (H + 2 * pH < R || W + 2 * pW < S) return false;
  d = {N, C, H, W, K, R, S, sH, sW, pH, pW, (H + 2 * pH - R) / sH + 1, (W + 2 * pW - S) / sW + 1};
  const int64_t lim = 0x20000000LL;   // 2 GiB of fp32 per tensor: byte offsets of the buffer loads stay below 2^31
  if ((int64_t)N * C * H * W >= lim || (int64_t)N * K * d.P * d.Q >= lim || (int64_t)K * C * R * S >= lim) return false;
  return true;
}

// ---- B operand of the forward pass: im2col gather of x --------------------------------------
// column j = (n, p, q) fixed per thread; k = (c, r, s) is uniform across a wavefront.
struct LoadConvFwdB {
  static constexpr bool ALONG_K = false;
  static constexpr bool VEC4 = false;
  static constexpr bool SPLIT = false;
  const float* base; uint32_t nbytes;
  int C, H, W, sH, sW, pH, pW, HW;
  FastDiv dPQ, dQ, dRS, dS;
  struct State { int pix, h0, w0; bool valid; };     // pix = n*C*H*W + h0*W + w0 (may be negative)
  __device__ __forceinline__ void init(State& s, int j, int ncols) const {
    s.valid = j < ncols;
    uint32_t n, pq, p, q;
    dPQ.divmod(s.valid ? j : 0, n, pq); dQ.divmod(pq, p, q);
    s.h0 = (int)p * sH - pH; s.w0 = (int)q * sW - pW;
    s.pix = (int)n * C * HW + s.h0 * W + s.w0;
  }
  __device__ __forceinline__ uint32_t off1(const State& s, int k, int kend, int e) const {
    uint32_t c, rs, r, ss;
    dRS.divmod(k + e, c, rs); dS.divmod(rs, r, ss);
    const int tap = ((int)c * H + (int)r) * W + (int)ss;       // wave-uniform
    const bool ok = s.valid && k + e < kend && (unsigned)(s.h0 + (int)r) < (unsigned)H && (unsigned)(s.w0 + (int)ss) < (unsigned)W;
    return ok ? (uint32_t)(s.pix + tap) * 4u : LH_OOB;
  }
};

// ---- fast B operands for channel counts that are a multiple of the k-slab (16) -------------------------
// The reduction index is ordered tap-major, channel-minor: k = tap*CH + ch.  A 16-wide k-slab
// then lies inside one filter tap, so the tap decode and the bounds check are done once per
// slab on wave-uniform values and each element costs an add and a select.  The filter operand
// is brought into the matching [row][tap][ch] layout by a small transform kernel.
//
// Forward: column j = (n, p, q); element = x[n][ch][p*sH - pH + r][q*sW - pW + s], tap = r*S + s.
struct LoadConvFwdTapB {
  static constexpr bool ALONG_K = false;
  static constexpr bool VEC4 = false;
  static constexpr bool SPLIT = true;
  static constexpr bool STEP = true;
  const float* base; uint32_t nbytes;
  int C, H, W, sH, sW, pH, pW, HW;
  FastDiv dPQ, dQ, dC, dS;
  // inside a tap the next slab is the same pixels, bk channel planes further on
  __device__ __forceinline__ uint32_t step_bytes(int bk) const { return (uint32_t)(bk * HW) * 4u; }
  __device__ __forceinline__ int run_slabs(int k, int bk) const {
    uint32_t tap, ch;
    dC.divmod(k, tap, ch);
    return (C % bk) ? 1 : (C - (int)ch) / bk;
  }
  struct State { int pix, h0, w0; bool valid; };
  __device__ __forceinline__ void init(State& s, int j, int ncols) const {
    s.valid = j < ncols;
    uint32_t n, pq, p, q;
    dPQ.divmod(s.valid ? j : 0, n, pq); dQ.divmod(pq, p, q);
    s.h0 = (int)p * sH - pH; s.w0 = (int)q * sW - pW;
    s.pix = (int)n * C * HW + s.h0 * W + s.w0;
  }
  // per-lane part: the pixel under the tap of this group of four k (same tap for all four), or LH_OOB
  __device__ __forceinline__ uint32_t voff(const State& s, int k, int kend) const {
    uint32_t tap, ch, r, ss;
    dC.divmod(k, tap, ch); dS.divmod(tap, r, ss);                 // wave-uniform
    const bool ok = s.valid && k < kend && (unsigned)(s.h0 + (int)r) < (unsigned)H && (unsigned)(s.w0 + (int)ss) < (unsigned)W;
    return ok ? (uint32_t)(s.pix + (int)r * W + (int)ss) * 4u : LH_OOB;
  }
  // wave-uniform part: the channel plane of element e
  __device__ __forceinline__ uint32_t soff(int k, int e) const {
    uint32_t tap, ch;
    dC.divmod(k, tap, ch);
    return (uint32_t)(((int)ch + e) * HW) * 4u;
  }
};
// ---- epilogue writing an NCHW activation: row i = channel, column j = (n, u, v) on a grid of
//      Wc columns; the element lands at out[n][i][aH + eH*u][aW + eW*v] of an image W wide with PIX pixels.
struct EpiConvOut {
  static constexpr bool STATS = false;
  static constexpr bool SLICED = false;
  float* out; const float* bias; int chan, PIX, W, eH, eW, aH, aW; float beta;
  int relu = 0;             // complete sums are stored as max(v, 0); a launch that adds partial sums leaves that to a pass of its own (conv_fwd_impl)
  int zfill2 = 0;           // the grid is every second pixel of every second row of an image with even sides (a 1x1 filter, stride 2):
                            // the element is stored together with the three zeros of its 2x2 cell, so the output needs no clearing
  FastDiv dPIXc, dWc;
  struct Col { int off; bool valid; };
  __device__ __forceinline__ Col col(int j, int N) const {
    Col c; c.valid = j < N;
    uint32_t n, pix, u, v; dPIXc.divmod(c.valid ? j : 0, n, pix); dWc.divmod(pix, u, v);
    c.off = (int)n * chan * PIX + (aH + eH * (int)u) * W + aW + eW * (int)v;
    return c;
  }
  // lean stores: element (i, j) at lane_bytes(col(j)) + i * row_bytes() from `out` (the tensor is below 2 GiB); the bias of
  // the row and the clamp are applied to the value on its way (lean_fix)
  static constexpr bool LEAN = true;
  static constexpr bool LEAN_FIX = true;
  __device__ __forceinline__ bool lean_ok(int M) const { return (M & 7) == 0; }
  __device__ __forceinline__ float lean_fix(float v, int row) const {
    if (bias) v += bias[row];
    if (relu) v = v < 0.f ? 0.f : v;
    return v;
  }
  __device__ __forceinline__ float* lean_base() const { return out; }
  __device__ __forceinline__ uint32_t lane_bytes(const Col& c) const { return (uint32_t)c.off * 4u; }
  __device__ __forceinline__ uint32_t row_bytes() const { return (uint32_t)PIX * 4u; }
  __device__ __forceinline__ uint32_t cell_row_bytes() const { return (uint32_t)W * 4u; }
  __device__ __forceinline__ int lean_mode() const { return zfill2 ? 2 : (beta == 0.f ? 0 : 1); }
  __device__ __forceinline__ float lean_scale() const { return 1.f; }
  // part: 0 = complete sum; 1 = first partial, 2 = later partial (atomic adds onto a prepared output)
  __device__ __forceinline__ void store(const Col& c, int i, int M, float v, int part) const {
    if (!c.valid || i >= M) return;
    float* p = out + c.off + i * PIX;
    if (bias && part < 2) v += bias[i];
    if (relu && part == 0) v = v < 0.f ? 0.f : v;
    if (zfill2) {             // only set for overwriting, complete sums (host side)
      *reinterpret_cast<float2*>(p) = make_float2(v, 0.f);
      *reinterpret_cast<float2*>(p + W) = make_float2(0.f, 0.f);
      return;
    }
    if (part) atomicAdd(p, v);
    else *p = beta == 0.f ? v : v + beta * *p;
  }
};
static inline EpiConvOut make_epi(float* out, const float* bias, int chan, int Himg, int Wimg, float beta) {   // dense: grid == image
  EpiConvOut ep; ep.out = out; ep.bias = bias; ep.chan = chan; ep.PIX = Himg * Wimg; ep.W = Wimg; ep.eH = 1; ep.eW = 1; ep.aH = 0; ep.aW = 0; ep.beta = beta;
  ep.dPIXc.init(Himg * Wimg); ep.dWc.init(Wimg);
  return ep;
}

#ifndef LH_CONV_BK
#define LH_CONV_BK 16
#endif
constexpr int CONV_BK = LH_CONV_BK;      // k-slab of the forward / input-gradient kernels
// Tile choice of the forward / input-gradient launches.  With a reduction of at most 512 (1x1 filters over up to 512
// channels) a tile is finished after at most 32 slabs, and the fixed cost per tile (pipeline fill, epilogue) and the
// low occupancy of the 128-wide tiles weigh more than their better operand reuse: measured over the ResNet-50 layers,
// 64x64 tiles are 4-17 % faster there and equal or slower for longer reductions.
static inline TilePick pick_tile_conv(int M, int N, int K) {
  if (K <= 512) return {64, 64};
  return pick_tile(M, N);
}
// The built-in rule's other half: few tiles over a long reduction run stream-K (a worker's share must span many slabs for the
// per-segment set-up to pay off).
static inline bool stream_k_rule(int M, int N, int K) {
  const int64_t tiles = M > 64 ? cdiv(M, 128) * cdiv(N, 128) : cdiv(M, 64) * cdiv(N, 128), slabs = cdiv(K, CONV_BK);
  return !g_deterministic && tiles < 6 * (int64_t)g_num_cu && slabs >= 64 && slabs * tiles >= 48 * (int64_t)(2 * g_num_cu);
}
// The filter in the layout a launch reads: the library's kept copy (written now if it is stale), or, where none is kept,
// scratch from the arena top that the caller pops behind the launch (stream order keeps that safe).
struct FilterCopy { float* p = nullptr; size_t scratch = 0; };
static inline bool filter_copy(FilterCopy& fc, const float* w, size_t wbytes, int kind, const int* prm, size_t bytes) {
  bool build = false;
  fc.scratch = 0;
  fc.p = lazy::layout_lookup(w, wbytes, kind, prm, bytes, build);
  if (fc.p == nullptr) {
    fc.p = (float*)lh_malloc_uninit(bytes);
    if (fc.p == nullptr) return false;
    fc.scratch = bytes; build = true;
  }
  if (build) build_filter_layout(kind, prm, w, fc.p);
  return true;
}

// LH_FORCE_PLAN=n in the environment: forward / input-gradient products take launch plan n where it is valid (for tests that
// compare the plans' results with each other).
static inline int force_plan() { const char* e = getenv("LH_FORCE_PLAN"); return e ? atoi(e) : -1; }
// A launch shape a measured choice is remembered for.
struct PlanKey {
  int v[7];
  bool operator<(const PlanKey& o) const { for (int i = 0; i < 7; i++) if (v[i] != o.v[i]) return v[i] < o.v[i]; return false; }
};
}  // namespace
}  // namespace lh
