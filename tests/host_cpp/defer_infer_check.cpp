// The inference chain of the deferred work (conv -> batch norm with running statistics -> [+ shortcut] -> relu in place as one
// launch that leaves the convolution's output, and under a join the batch norm's, unwritten) over defer_check.cpp's simulated
// device: seeded random programs run deferred and as issued, with read-backs of what was left out, writes over what a recipe
// still has to read (input, filter, channel parameters), outputs that lie over the chain's own operands, undeclared calls and
// rewinds.  Every read-back and the final arena must be identical bit for bit.
// Usage: defer_infer_check [programs] [seed]
#define main defer_check_main
#include "defer_check.cpp"
#undef main
#include "../../lantern_amd/csrc/lh_infer.h"

static long long g_chains = 0;
static void k_bn_infer(const float* x, const float* g, const float* b, const float* m, const float* v, float eps, const float* sc, float* y, int relu) {
  std::vector<float> r(NE);
  for (int i = 0; i < NE; i++) { const int c = chan(i); float a = (x[i] - m[c]) * (g[c] / sqrtf(v[c] * v[c] + eps)) + b[c]; if (sc) a += sc[i]; r[i] = relu && a < 0.f ? 0.f : a; }
  memcpy(y, r.data(), SZ(NE));
  g_kernels++;
}
namespace lh {
void conv2d_bn_infer_now(const float* x, const float* w, const float* bias, int, int, int, int, int, int, int, int, int, int, int, const float* g, const float* b, const float* m,
                         const float* v, float eps, const float* sc, float* out, int relu) {
  (void)ordered_stream();
  // as the device would: an output over an operand of the launch shows as a wrong value
  for (int i = 0; i < NE; i++) {
    const int c = chan(i);
    float a = bias ? bias[c] : 0.f;
    for (int k = 0; k < 3; k++) a += x[(i + 7 * k) % NE] * sim_filter(w)[(c + k) % 12];
    float r = (a - m[c]) * (g[c] / sqrtf(v[c] * v[c] + eps)) + b[c];
    if (sc) r += sc[i];
    out[i] = relu && r < 0.f ? 0.f : r;
  }
  g_kernels++; g_chains++;
}
void bn_infer_now(const float* x, const float* g, const float* b, const float* m, const float* v, float eps, const float* sc, float* y, int relu, int, int, int) {
  (void)ordered_stream(); k_bn_infer(x, g, b, m, v, eps, sc, y, relu);
}
}  // namespace lh
static void t_bn_infer(const float* x, const float* g, const float* b, const float* m, const float* v, float* y) {
  LZ_SCOPE();
  if (lazy::park_bn_infer(x, g, b, m, v, y, N_, C_, HW_, 1e-5f)) return;
  if (lazy::g_busy && !lazy::g_replay) lazy::flush_parked();
  lazy::rd_f(x, NE); lazy::rd_f(g, C_); lazy::rd_f(b, C_); lazy::rd_f(m, C_); lazy::rd_f(v, C_);
  lazy::out_f(y, NE, y == x);
  bn_infer_now(x, g, b, m, v, 1e-5f, nullptr, y, 0, N_, C_, HW_);
}

static void infer_program(uint64_t seed, bool enabled, std::vector<float>& trace, std::vector<char>& image) {
  g_rng = seed;
  lazy::reset(); lazy::g_enabled = enabled; lazy::g_depth = 0;
  memset(g_heap, 0xCD, g_arena.bytes); { const size_t b = g_arena.bytes; g_arena = ArenaState(); g_arena.bytes = b; }
  auto fill = [&](float* p, int n) { std::vector<float> h(n); for (auto& v : h) v = rf(); lazy::Scope s_; if (lazy::g_busy) lazy::flush_parked(); lazy::wr(p, SZ(n)); memcpy(p, h.data(), SZ(n)); };
  auto vec = [&](int n) { float* p = (float*)sim_malloc(SZ(n), true); fill(p, n); return p; };
  struct L { float *w, *bias, *g, *b, *m, *v, *in, *y, *t, *out; };
  const int nl = ri(1, 6);
  std::vector<L> ls(nl);
  for (auto& l : ls) { l.w = vec(12); l.bias = vec(C_); l.g = vec(C_); l.b = vec(C_); l.m = vec(C_); l.v = vec(C_); }
  float* input = vec(NE);
  const size_t mark = g_arena.top;
  const int passes = ri(1, 3);
  for (int pass = 0; pass < passes; pass++) {
    float* h = input;
    for (auto& l : ls) {
      l.in = h; l.y = (float*)sim_malloc(SZ(NE), true);
      lh_conv2d_fwd(h, l.w, ri(0, 2) == 0 ? l.bias : nullptr, l.y, N_, C_, 1, HW_, C_, 1, 1, 1, 1, 0, 0);
      if (ri(0, 11) == 0) t_d2h(trace, l.y, 5);
      const int where = ri(0, 9);                          // the batch norm's output: mostly of its own, sometimes in place, or over the convolution's input
      l.t = where == 0 ? l.y : (where == 1 && h != input ? h : (float*)sim_malloc(SZ(NE), true));
      t_bn_infer(l.y, l.g, l.b, l.m, l.v, l.t);
      l.out = l.t;
      if (ri(0, 13) == 0) t_d2h(trace, l.t + 3, 4);
      if (ri(0, 15) == 0) fill(l.m, C_);                    // a parameter of a chain that may still be parked
      if (ri(0, 2) == 0 && l.t != h) {
        const int o = ri(0, 9);
        float* sc = ri(0, 5) == 0 ? l.y : h;
        l.out = o == 0 && h != input && sc != h ? h : (o == 1 && sc != l.t ? l.y : (float*)sim_malloc(SZ(NE), true));
        if (l.out == sc || l.out == l.t) l.out = (float*)sim_malloc(SZ(NE), true);
        if (ri(0, 1)) t_add(l.t, sc, l.out, NE); else t_add(sc, l.t, l.out, NE);
      }
      if (ri(0, 11) == 0) { float* tmp = (float*)sim_malloc(SZ(NE), true); t_geam(l.out, 1.f, l.out, 0.f, tmp, NE); }
      if (ri(0, 3) != 0) t_relu_inplace(l.out, NE);
      h = l.out;
      switch (ri(0, 15)) {
        case 0: t_d2h(trace, l.y, NE); break;               // what the chain left out
        case 1: t_d2h(trace, l.t + 7, 20); break;
        case 2: t_geam(l.in, -1.f, l.in, 0.f, l.in, NE); t_d2h(trace, l.y, NE); break;        // over what its recipe reads
        case 3: fill(l.w, 12); t_d2h(trace, l.y, 9); break;
        case 4: fill(l.g, C_); t_d2h(trace, l.t, 9); break;
        case 5: t_fill(l.y + 8, 2.5f, 16); t_d2h(trace, l.y, NE); break;                       // over part of what was left out
        case 6: t_undeclared(l.in, 7); break;
        case 7: t_geam(l.y, 1.f, l.t, 1.f, l.y, NE); break;
        default: break;
      }
    }
    t_d2h(trace, h, NE);
    if (pass + 1 < passes || ri(0, 1)) sim_rewind(mark);
  }
  { lazy::Scope s_; lazy::flush_all(); }
  image.assign(g_heap, g_heap + g_arena.top);
}

#ifndef DEFER_INFER_NO_MAIN          // (defer_infer_launches.cpp has one of its own)
int main(int argc, char** argv) {
  const int programs = argc > 1 ? atoi(argv[1]) : 2000;
  const uint64_t seed0 = argc > 2 ? (uint64_t)atoll(argv[2]) : 1;
  g_arena.bytes = 4u << 20;
  g_heap = (char*)aligned_alloc(256, g_arena.bytes);
  for (int p = 0; p < programs; p++) {
    std::vector<float> t_off, t_on; std::vector<char> i_off, i_on;
    infer_program(seed0 * 1000003ull + p, false, t_off, i_off);
    infer_program(seed0 * 1000003ull + p, true, t_on, i_on);
    if (t_off.size() != t_on.size() || memcmp(t_off.data(), t_on.data(), t_off.size() * 4) != 0 || i_off.size() != i_on.size() || memcmp(i_off.data(), i_on.data(), i_off.size()) != 0) {
      size_t i = 0; while (i < t_off.size() && i < t_on.size() && memcmp(&t_off[i], &t_on[i], 4) == 0) i++;
      fprintf(stderr, "program %d: read-back %zu of %zu differs, or the final arena\n", p, i, t_off.size());
      return 1;
    }
  }
  printf("defer_infer_check: %d programs identical, %lld chains in one launch, %lld recipes run\n", programs, g_chains, (long long)lazy::g_stat[lazy::ST_RECIPES]);
  lazy::reset();
  free(g_heap);
  return 0;
}
#endif
