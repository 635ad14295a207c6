// How many launches, and how many convolutions among them, the inference chain of the deferred work costs (conv -> batch norm with running statistics -> [+ shortcut] ->
// relu in place as one launch, what it leaves out noted with a recipe) over defer_infer_check.cpp's simulated device: a network of
// 20 layers, six of them with a join, passed over again by programs that use memory in different ways.
//   rewind     every pass in fresh arena memory that a rewind releases: one launch a layer, no recipe ever runs
//   flush      the same with lh_flush_deferred in front of the rewind
//   fixed      every buffer allocated once
//   ping-pong  activations in two buffers in turn, one buffer each for the convolution's and the batch norm's outputs
// In the last three the results left out have to be produced after all: once, and from then on no pass may run a convolution
// twice or cost more launches than the same calls run as issued.  A filter released and another in its place starts afresh.
#define DEFER_INFER_NO_MAIN
#include "defer_infer_check.cpp"

static char* g_block;                          // the arena's memory with room for parameters below and above it
static float* foreign_at;
static const size_t OUTSIDE = 1 << 16;
enum { REWIND, FLUSH, FIXED, PING_PONG };
static const int NL = 20, PASSES = 8;
struct ChainLayer { float *w, *g, *b, *m, *v, *y, *t, *o; };

struct Cost { long long launches, convs; };          // of one pass
static std::vector<Cost> costs(int how, bool enabled, bool second_network, bool outside = false) {       // outside: the parameters lie in memory that is not the arena's
  g_rng = 77;
  lazy::reset(); lazy::g_enabled = enabled; lazy::g_depth = 0;
  memset(g_heap, 0xCD, g_arena.bytes); { const size_t b = g_arena.bytes; g_arena = ArenaState(); g_arena.bytes = b; }
  auto fill = [&](float* p, int n) { lazy::Scope s_; if (lazy::g_busy) lazy::flush_parked(); lazy::wr(p, SZ(n)); for (int i = 0; i < n; i++) p[i] = rf(); };
  std::vector<Cost> counts;
  for (int network = 0; network <= (second_network ? 1 : 0); network++) {
    const size_t base = g_arena.top;
    ChainLayer ls[NL];
    int at = 0;
    for (auto& l : ls) for (float** p : {&l.w, &l.g, &l.b, &l.m, &l.v}) { const int n = p == &l.w ? 12 : C_; *p = outside ? foreign_at + 64 * (at++) : (float*)sim_malloc(SZ(n), false); fill(*p, n); }
    auto make = [&]() { return (float*)sim_malloc(SZ(NE), false); };
    float *input = make(), *ping[2] = {make(), make()}, *y1 = make(), *t1 = make();
    for (auto& l : ls) { l.y = make(); l.t = make(); l.o = make(); }
    const size_t mark = g_arena.top;
    const bool flushes = how == FLUSH && network == 0;         // the second network's program rewinds only
    for (int pass = 0; pass < PASSES; pass++) {
      const long long before = g_kernels, convs = g_convs + g_chains;
      fill(input, NE);
      float *h = input, *shortcut = nullptr;
      for (int i = 0; i < NL; i++) {
        ChainLayer& l = ls[i];
        const bool join = i % 3 == 2 && i < 18;
        if (i % 3 == 0 || how == PING_PONG) shortcut = h;
        float* y = how == FIXED ? l.y : (how == PING_PONG ? y1 : make());
        float* t = how == FIXED ? l.t : (how == PING_PONG ? (join ? t1 : ping[i % 2]) : make());
        float* o = !join ? t : (how == FIXED ? l.o : (how == PING_PONG ? ping[i % 2] : make()));
        lh_conv2d_fwd(h, l.w, nullptr, y, N_, C_, 1, HW_, C_, 1, 1, 1, 1, 0, 0);
        t_bn_infer(y, l.g, l.b, l.m, l.v, t);
        if (join) t_add(t, shortcut, o, NE);
        t_relu_inplace(o, NE);
        h = o;
      }
      std::vector<float> logits;
      t_d2h(logits, h, NE);
      if (flushes) { lazy::Scope s_; lazy::flush_all(); }
      if (how == REWIND || how == FLUSH) sim_rewind(mark);
      counts.push_back({g_kernels - before, g_convs + g_chains - convs});
    }
    if (second_network && network == 0) { sim_rewind(base); { lazy::Scope s_; lazy::filters_released(g_heap + base); } }
  }
  { lazy::Scope s_; lazy::flush_all(); }
  return counts;
}

// A chain (with or without a join) whose outputs, or whose operands, lie outside the arena, read back behind a rewind.
static std::vector<float> outside_results(char* where, bool enabled, bool operands, bool join) {
  g_rng = 5;
  lazy::reset(); lazy::g_enabled = enabled; lazy::g_depth = 0;
  memset(g_heap, 0xCD, g_arena.bytes); { const size_t b = g_arena.bytes; g_arena = ArenaState(); g_arena.bytes = b; }
  float* at = (float*)where;
  auto out = [&]() { float* p = at; at += 256; memset(p, 0xCD, SZ(NE)); return p; };
  auto in = [&]() { return (float*)sim_malloc(SZ(NE), false); };
  const size_t low = g_arena.top;
  float* p[8];
  for (auto& q : p) { q = operands ? out() : in(); lazy::Scope s_; if (lazy::g_busy) lazy::flush_parked(); lazy::wr(q, SZ(NE)); for (int i = 0; i < NE; i++) q[i] = rf(); }
  const size_t mark = operands ? low : g_arena.top;
  float *y = operands ? in() : out(), *t = operands ? in() : out(), *o = operands ? in() : out();
  lh_conv2d_fwd(p[0], p[1], nullptr, y, N_, C_, 1, HW_, C_, 1, 1, 1, 1, 0, 0);
  t_bn_infer(y, p[2], p[3], p[4], p[5], t);
  if (join) t_add(t, p[6], o, NE);
  t_relu_inplace(join ? o : t, NE);
  std::vector<float> got;
  if (operands) t_d2h(got, join ? o : t, NE);
  sim_rewind(mark);
  if (!operands) { t_d2h(got, y, NE); t_d2h(got, t, NE); if (join) t_d2h(got, o, NE); }
  return got;
}

int main() {
  g_arena.bytes = 4u << 20;
  g_block = (char*)aligned_alloc(256, g_arena.bytes + 2 * OUTSIDE);
  g_heap = g_block + OUTSIDE;
  const char* names[] = {"rewind", "flush", "fixed", "ping-pong"};
  int bad = 0;
  for (int how = REWIND; how <= PING_PONG; how++) {
    const std::vector<Cost> issued = costs(how, false, false);
    const long long recipes = lazy::g_stat[lazy::ST_RECIPES];
    const std::vector<Cost> deferred = costs(how, true, false);
    printf("%s: as issued %lld launches (%lld convolutions) a pass, deferred", names[how], issued[0].launches, issued[0].convs);
    for (const Cost& c : deferred) printf(" %lld (%lld)", c.launches, c.convs);
    printf(", recipes %lld\n", (long long)(lazy::g_stat[lazy::ST_RECIPES] - recipes));
    if (how == REWIND) {
      if (lazy::g_stat[lazy::ST_RECIPES] != recipes) bad = 1;
      for (const Cost& c : deferred) if (c.launches != NL) bad = 1;
    }
    // what the first pass left out may still have to be produced in the second
    for (int pass = how == FLUSH ? 1 : 2; pass < PASSES; pass++)
      if (deferred[pass].launches > issued[pass].launches || deferred[pass].convs > issued[pass].convs) { printf("%s: pass %d costs more than its calls as issued\n", names[how], pass); bad = 1; }
  }
  for (bool high : {false, true}) {                       // the parameters below and above the arena: a rewind releases neither
    float* const keep = foreign_at;
    foreign_at = high ? (float*)(g_heap + g_arena.bytes) : (float*)g_block;
    const std::vector<Cost> deferred = costs(FLUSH, true, false, true);
    foreign_at = keep;
    if (deferred[PASSES - 1].convs != NL) { printf("parameters outside the arena: %lld convolutions a pass\n", deferred[PASSES - 1].convs); bad = 1; }
  }
  for (char* where : {g_block, g_heap + g_arena.bytes})
    for (int form = 0; form < 4; form++) {
      const std::vector<float> a = outside_results(where, false, form & 1, form & 2), b = outside_results(where, true, form & 1, form & 2);
      if (a.size() != b.size() || memcmp(a.data(), b.data(), a.size() * 4) != 0) { printf("a chain over memory outside the arena (form %d, %s it): other values\n", form, where == g_block ? "below" : "above"); bad = 1; }
    }
  const std::vector<Cost> again = costs(FLUSH, true, true);
  if (again[PASSES - 1].launches <= NL || again[2 * PASSES - 1].launches != NL) { printf("a network in the place of another: %lld launches a pass\n", again[2 * PASSES - 1].launches); bad = 1; }
  lazy::reset();
  free(g_block);
  if (!bad) printf("defer_infer_launches: ok\n");
  return bad;
}
