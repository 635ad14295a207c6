// The recurrence of the Elman, LSTM and GRU layers as one launch for all time steps.
// Reference behaviour being replaced: the time loop inside cudnnRNNForwardTraining / cudnnRNNBackwardData
// (src/main/scala/lantern/TensorDslCudnn.scala:1638-1893).
//
// A time step is a [B, H] x [H, gates * H] product of microseconds whose operands are 0.1 MB of state and 3 to 10 MB of weights.
// One launch per step reads the weights again every time (no L2 keeps them over a launch) and pays for the launch.  Here every
// block keeps the weights of its 4 to 16 hidden units in registers for the whole sequence, and what travels between the blocks
// of a step is the state alone, through a ring of SEQ_RING slots in memory of the library's own (not the arena's: a graph's replay
// clears and writes the ring at the address it was recorded with, long after the arena has handed out what lay above its top then):
//
//   - a word of a slot is SEQ_EMPTY until the thread that owns it writes the step's value, and readers ask again until no word
//     they were given is SEQ_EMPTY.  The word is the message: nothing depends on the order in which two words become visible,
//     so there is no flag, no fence and no barrier across blocks.  (A value whose bits are SEQ_EMPTY, one of the NaNs, is sent
//     as the canonical NaN.)  Words are written and read with the device-coherent cache policy (sc0 sc1), since blocks on
//     different XCDs share no L2.
//   - the owner empties a word again two steps after it was written: it has then read the state that every reader could only
//     write after having read that word.  The slot comes round two steps later still, and before a block publishes anything more
//     it has waited for its own stores (s_waitcnt vmcnt(0) behind every step's first loads), so no reader can meet an old value.
//
// All blocks of a launch have to be resident together: at most one block per compute unit is launched, on the main stream only
// (so no second launch of this kind, nor the command list's, runs beside it), and whatever else of this process holds a compute unit
// ends by itself.  A second process that runs such layers on the same card can hold the units this launch still needs while it waits
// for those this one holds: the waits then run out, and from the first one that did the process keeps one launch
// per step (graphs recorded before hold what they hold).  Every step's waits are bounded all the same; a wavefront whose wait runs
// out says so in a pinned word and goes on without waiting, to the end of the sequence.
//
// What bounds it is latency: of an Elman step's 2.4 us (B 32, H 800) the matrix instructions take 0.7, the rest is a word's way out
// (a write-through store) and in (polls of 0.7 us a round), LDS and the activation.  Per step, one launch per step -> now, B 32,
// H 800: Elman, both directions 5.1 -> 2.5 us, LSTM forward 9.4 -> 4.1, backward 14.8 -> 6.4 (3200 k, 100 blocks: 2.7 us of matrix
// instructions).  DeepSpeech2 step 11.24 -> 8.37 ms, LSTM layer (T 185) 5.04 -> 2.84, GRU 4.48 -> 2.47, hidden sizes that are no
// multiple of 4 (which kept the per-step vector kernels or a cut product) 4 to 7 times as fast.  Measured and dropped: a slot per
// step read through L2 once its first words are there (equal: bandwidth is not the bound), asking for one group first and the
// rest behind it (equal to 4 % slower), waiting 0.2 to 0.9 us before the first poll (2 to 8 % slower), sc1 alone (equal).
#include "lh_rnn_seq.h"
#include "lh_rnn_tile.h"
#include "../../include/lantern_hip.h"

namespace lh {
bool g_captured_seq = false;
namespace {

constexpr unsigned SEQ_EMPTY = 0xffffffffu;
constexpr int SEQ_RING = 4;
constexpr int SEQ_COHERENT = 17;             // cache policy bits of the buffer instructions: sc0 | sc1
constexpr int SEQ_SPINS = 4000000;           // polls in one step before a wavefront gives up: seconds, where a real wait is microseconds
constexpr int RS = 68;                       // floats of LDS per accumulator register of a tile (64 lanes, padded: the finishing threads read it transposed)

struct SeqArgs {
  SeqLayer a;
  unsigned* ring; unsigned ring_bytes, slot_bytes;
  int first_dir, groups, spins;
  unsigned* flag;
};

__device__ __forceinline__ float seq_sigm(float v) { return 1.0f / (1.0f + expf(-v)); }

__device__ __forceinline__ void seq_stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// The product of a block's weights with the state in a slot, asked for straight into matrix-instruction operands: group g (16
// values of k) of the slot is 1 KiB, lane l holds batch row l % 16 and k = 4 * (l / 16) .. + 3 of it; wavefront w takes the groups
// w, w + 4, ...  Up to 16 groups a wavefront are asked for together until none is empty; of more, the first SEQ_PART are, and the
// others follow behind them while the matrix instructions run (all blocks are about as far as each other: what comes after the
// first parts is there as a rule, and is asked for again where it is not).
//   last(): requests what the next step needs, behind everything this step asked for (ahead of the matrix instructions the step took
//   3.0 instead of 2.7 us at B 32, H 800, two directions: the next step's words queue behind it)
constexpr int SEQ_PART = 10;
template <int NIT, int CT>
struct SeqProduct {
  rnn_u32x4 h[NIT];
  rnn_f32x4 acc[CT];
  __device__ __forceinline__ void begin() {
#pragma unroll
    for (int ct = 0; ct < CT; ct++) acc[ct] = {0.f, 0.f, 0.f, 0.f};
  }
  template <int I0, int I1>
  __device__ __forceinline__ void ask(__amdgpu_buffer_rsrc_t rs, int slot, int groups) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
#pragma unroll
    for (int i = I0; i < I1; i++) h[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, wave + 4 * i < groups ? lane * 16 : (int)RNN_OOB, slot + (wave + 4 * i) * 1024, SEQ_COHERENT);
  }
  template <int I0, int I1>
  __device__ __forceinline__ void wait(__amdgpu_buffer_rsrc_t rs, int slot, int groups, int& spins, unsigned* flag) {
    for (;;) {
      unsigned top = 0;
#pragma unroll
      for (int i = I0; i < I1; i++)
#pragma unroll
        for (int c = 0; c < 4; c++) top = max(top, h[i][c]);
      if (__builtin_amdgcn_ballot_w64(top == SEQ_EMPTY) == 0) return;
      if (spins <= 0) { if (spins == 0 && (threadIdx.x & 63) == 0) *(volatile unsigned*)flag = 1u; spins = -1; return; }
      spins--;
      asm volatile("" ::: "memory");           // the words are loaded again
      ask<I0, I1>(rs, slot, groups);
    }
  }
  template <int I0, int I1>
  __device__ __forceinline__ void multiply(const float (&w)[CT][NIT][4]) {
#pragma unroll
    for (int i = I0; i < I1; i++)
#pragma unroll
      for (int c = 0; c < 4; c++)
#pragma unroll
        for (int ct = 0; ct < CT; ct++) acc[ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(h[i][c]), w[ct][i][c], acc[ct], 0, 0, 0);
  }
  template <int I0>
  __device__ __forceinline__ void rest(__amdgpu_buffer_rsrc_t rs, int slot, int groups, const float (&w)[CT][NIT][4], int& spins, unsigned* flag) {
    if constexpr (I0 < NIT) {
      constexpr int I1 = I0 + SEQ_PART < NIT ? I0 + SEQ_PART : NIT;
      wait<I0, I1>(rs, slot, groups, spins, flag);
      multiply<I0, I1>(w);
      rest<I1>(rs, slot, groups, w, spins, flag);
    }
  }
  template <class F>
  __device__ __forceinline__ void of_slot(__amdgpu_buffer_rsrc_t rs, int slot, int groups, const float (&w)[CT][NIT][4], int& spins, unsigned* flag, F last) {
    constexpr int I1 = NIT <= 16 ? NIT : SEQ_PART;
    begin();
    ask<0, I1>(rs, slot, groups);
    wait<0, I1>(rs, slot, groups, spins, flag);
    seq_stores_done();
    if constexpr (I1 < NIT) ask<I1, NIT>(rs, slot, groups);
    __builtin_amdgcn_sched_barrier(0);
    multiply<0, I1>(w);
    rest<I1>(rs, slot, groups, w, spins, flag);
    last();
  }
  // D layout of a 16 x 16 tile: lane holds column lane % 16, rows (batch) 4 * (lane / 16) + v
  __device__ __forceinline__ void to_lds(float* red) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
      for (int v = 0; v < 4; v++) red[((wave * CT + ct) * 4 + v) * RS + lane] = acc[ct][v];
    __syncthreads();
  }
};
// the sum of batch row b, column col of the block's CT * 16
template <int CT>
__device__ __forceinline__ float seq_sum(const float* red, int b, int col) {
  const float* p = red + ((col >> 4) * 4 + (b & 3)) * RS + 16 * (b >> 2) + (col & 15);
  return (p[0] + p[CT * 4 * RS]) + (p[2 * CT * 4 * RS] + p[3 * CT * 4 * RS]);
}
__device__ __forceinline__ void seq_put(__amdgpu_buffer_rsrc_t rs, int slot, int word, float v) {
  const unsigned bits = __float_as_uint(v);
  __builtin_amdgcn_raw_buffer_store_b32(bits == SEQ_EMPTY ? 0x7fc00000u : bits, rs, word * 4, slot, SEQ_COHERENT);
}
__device__ __forceinline__ void seq_empty(__amdgpu_buffer_rsrc_t rs, int slot, int word) { __builtin_amdgcn_raw_buffer_store_b32(SEQ_EMPTY, rs, word * 4, slot, SEQ_COHERENT); }

// Forward.  A block owns U units (all their gates: column g * U + u of its CT * 16 stands for gate g of unit u0 + u) for 16 batch rows.
// Thread t < 16 U finishes batch row (t / 4) % 16 of unit u0 + 4 * (t / 64) + t % 4: its word of the slot is then its own index.
template <int KIND, int NIT, int CT>
__global__ void __launch_bounds__(256, 1) k_rnn_seq_fwd(const SeqArgs s) {
  constexpr int NG = KIND == SEQ_ELMAN ? 1 : (KIND == SEQ_LSTM ? 4 : 3);
  constexpr int U = KIND == SEQ_ELMAN ? 16 : (CT >= 3 ? 16 : 4 * CT);
  static_assert(NG * U <= CT * 16, "the block's gates fit its columns");
  __shared__ float red_all[2][4 * CT * 4 * RS];
  const SeqLayer& a = s.a;
  const int T = a.T, B = a.B, H = a.H, ld = a.ld;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int d = s.first_dir + blockIdx.y, u0 = blockIdx.x * U, b0 = blockIdx.z * 16;
  const SeqDir& p = a.dir[d];
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)s.ring, 0, (int)s.ring_bytes, RNN_RSRC_FLAGS);
  const int tile = (int)((blockIdx.y * gridDim.z + blockIdx.z) * s.groups) * 1024;      // this direction's and batch tile's part of a slot
  float w[CT][NIT][4];
#pragma unroll
  for (int ct = 0; ct < CT; ct++) {
    const int cc = ct * 16 + (lane & 15), g = cc / U, u = u0 + cc % U;
#pragma unroll
    for (int i = 0; i < NIT; i++) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        const int k = 16 * (wave + 4 * i) + 4 * (lane >> 4) + c;
        w[ct][i][c] = (g < NG && u < H && k < H) ? p.W[(int64_t)(g * H + u) * H + k] : 0.f;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  const bool mine = t < 16 * U;                                   // a thread that finishes (and owns) words
  const int bl = (t >> 2) & 15, ul = 4 * (t >> 6) + (t & 3), b = b0 + bl, j = u0 + ul;
  const bool fin = mine && b < B && j < H;
  const int word = (u0 >> 4) * 256 + ((u0 & 15) >> 2) * 64 + t;   // of the tile
  float bi[NG], bh[NG], x[NG], c_prev = 0.f, h_prev = 0.f;
#pragma unroll
  for (int g = 0; g < NG; g++) { bi[g] = fin ? p.b1[g * H + j] : 0.f; bh[g] = fin ? p.b2[g * H + j] : 0.f; x[g] = 0.f; }
  if (fin && p.c0) c_prev = p.c0[(int64_t)b * H + j];
  if (fin && p.h0) h_prev = p.h0[(int64_t)b * H + j];
  auto fetch = [&](int step) {
    const int tt = d == 0 ? step : T - 1 - step;
#pragma unroll
    for (int g = 0; g < NG; g++)
      if (fin) x[g] = KIND == SEQ_ELMAN ? a.y[((int64_t)tt * B + b) * ld + d * H + j] : p.act[((int64_t)tt * B + b) * (NG * H) + g * H + j];
  };
  fetch(0);
  int spins = s.spins;
  SeqProduct<NIT, CT> m;
  for (int step = 0; step < T; step++) {
    if (spins >= 0) spins = s.spins;              // the bound is a step's
    const int tt = d == 0 ? step : T - 1 - step;
    float* red = red_all[step & 1];
    const bool use = step > 0 || (KIND != SEQ_ELMAN && p.h0 != nullptr);
    float xc[NG], sum[NG];
#pragma unroll
    for (int g = 0; g < NG; g++) sum[g] = 0.f;
    auto next = [&]() {
#pragma unroll
      for (int g = 0; g < NG; g++) xc[g] = x[g];
      if (step + 1 < T) fetch(step + 1);
    };
    if (step > 0) m.of_slot(rs, ((step - 1) % SEQ_RING) * (int)s.slot_bytes + tile, s.groups, w, spins, s.flag, next);
    else {
      next();
      m.begin();
      if constexpr (KIND != SEQ_ELMAN) if (use) {
#pragma unroll
        for (int i = 0; i < NIT; i++)
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const int k = 16 * (wave + 4 * i) + 4 * (lane >> 4) + c, br = b0 + (lane & 15);
            m.h[i][c] = k < H && br < B ? __float_as_uint(p.h0[(int64_t)br * H + k]) : 0u;
          }
        m.template multiply<0, NIT>(w);
      }
    }
    if (use) {
      m.to_lds(red);
      if (mine) {
#pragma unroll
        for (int g = 0; g < NG; g++) sum[g] = seq_sum<CT>(red, bl, g * U + ul);
      }
    }
    if (!mine) continue;
    float hn, o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f, ax = 0.f;
    if constexpr (KIND == SEQ_ELMAN) {
      const float v = ((xc[0] + bi[0]) + bh[0]) + sum[0];
      hn = a.relu ? (v < 0.f ? 0.f : v) : tanhf(v);
    } else if constexpr (KIND == SEQ_LSTM) {
      o0 = seq_sigm(((xc[0] + sum[0]) + bi[0]) + bh[0]); o1 = seq_sigm(((xc[1] + sum[1]) + bi[1]) + bh[1]);
      o2 = tanhf(((xc[2] + sum[2]) + bi[2]) + bh[2]); o3 = seq_sigm(((xc[3] + sum[3]) + bi[3]) + bh[3]);
      ax = c_prev = o1 * c_prev + o0 * o2;
      hn = o3 * tanhf(ax);
    } else {
      o0 = seq_sigm(((xc[0] + bi[0]) + bh[0]) + sum[0]); o1 = seq_sigm(((xc[1] + bi[1]) + bh[1]) + sum[1]);
      ax = sum[2] + bh[2];
      o2 = tanhf((xc[2] + bi[2]) + o0 * ax);
      hn = (1.f - o1) * o2 + o1 * h_prev;
      h_prev = hn;
    }
    if (step + 1 < T) {
      seq_put(rs, (step % SEQ_RING) * (int)s.slot_bytes + tile, word, fin ? hn : 0.f);
      if (step >= 2) seq_empty(rs, ((step - 2) % SEQ_RING) * (int)s.slot_bytes + tile, word);
    }
    if (fin) {
      a.y[((int64_t)tt * B + b) * ld + d * H + j] = hn;
      if constexpr (KIND != SEQ_ELMAN) {
        float* q = p.act + ((int64_t)tt * B + b) * (NG * H) + j;
        q[0] = o0; q[H] = o1; q[2 * H] = o2;
        if constexpr (KIND == SEQ_LSTM) q[3 * H] = o3;
        p.aux[((int64_t)tt * B + b) * H + j] = ax;
      }
    }
  }
}

// Backward.  What travels is the hidden-side gradient of the pre-activations; a block sums it over all gate rows for 16 units and
// 16 batch rows (group ug * NG + gate of the slot: 16 units of one gate), and forms those of its units one step earlier.
template <int KIND, int NIT>
__global__ void __launch_bounds__(256, 1) k_rnn_seq_bwd(const SeqArgs s) {
  constexpr int NG = KIND == SEQ_ELMAN ? 1 : (KIND == SEQ_LSTM ? 4 : 3);
  __shared__ float red_all[2][4 * 4 * RS];
  const SeqLayer& a = s.a;
  const int T = a.T, B = a.B, H = a.H, ld = a.ld;
  const int t = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
  const int d = s.first_dir + blockIdx.y, u0 = blockIdx.x * 16, b0 = blockIdx.z * 16;
  const SeqDir& p = a.dir[d];
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)s.ring, 0, (int)s.ring_bytes, RNN_RSRC_FLAGS);
  const int tile = (int)((blockIdx.y * gridDim.z + blockIdx.z) * s.groups) * 1024;
  float w[1][NIT][4];
#pragma unroll
  for (int i = 0; i < NIT; i++) {
    const int g = wave + 4 * i, ug = g / NG, gate = g - ug * NG;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      const int k = 16 * ug + 4 * (lane >> 4) + c, u = u0 + (lane & 15);
      w[0][i][c] = (g < s.groups && k < H && u < H) ? p.W[(int64_t)(gate * H + k) * H + u] : 0.f;
    }
  }
  const int bl = (t >> 2) & 15, ul = 4 * (t >> 6) + (t & 3), b = b0 + bl, j = u0 + ul;
  const bool fin = b < B && j < H;
  const int word = (u0 >> 4) * NG * 256 + t;
  // LSTM: i f g o, cell, previous cell, dy; GRU: r z n, q, previous hidden, dy; Elman: h, dy
  float v[4], ax = 0.f, pv = 0.f, gy = 0.f, nv[4], nax = 0.f, npv = 0.f, ngy = 0.f;
#pragma unroll
  for (int g = 0; g < 4; g++) { v[g] = 0.f; nv[g] = 0.f; }
  auto fetch = [&](int k) {
    if (!fin) return;
    const int tt = d == 0 ? T - 1 - k : k, tp = d == 0 ? tt - 1 : tt + 1;
    const int64_t row = (int64_t)tt * B + b, prow = (int64_t)tp * B + b;
    ngy = a.dy[row * ld + d * H + j];
    if constexpr (KIND == SEQ_ELMAN) nv[0] = a.y[row * ld + d * H + j];
    else {
#pragma unroll
      for (int g = 0; g < NG; g++) nv[g] = p.act[row * (NG * H) + g * H + j];
      nax = p.aux[row * H + j];
      if constexpr (KIND == SEQ_LSTM) npv = k + 1 < T ? p.aux[prow * H + j] : (p.c0 ? p.c0[(int64_t)b * H + j] : 0.f);
      else npv = k + 1 < T ? a.y[prow * ld + d * H + j] : (p.h0 ? p.h0[(int64_t)b * H + j] : 0.f);
    }
  };
  fetch(0);
  int spins = s.spins;
  float carry = 0.f;                    // LSTM: cell gradient, GRU: dh * z
  SeqProduct<NIT, 1> m;
  for (int k = 0; k < T; k++) {
    if (spins >= 0) spins = s.spins;              // the bound is a step's
    const int tt = d == 0 ? T - 1 - k : k;
    const int64_t row = (int64_t)tt * B + b;
    float* red = red_all[k & 1];
    float tc = 0.f, sum = 0.f;
    auto next = [&]() {
#pragma unroll
      for (int g = 0; g < 4; g++) v[g] = nv[g];
      ax = nax; pv = npv; gy = ngy;
      if (k + 1 < T) fetch(k + 1);
    };
    if (k > 0) {
      m.of_slot(rs, ((k - 1) % SEQ_RING) * (int)s.slot_bytes + tile, s.groups, w, spins, s.flag, next);
      m.to_lds(red);
      sum = seq_sum<1>(red, bl, ul);
    } else next();
    if constexpr (KIND == SEQ_LSTM) tc = tanhf(ax);
    float o[4];
    if constexpr (KIND == SEQ_ELMAN) {
      const float g = gy + sum;
      o[0] = a.relu ? (v[0] > 0.f ? g : 0.f) : g * (1.0f - v[0] * v[0]);
    } else if constexpr (KIND == SEQ_LSTM) {
      const float dh = gy + sum;
      const float dcc = dh * v[3] * (1.f - tc * tc) + carry;
      o[0] = dcc * v[2] * v[0] * (1.f - v[0]);
      o[1] = dcc * pv * v[1] * (1.f - v[1]);
      o[2] = dcc * v[0] * (1.f - v[2] * v[2]);
      o[3] = dh * tc * v[3] * (1.f - v[3]);
      carry = dcc * v[1];
    } else {
      const float dh = gy + (carry + sum);
      const float dn = dh * (1.f - v[1]) * (1.f - v[2] * v[2]);
      o[1] = dh * (pv - v[2]) * v[1] * (1.f - v[1]);
      o[0] = dn * ax * v[0] * (1.f - v[0]);
      o[2] = dn * v[0];
      o[3] = dn;                        // the input side of the n gate
      carry = dh * v[1];
    }
    if (k + 1 < T) {
#pragma unroll
      for (int g = 0; g < NG; g++) seq_put(rs, (k % SEQ_RING) * (int)s.slot_bytes + tile, word + g * 256, fin ? o[g] : 0.f);
      if (k >= 2)
#pragma unroll
        for (int g = 0; g < NG; g++) seq_empty(rs, ((k - 2) % SEQ_RING) * (int)s.slot_bytes + tile, word + g * 256);
    }
    if (fin) {
      if constexpr (KIND == SEQ_ELMAN) a.dpre[row * ld + d * H + j] = o[0];
      else if constexpr (KIND == SEQ_LSTM) {
        float* q = p.act + row * (4 * H) + j;
        q[0] = o[0]; q[H] = o[1]; q[2 * H] = o[2]; q[3 * H] = o[3];
      } else {
        float* q = p.act + row * (3 * H) + j;
        float* e = p.dgh + row * (3 * H) + j;
        q[0] = o[0]; q[H] = o[1]; q[2 * H] = o[3];
        e[0] = o[0]; e[H] = o[1]; e[2 * H] = o[2];
      }
    }
  }
}

__global__ void __launch_bounds__(256) k_seq_clear(uint4* p, int n16) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n16; i += gridDim.x * 256) p[i] = make_uint4(SEQ_EMPTY, SEQ_EMPTY, SEQ_EMPTY, SEQ_EMPTY);
}

unsigned* g_flag = nullptr;
unsigned* g_flag_dev = nullptr;
bool g_given_up = false;              // a wait has run out: the card is shared, or something else keeps blocks from it
unsigned* g_ring = nullptr;           // one, since all launches of this kind follow each other on the main stream (replays: lh_graph_launch)
size_t g_ring_bytes = 0;

// How a launch is laid out: `ct` column tiles and `units` units a block, gx * gz blocks per direction, `dirs` directions per launch,
// `groups` groups of 16 k in a slot's tile, `nit` of them per wavefront.  Units per block: as few as leave every block a compute
// unit of its own (a step's matrix instructions, 0.7 us per column tile at H 800, are then spread widest); both directions in one
// launch where they fit, one after the other where only one does.  Layers that fit neither way (more than 16 batch rows times 16
// units per compute unit: B 64 from H 1024 on; LSTM backward above H 800, where the largest form built, 50 groups a wavefront and 436
// of 512 registers, ends) keep one launch per step.
struct Plan { bool ok; int ct, units, nit, gx, gz, dirs, groups; };
Plan plan_of(int kind, bool backward, int D, int T, int B, int H) {
  Plan p{};
  const int ng = kind == SEQ_ELMAN ? 1 : (kind == SEQ_LSTM ? 4 : 3), ug = (int)cdiv(H, 16);
  p.gz = (int)cdiv(B, 16);
  p.groups = backward ? ug * ng : ug;
  p.nit = (int)cdiv(p.groups, 4);
  // A short sequence does not earn back the clearing of the ring and the weights' way into the registers: B 32, H 800, forward and
  // backward, one launch per step / one launch: tanh T 6 159 / 166 us, T 12 250 / 254, T 20 307 / 230; LSTM T 3 153 / 161;
  // GRU (B 4, H 64) T 6 164 / 91.
  if (T < (kind == SEQ_ELMAN ? 12 : 4) || p.gz > g_num_cu) return p;
  const int cts[4] = {1, 2, kind == SEQ_LSTM ? 4 : 3, 0};
  for (int dirs = D; dirs >= 1 && !p.ok; dirs--)
    for (int i = 0; i < (kind == SEQ_ELMAN || backward ? 1 : 3) && !p.ok; i++) {
      p.ct = cts[i];
      p.units = kind == SEQ_ELMAN || backward ? 16 : (p.ct >= 3 ? 16 : 4 * p.ct);
      p.gx = ug * (16 / p.units);
      p.dirs = dirs;
      p.ok = (int64_t)p.gx * p.gz * dirs <= g_num_cu;
    }
  // Two launches one after the other in place of both directions at once: a forward pass of few units has too little to do in each
  // (one launch per step | two of these: B 512, H 128 T 12 54.6 | 57.7 us, T 24 98.1 | 99.6, T 48 185 | 179; B 1024, H 64 T 24 94.6 | 98.0, T 48
  // 172 | 175, T 100 342 | 337; B 256, H 256 T 12 60.8 | 59.0).
  if (kind == SEQ_ELMAN && !backward && p.dirs < D && ug <= 8 && T < 48) p.ok = false;
  const int most = backward ? (kind == SEQ_ELMAN ? 32 : 50) : (p.ct >= 4 ? 13 : 16);
  if (p.nit > (kind == SEQ_ELMAN ? 32 : most)) p.ok = false;
  return p;
}
size_t slot_bytes(const Plan& p) { return (size_t)p.dirs * p.gz * p.groups * 1024; }
}  // namespace

bool rnn_seq_takes(int kind, bool backward, int D, int T, int B, int H) {
  if (!rnn_mfma_enabled() || g_stream_cur != g_stream_raw || g_ring == nullptr) return false;
  if (*(volatile unsigned*)g_flag != 0) g_given_up = true;
  if (const char* e = getenv("LH_RNN_SEQ")) {        // (the tests' switch: 0 one launch per time step, 1 the one launch again after a wait that ran out)
    if (e[0] == '0') return false;
    if (e[0] == '1') g_given_up = false;
  }
  if (g_given_up) return false;
  const Plan p = plan_of(kind, backward, D, T, B, H);
  return p.ok && SEQ_RING * slot_bytes(p) <= g_ring_bytes;
}

void rnn_seq_run(int kind, bool backward, const SeqLayer& a) {
  const Plan p = plan_of(kind, backward, a.D, a.T, a.B, a.H);
  if (!p.ok) { LH_FAIL("recurrence: no launch plan for T%d B%d H%d", a.T, a.B, a.H); return; }
  SeqArgs s;
  if (g_capturing) g_captured_seq = true;
  g_rnn_seq_runs++;
  s.a = a; s.ring = g_ring; s.slot_bytes = (unsigned)slot_bytes(p); s.ring_bytes = SEQ_RING * s.slot_bytes;
  s.groups = p.groups; s.flag = g_flag_dev; s.spins = SEQ_SPINS;
  if (const char* e = getenv("LH_RNN_SEQ_SPINS")) s.spins = atoi(e);          // (the tests' switch: a wait that gives up at once)
  const dim3 grid((unsigned)p.gx, (unsigned)p.dirs, (unsigned)p.gz);
  for (s.first_dir = 0; s.first_dir < a.D; s.first_dir += p.dirs) {
    const int n16 = (int)(s.ring_bytes / 16);
    hipLaunchKernelGGL(k_seq_clear, dim3((unsigned)stream_grid(n16, 1024)), dim3(256), 0, g_stream, (uint4*)s.ring, n16);
#define FWD(K, N, C) hipLaunchKernelGGL((k_rnn_seq_fwd<K, N, C>), grid, dim3(256), 0, g_stream, s)
#define BWD(K, N) hipLaunchKernelGGL((k_rnn_seq_bwd<K, N>), grid, dim3(256), 0, g_stream, s)
#define FWD_N(K, C) do { if (p.nit <= 4) FWD(K, 4, C); else if (p.nit <= 8) FWD(K, 8, C); else if (p.nit <= 13) FWD(K, 13, C); else FWD(K, 16, C); } while (0)
    if (kind == SEQ_ELMAN && !backward) { if (p.nit <= 16) FWD_N(SEQ_ELMAN, 1); else FWD(SEQ_ELMAN, 32, 1); }
    else if (kind == SEQ_ELMAN) { if (p.nit <= 4) BWD(SEQ_ELMAN, 4); else if (p.nit <= 8) BWD(SEQ_ELMAN, 8); else if (p.nit <= 13) BWD(SEQ_ELMAN, 13); else if (p.nit <= 16) BWD(SEQ_ELMAN, 16); else BWD(SEQ_ELMAN, 32); }
    else if (kind == SEQ_LSTM && !backward) { if (p.ct == 1) FWD_N(SEQ_LSTM, 1); else if (p.ct == 2) FWD_N(SEQ_LSTM, 2); else if (p.nit <= 4) FWD(SEQ_LSTM, 4, 4); else if (p.nit <= 8) FWD(SEQ_LSTM, 8, 4); else FWD(SEQ_LSTM, 13, 4); }
    else if (kind == SEQ_GRU && !backward) { if (p.ct == 1) FWD_N(SEQ_GRU, 1); else if (p.ct == 2) FWD_N(SEQ_GRU, 2); else FWD_N(SEQ_GRU, 3); }
    else if (kind == SEQ_LSTM) { if (p.nit <= 8) BWD(SEQ_LSTM, 8); else if (p.nit <= 16) BWD(SEQ_LSTM, 16); else if (p.nit <= 32) BWD(SEQ_LSTM, 32); else BWD(SEQ_LSTM, 50); }
    else { if (p.nit <= 8) BWD(SEQ_GRU, 8); else if (p.nit <= 16) BWD(SEQ_GRU, 16); else if (p.nit <= 32) BWD(SEQ_GRU, 32); else BWD(SEQ_GRU, 50); }
#undef FWD_N
#undef BWD
#undef FWD
  }
}

bool rnn_seq_setup() {
  if (g_flag) return true;
  if (hipHostMalloc((void**)&g_flag, 64, hipHostMallocDefault) != hipSuccess || hipHostGetDevicePointer((void**)&g_flag_dev, g_flag, 0) != hipSuccess) {
    LH_FAIL("recurrence: cannot allocate the pinned flag"); return false;
  }
  *g_flag = 0; g_given_up = false;
  // a slot has at most four groups (the gates of a backward pass) of 1 KiB per block, and there is a compute unit for every block
  g_ring_bytes = SEQ_RING * 4 * 1024 * (size_t)g_num_cu;
  g_ring = (unsigned*)persistent_alloc(g_ring_bytes);
  if (g_ring == nullptr) { LH_FAIL("recurrence: cannot allocate the ring of %zu bytes", g_ring_bytes); return false; }
  return true;
}
void rnn_seq_release() {
  if (g_flag) (void)hipHostFree(g_flag);
  persistent_free(g_ring);
  g_flag = g_flag_dev = g_ring = nullptr;
}
bool rnn_seq_report_timeout() {
  if (g_flag == nullptr || *(volatile unsigned*)g_flag == 0) return false;
  *g_flag = 0;
  g_given_up = true;
  LH_FAIL("recurrent layer: a block waited too long for the others; the layer's results are incomplete (the layers that follow take one launch per time step)");
  return true;
}
}  // namespace lh
