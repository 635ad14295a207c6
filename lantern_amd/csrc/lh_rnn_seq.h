// The recurrence of a layer as ONE launch (lh_rnn_seq.hip): what lh_rnn.hip and lh_rnn_gated.hip ask for.
#pragma once
#include "lh_common.h"

namespace lh {
enum { SEQ_ELMAN = 0, SEQ_LSTM = 1, SEQ_GRU = 2 };
// One direction of a layer.  Forward: act holds the input projection [T, B, gates * H] (LSTM: gate activations on exit, GRU: r, z, n;
// the Elman layer's projection lies in y itself, act is not used), aux [T, B, H] receives the cell state (GRU: W_hn h + b_hn).
// Backward: act holds the activations on entry and the pre-activation gradients on exit, dgh [T, B, 3H] the GRU's hidden-side ones.
struct SeqDir {
  const float* W;                    // W_hh [gates * H, H]
  const float* b1; const float* b2;  // b_ih, b_hh (forward)
  const float* h0; const float* c0;  // initial state [B, H] or nullptr (the Elman layer's has been added to its projection)
  float* act; float* aux; float* dgh;
};
struct SeqLayer {
  SeqDir dir[2];
  float* y;                          // [T, B, ld]: hidden states (Elman forward: the projection on entry)
  const float* dy; float* dpre;      // backward: incoming gradient; Elman: pre-activation gradient out, both [T, B, ld]
  int D, T, B, H, ld, relu;          // relu: the Elman layer's activation (0: tanh)
};
// Does the layer run that way?  (see the rule in lh_rnn_seq.hip)
bool rnn_seq_takes(int kind, bool backward, int D, int T, int B, int H);
// The whole recurrence on the current stream, in one launch or one per direction.
void rnn_seq_run(int kind, bool backward, const SeqLayer& a);
extern int64_t g_rnn_seq_runs;     // passes run (or recorded) that way since the library was loaded
extern bool g_captured_seq;        // the graph being recorded holds such a launch
bool rnn_seq_setup();              // the ring and the flag word, for lh_setup / lh_cleanup
void rnn_seq_release();
bool rnn_seq_report_timeout();     // true (and an error reported) if a launch gave up waiting for a block since the last look
}  // namespace lh
