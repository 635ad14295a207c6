// Convolution -> batch norm with running statistics [-> + shortcut] [-> relu in place] as one launch: what the deferred work
// (lh_defer.hip) hands to the convolution (lh_conv.hip), and the pass over a finished convolution where its launch plan needs one.
#pragma once
#include "lh_common.h"

namespace lh {
// out = act(bn(conv(x) + bias) + shortcut); shortcut may be nullptr, relu 0 leaves the values as they are.  `out` overlaps no operand.
// (weak: the deferred work does not park such a chain in a build without it)
__attribute__((weak)) void conv2d_bn_infer_now(const float* x, const float* w, const float* bias, int N, int C, int H, int W, int K, int R, int S, int sH, int sW, int pH, int pW,
                                               const float* gamma, const float* beta, const float* mean, const float* var, float eps, const float* shortcut, float* out, int relu);
// y = act(bn(x) + shortcut) on its own, y == x allowed
__attribute__((weak)) void bn_infer_now(const float* x, const float* gamma, const float* beta, const float* mean, const float* var, float eps, const float* shortcut, float* y,
                                        int relu, int N, int C, int HW);
namespace lazy {
bool park_bn_infer(const float* x, const float* gamma, const float* beta, const float* mean, const float* var, float* y, int N, int C, int HW, float eps);
void filters_released(const char* from);       // the arena above `from` is released: what is remembered of the chains of filters there goes too
}
const char* arena_end();
}  // namespace lh
