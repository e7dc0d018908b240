// Layout of the packed parameters of the 3-256-256-256-3 softplus field
// (mo_flow256_pack), shared by the FP32-MFMA kernels (mo_flow256.hip) and
// the split-bf16 ones (mo_flow256_split.hip).
#pragma once

#include "mo_common.h"

namespace mo {

constexpr int kH = 256;
// offsets in floats
constexpr int kPW0 = 0;                 // W0 [256][4] (k = 3 padded with 0)
constexpr int kPB0 = kPW0 + kH * 4;     // b0 [256]
constexpr int kPW1 = kPB0 + kH;         // W1 fragments [8 col blocks][32 groups][64 lanes][4]
constexpr int kPB1 = kPW1 + kH * kH;
constexpr int kPW2 = kPB1 + kH;
constexpr int kPB2 = kPW2 + kH * kH;
constexpr int kPW3 = kPB2 + kH;         // W3 [3][256]
constexpr int kPB3 = kPW3 + 3 * kH;     // b3 [3] (+1 pad)
constexpr int kPW1T = kPB3 + 4;         // W1^T fragments (backward: dH1 = dA2 W1)
constexpr int kPW2T = kPW1T + kH * kH;  // W2^T fragments (backward: dH2 = dA3 W2)
// Split-bf16 fragments of W1, W2, W1^T, W2^T: a weight is the sum of three
// bf16 (high, middle, low: 24 significant bits, so the sum is exact), each
// plane in the A-operand order of v_mfma_f32_32x32x16_bf16,
// [8 row blocks][16 k-steps][64 lanes][8]: lane l holds row 32 rb + l % 32,
// k = 16 ks + 8 (l / 32) + 0..7.
constexpr int kPSplit = kPW2T + kH * kH;
constexpr int kSplitPlane = kH * kH / 2;         // floats of one plane
constexpr int kSplitLayer = 3 * kSplitPlane;     // floats of one matrix
constexpr int kPacked = kPSplit + 4 * kSplitLayer;
static_assert(kPSplit % 4 == 0, "fragments are read as 16-byte words");

}  // namespace mo
