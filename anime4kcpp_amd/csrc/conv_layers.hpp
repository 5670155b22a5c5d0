// The conv3x3 layers of the layer-by-layer networks (ACNet<8>, ArtCNN<F>, FSRCNNX<F>): their
// epilogues (LayerMode), which keep the reference's separately rounded steps after the conv sum
// (Common.hpp:116-164, 227-288, 290-341).  The 8-channel layers are conv8_rows.hpp's, the 16- and
// 32-channel ones convf_rows.hpp's.
//   kRelu          max(v, 0)                                        ArtCNN body
//   kPrelu         max(v, 0) + a * min(v, 0)                        ACNet<8>, FSRCNNX body
//   kAddFeat       v * 1 + feat                                     ArtCNN's last F -> F
//   kPreluConv1x1  PReLU, then conv1x1 F -> F + bias, * 1 + feat, PReLU
//                                                                   FSRCNNX's last block
//   kShuffle       conv F -> 4, pixel shuffle to 2x                 ArtCNN, FSRCNNX tail
//   kShuffleSrc    the same, + the source pixel                     ACNet<8> final
//   kReluDeconv    ReLU, then the 2x2 stride-2 deconv 8 -> 1 to 2x  ACNetLegacy's last layer
//                  (Common.hpp:344-393), layer by layer
#pragma once

#include "acnet_device.hpp"
#include "acnet_kernels.hpp"

namespace achip {

#pragma clang fp contract(off)

enum LayerMode : int { kRelu = 0, kPrelu = 1, kAddFeat = 2, kPreluConv1x1 = 3, kShuffle = 4, kShuffleSrc = 5,
                       kReluDeconv = 6 };

// Arguments of one layer launch; a mode leaves the fields it does not read null.
struct LayerArgs {
    const float* wa;        // this layer's per-lane A operands
    const float* bias;      // F biases (4 for the shuffle modes)
    const float* alpha;     // F PReLU slopes
    const float* w1;        // conv1x1 A operands
    const float* b1;        // conv1x1 biases (F)
    const float* alpha1;    // F PReLU slopes after the skip connection
    const float4* feat;     // skip-connection map, same pitch as the input map
    const float* k2;        // deconv weights k2[c][q] (kReluDeconv)
    const void* src;        // source image (kShuffleSrc)
    long ss;
    void* dst;              // output image (shuffle modes)
    long ds;
};

// PReLU (Common.hpp:42-49): max(v, 0) + alpha * min(v, 0), each step rounded
__device__ inline float prelu(float v, float alpha)
{
    return __fadd_rn(fmaxf(v, 0.0f), __fmul_rn(alpha, fminf(v, 0.0f)));
}

__device__ inline float add_skip(float v, float f) { return __fadd_rn(__fmul_rn(v, 1.0f), f); }

} // namespace achip
