// Fused layers of the FNO in bfloat16 (fno_layer.hip).
#pragma once
#include <cstdint>

#include "common.h"

namespace tara {

struct FnoLayerArgs {
    int n, c, q2, nb;         // grid, width, 2 MX, samples
    int act;                  // GELU after the mixing
    // inputs
    const uint16_t* v;        // [b][c][y][x] (null: the lift of om)
    const float* om;          // [b][y][x]
    const float* sig;         // [b]
    const float* wl;          // lift weights and biases [c]
    const float* bl;
    const uint16_t* z;        // [b c][y][q2]
    const uint16_t* w;        // padded mixing weights [CP][CP]
    const float* bias;        // [c]
    const uint16_t* hxt;      // inverse x transform, transposed and padded [256][32]
    const uint16_t* fx;       // forward x transform, padded [32][256]
    const uint16_t* w1;       // padded projection weights [2 CP][CP]
    const float* b1;          // padded [2 CP]
    const float* w2;          // padded [2 CP]
    const float* b2;
    // outputs (null: not wanted)
    uint16_t* vn;             // [b][c][y][x]
    uint16_t* t1;             // [y][q2][b c]
    float* v32;               // training: activation and pre-activation in FP32
    float* pre;
    float* out;               // prediction [b][y][x] (projection and residual)
};

// Whether the fused layers take this network.
bool fno_fused_ok(int n, int c, int q2);
// Rows (= columns) of the padded weight blocks: 32 or 64.
int fno_pad(int c);
// T1 of the lifted input.
int fno_lift_x(const FnoLayerArgs& a, hipStream_t st);
// One layer after its inverse y transform (z): v <- act(inverse x of z + W v + b),
// then what the next step of the network reads: T1, or the projected output.
int fno_layer(const FnoLayerArgs& a, hipStream_t st);
// Padded copies of the weights (bfloat16 matrices, FP32 vectors), cp = fno_pad(c).
struct FnoPadArgs {
    int c, cp, layers;
    const float *w, *w1, *b1, *w2;  // [layers][c][c], [2 c][c], [2 c], [2 c]
    uint16_t *wp, *w1p;             // [layers][cp][cp], [2 cp][cp]
    float *b1p, *w2p;               // [2 cp]
};
int fno_pad_weights(const FnoPadArgs& a, hipStream_t st);

}  // namespace tara
