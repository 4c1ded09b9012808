// conv_weights.h — the order of a 3x3 convolution's bf16 weights, as the lanes
// of k_conv (denoise.hip) hold them: [K-step][16 outputs][lane][8], K = (tap,
// input channel) padded with zeros to whole steps of 32; lane l holds output
// l % 16 and the (l / 16)-th 8 of a step's K. Plain constexpr functions: the
// kernel that prepares the weights and programs without a GPU use the same.
#pragma once

namespace rgrt {

// Weights of a convolution of kin to nout channels in that order, padding included.
constexpr int conv_weights(int kin, int nout) { return (9 * kin + 31) / 32 * 32 * nout; }

struct ConvWeight {
    int tap, in, out; // tap 9 and above: padding
};

constexpr ConvWeight conv_weight_at(int e, int kin, int nout)
{
    const int lane = (e >> 3) & 63, block = e >> 9, nt = nout / 16;
    const int k = 32 * (block / nt) + 8 * (lane >> 4) + (e & 7);
    return {k / kin, k % kin, 16 * (block % nt) + (lane & 15)};
}

// Where weight e of a layer of cin to cout channels comes from in its fp32
// master [9][cin][cout]; -1: padding (zero).
constexpr int conv_master_index(int e, int cin, int cout)
{
    const ConvWeight w = conv_weight_at(e, cin, cout);
    return w.tap < 9 ? (w.tap * cin + w.in) * cout + w.out : -1;
}

// The same for the layer's data gradient, a convolution of cout to cin
// channels with mirrored taps.
constexpr int conv_gradient_master_index(int e, int cin, int cout)
{
    const ConvWeight w = conv_weight_at(e, cout, cin);
    return w.tap < 9 ? ((8 - w.tap) * cin + w.out) * cout + w.in : -1;
}

} // namespace rgrt
