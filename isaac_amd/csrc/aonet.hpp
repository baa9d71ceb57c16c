// Kernels of the learned occlusion pass: a U-Net over the G-buffer whose 3x3
// convolutions run as implicit GEMMs on the gfx950 matrix cores
// (v_mfma_f32_16x16x32_f16: FP16 operands, FP32 accumulation).
//
// Tensors are channels-last: element (n, y, x, c) at ((n*H + y)*W + x)*C + c.
// Forward convolution weights are [Cout][Kp] FP16 with k = tap*Cin + ci (tap =
// ky*3 + kx reads pixel (y + ky - 1, x + kx - 1), zero padding), Kp = 9*Cin
// rounded up to a multiple of 32 with zero columns.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include <cstdint>

namespace isaac_hip
{
    // Input of a convolution: channels [0, ca) of pixel (y, x) come from `up` at
    // (y/2, x/2) (nearest-neighbour upsampling of an (h/2, w/2, ca) tensor) and
    // channels [ca, cin) from `x` (h, w, cin - ca); with up == nullptr all cin
    // channels come from x.  This fuses the decoder's upsample + concat.
    struct ConvArgs
    {
        const _Float16* x; // [n][h][w][cin - ca]
        const _Float16* up; // [n][h/2][w/2][ca] or nullptr
        int32_t ca; // channels from `up` (a multiple of 4; 0 without `up`)
        const _Float16* w; // [cout][kp]
        const float* bias; // [cout] (forward only)
        void* y; // forward: _Float16 [n][h][w][cout] = relu(conv + bias) (nullable); backward data: float
        int32_t n, h, w_, cin, kp; // cin a multiple of 4
        // forward only (launch_conv_fwd), all optional:
        _Float16* pool; // [n][h/2][w/2][cout]: 2x2 average of the FP16 activation (h, w even)
        float* head; // cout 16: [n][imgH][imgW] = clamp(act . headW[0..15] + headW[16], 0, 1)
        const float* headW;
        int32_t imgW, imgH;
    };

    // Backward data of a layer: y (FP32 [n][h][w][cout]) = 3x3 convolution of x (the
    // layer's dz) with its flipped, transposed weights ([cout][kp], kp as for the forward
    // weights of a.cin channels); `cout` here is the layer's cin and a.cin its cout:
    // (a.cin, cout) = (16, 16) (16, 48) (32, 16) (32, 32) (32, 96) (64, 32) (64, 64) (64, 128).
    hipError_t launch_conv_bwd(const ConvArgs& a, int cout, size_t max_lds, hipStream_t s);

    // Forward layer y = relu(conv(x) + bias) on v_mfma_f32_16x16x32_f16 for the
    // network's (cin, cout, ca) shapes: (8,16,0) (16,16,0) (16,32,0) (32,32,0)
    // (32,64,0) (64,64,0) (128,64,64) (96,32,64) (48,16,32); weights [cout][kp] with
    // kp = 9*cin rounded up to a multiple of 32 (zero columns).  The fused pool and
    // head outputs are formed from the activation as it is stored (binary16).
    hipError_t launch_conv_fwd(const ConvArgs& a, int cout, size_t max_lds, hipStream_t s);

    // Where the gradient of a layer's output comes from
    enum DyMode : int32_t
    {
        kDyPlain = 0, // g [n][h][w][gStride], channels gOff ..
        kDyUpsampled = 1, // g [n][2h][2w][gStride], channels gOff ..: the sum of the 2x2 positions that read it
        kDySkipAndPool = 2 // as kDyPlain, plus gPool [n][h/2][w/2][cout] / 4 (the 2x2 average pool's gradient)
    };
    // One layer of the weight gradient: dz = half(dy * (act > 0)) is formed and stored, and
    // dw / db are the sums over all pixels (launch_conv_grad, then launch_grad_sum)
    struct GradLayer
    {
        const _Float16* x; // the layer's input, as in ConvArgs
        const _Float16* up;
        int32_t ca, cin, cout; // cout 16, 32 or 64
        const _Float16* act; // the layer's output [n][h][w][cout]
        int32_t dyMode;
        const float* g;
        int32_t gStride, gOff; // multiples of 4
        const float* gPool;
        _Float16* dz; // out: [n][h][w][cout]
        float* partial; // grad_shape(...).partial floats
        float* partialBias; // grad_shape(...).splits * cout floats
        float* dw; // out: [cout][9][cin] (the master weight layout)
        float* db; // out: [cout]
        int32_t n, h, w;
    };
    struct GradShape
    {
        int32_t ct, groups, splits; // 16-channel input blocks per workgroup, groups of them, pixel splits
        size_t partial; // floats
    };
    constexpr int kGradMaxLayers = 11;
    GradShape grad_shape(int cin, int cout, int n, int h, int w);
    hipError_t launch_conv_grad(const GradLayer& L, hipStream_t s);
    // dw and db of all layers from their partial sums
    hipError_t launch_grad_sum(const GradLayer* layers, int count, hipStream_t s);

    // network input from a G-buffer window: 8 channels (depth / scale or 0, background
    // flag, normal xyz, 0, 0, 0); pixels outside the image are background.  With `ao`
    // and `target` set, also copies the occlusion term as the training target.
    struct FeatureArgs
    {
        const float* depth; // [imgH][imgW]
        const float* normal; // [imgH][imgW][3]
        const float* ao; // [imgH][imgW] or nullptr
        int32_t imgW, imgH;
        float invScale;
        const int32_t* origin; // per batch item: x0, y0 of the window (device), or nullptr = (0, 0)
        _Float16* x; // [n][h][w][8]
        float* target; // [n][h][w] or nullptr
        int32_t n, h, w;
        int64_t imgStride; // elements between the images of consecutive items (0: one image)
        const float* invScaleItem; // per item 1 / scale (device), or nullptr = invScale
    };
    hipError_t launch_features(const FeatureArgs& a, hipStream_t s);

    // Training: out = d0 . wh + bh (wh[16] = bh); loss += sum (out - t)^2;
    // gwh[0..15] += sum dout * d0, gwh[16] += sum dout; dd0 = dout * wh with
    // dout = 2 (out - t); `out` (nullable) receives the raw outputs
    hipError_t launch_head_train(
        const _Float16* d0,
        const float* wh,
        const float* target,
        float* loss,
        float* gwh,
        float* dd0,
        float* out,
        int64_t npx,
        hipStream_t s);

    // Adam over the flat FP32 parameter vector (gradients scaled by gscale first)
    hipError_t launch_adam(
        float* w,
        const float* g,
        float* m,
        float* v,
        int64_t count,
        float lr,
        float b1,
        float b2,
        float eps,
        float c1,
        float c2,
        float gscale,
        hipStream_t s);
    // Of every layer: FP16 forward weights [cout][kp] and flipped-transposed backward
    // weights [cin][kpb] (w'[ci][t*cout + co] = w[co][8-t][ci]) from FP32 master
    // [cout][9][cin], both rows padded with zeros (kp, kpb: multiples of 32)
    struct PackLayer
    {
        const float* master;
        _Float16 *wf, *wb;
        int32_t cin, cout, kp, kpb;
    };
    hipError_t launch_pack_weights(const PackLayer* layers, int count, hipStream_t s);
    // x (FP16) = f, `count` values
    hipError_t launch_to_half(const float* f, _Float16* x, int64_t count, hipStream_t s);
} // namespace isaac_hip
