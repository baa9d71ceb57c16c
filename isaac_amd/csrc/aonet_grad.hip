// Weight and bias gradients of the occlusion network's 3x3 convolutions on gfx950.
//
// One kernel per layer forms the layer's dz (the gradient behind its ReLU, rounded to
// binary16) from the gradients of the layers that read its output, stores it for the
// backward-data convolution, and accumulates
//   dW[co][tap][ci] = sum over pixels p of dz[p][co] * X[p + tap][ci],   db[co] = sum dz[p][co]
// on v_mfma_f32_16x16x32_f16 with the pixels as the contracted dimension: per step, lane l
// supplies A row l % 16 (output channel) and B column l % 16 (input channel), each with the 8
// consecutive pixels 8 * (l / 16) .. +7 of a row, and receives D rows 4 * (l / 16) .. +3 of column
// l % 16.  Partial sums of a workgroup go to memory and one kernel adds them for all layers.
#include "aonet.hpp"

#include <algorithm>

namespace isaac_hip
{
    namespace
    {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        typedef _Float16 h8 __attribute__((ext_vector_type(8)));
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        typedef float f4 __attribute__((ext_vector_type(4)));

        constexpr int kGradRows = 8, kGradCols = 32; // pixels of a tile: 4 waves, two rows of 32 each
        // LDS: both operands transposed to [channel][row][pixel], so that a fragment is one 16-byte
        // read.  X has one row and column more on every side (column c at index c + 8, rows of 48
        // halves).  A channel's stride is an odd number of 16-byte units, so the 16 channels of a
        // fragment read hit 16 bank groups.
        constexpr int kXRow = 48, kXCh = (kGradRows + 2) * kXRow + 8;
        constexpr int kDCh = kGradRows * kGradCols + 8;

        struct GradArgs
        {
            GradLayer L;
            int tilesX, tilesY, numTiles;
        };

        // 8 channels (c .. c + 7) of the gradient of the layer's output at pixel (n, y, x)
        __device__ inline void load_dy(const GradLayer& L, int n, int y, int x, int c, float dy[8])
        {
            auto get = [](const float* p, float v[8])
            {
                const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
                v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
            };
            if(L.dyMode == kDyUpsampled)
            {
                // read through a nearest-neighbour upsampling: the sum of its four positions
                const float* b = L.g + ((size_t(n) * (2 * L.h) + 2 * y) * (2 * L.w) + 2 * x) * L.gStride + L.gOff + c;
                const size_t row = size_t(2 * L.w) * L.gStride;
                float v1[8], v2[8], v3[8];
                get(b, dy);
                get(b + L.gStride, v1);
                get(b + row, v2);
                get(b + row + L.gStride, v3);
#pragma unroll
                for(int e = 0; e < 8; e++)
                    dy[e] = (dy[e] + v1[e]) + (v2[e] + v3[e]);
                return;
            }
            get(L.g + ((size_t(n) * L.h + y) * L.w + x) * L.gStride + L.gOff + c, dy);
            if(L.dyMode == kDySkipAndPool)
            {
                // read by a decoder layer and, through a 2x2 average pool, by the next encoder level
                float v[8];
                get(L.gPool + ((size_t(n) * (L.h / 2) + y / 2) * (L.w / 2) + x / 2) * L.cout + c, v);
#pragma unroll
                for(int e = 0; e < 8; e++)
                    dy[e] = dy[e] + 0.25f * v[e];
            }
        }

        // COUT output channels x CT 16-channel blocks of the input per workgroup, all 9 taps: at
        // most 36 accumulator tiles per wave, so that a wave's LDS reads (COUT / 16 fragments of dz and
        // 3 CT of X per 32 pixels) feed up to 36 MFMAs.  The x-shifted fragments of X are funnel
        // shifts of the aligned one and its two neighbouring words.
        // Bound by the staging of a workgroup's few tiles (load, transpose, compute in turn), not by the
        // matrix cores.  Measured on MI355X for 16 crops of 128x128: all layers' dz, dW and db 340 us
        // against 1670 us in separate ReLU, bias and weight-gradient kernels whose MFMA operands
        // came from LDS as single halves (before the waves' sums below were batched); the whole training
        // step 2.73 -> 1.08 ms.
        template<int COUT, int CT>
        __global__ __launch_bounds__(256) void conv_grad_kernel(const GradArgs a)
        {
            constexpr int NA = COUT / 16, NT = NA * CT * 9, DG = COUT / 8;
            extern __shared__ _Float16 lds[];
            _Float16* xt = lds;
            _Float16* dzt = lds + CT * 16 * kXCh;
            const GradLayer& L = a.L;
            const int tid = int(threadIdx.x), lane = tid & 63, wave = tid >> 6;
            const int l16 = lane & 15, g = lane >> 4;
            const int ci0 = int(blockIdx.y) * CT * 16;
            f4 acc[NA][CT][9];
#pragma unroll
            for(int i = 0; i < NA; i++)
#pragma unroll
                for(int c = 0; c < CT; c++)
#pragma unroll
                    for(int t = 0; t < 9; t++)
                        acc[i][c][t] = f4{0.f, 0.f, 0.f, 0.f};
            const int dgrp = tid % DG; // (256 is a multiple of DG: a thread keeps its channels)
            float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            const int tpi = a.tilesX * a.tilesY;
            for(int tile = int(blockIdx.x); tile < a.numTiles; tile += int(gridDim.x))
            {
                const int n = tile / tpi, rest = tile - n * tpi, ty = rest / a.tilesX;
                const int y0 = ty * kGradRows, x0 = (rest - ty * a.tilesX) * kGradCols;
                __syncthreads();
                // input patch: units of 4 pixels x 8 channels, transposed in registers
                for(int u = tid; u < CT * 2 * (kGradRows + 2) * 10; u += 256)
                {
                    const int g8 = u % (2 * CT), q = u / (2 * CT), quad = q % 10, r = q / 10;
                    const int c = ci0 + g8 * 8, yy = y0 + r - 1, xb = x0 + quad * 4 - 4;
                    h8 v[4];
#pragma unroll
                    for(int j = 0; j < 4; j++)
                    {
                        const int xx = xb + j;
                        v[j] = h8{0, 0, 0, 0, 0, 0, 0, 0};
                        if(c < L.cin && yy >= 0 && yy < L.h && xx >= 0 && xx < L.w)
                            v[j] = c < L.ca
                                ? *reinterpret_cast<const h8*>(L.up + ((size_t(n) * (L.h / 2) + yy / 2) * (L.w / 2) + xx / 2) * L.ca + c)
                                : *reinterpret_cast<const h8*>(L.x + ((size_t(n) * L.h + yy) * L.w + xx) * (L.cin - L.ca) + (c - L.ca));
                    }
#pragma unroll
                    for(int e = 0; e < 8; e++)
                        *reinterpret_cast<h4*>(xt + (g8 * 8 + e) * kXCh + r * kXRow + quad * 4 + 4) = h4{v[0][e], v[1][e], v[2][e], v[3][e]};
                }
                // dz, the same way
                for(int u = tid; u < DG * kGradRows * 8; u += 256)
                {
                    const int q = u / DG, quad = q % 8, r = q / 8;
                    const int y = y0 + r, c = dgrp * 8;
                    h8 v[4];
#pragma unroll
                    for(int j = 0; j < 4; j++)
                    {
                        const int x = x0 + quad * 4 + j;
                        v[j] = h8{0, 0, 0, 0, 0, 0, 0, 0};
                        if(y < L.h && x < L.w)
                        {
                            const size_t p = ((size_t(n) * L.h + y) * L.w + x) * COUT + c;
                            const h8 act = *reinterpret_cast<const h8*>(L.act + p);
                            float dy[8];
                            load_dy(L, n, y, x, c, dy);
#pragma unroll
                            for(int e = 0; e < 8; e++)
                            {
                                v[j][e] = _Float16(float(act[e]) > 0.0f ? dy[e] : 0.0f);
                                bsum[e] += float(v[j][e]);
                            }
                            if(blockIdx.y == 0)
                                *reinterpret_cast<h8*>(L.dz + p) = v[j];
                        }
                    }
#pragma unroll
                    for(int e = 0; e < 8; e++)
                        *reinterpret_cast<h4*>(dzt + (c + e) * kDCh + r * kGradCols + quad * 4) = h4{v[0][e], v[1][e], v[2][e], v[3][e]};
                }
                __syncthreads();
#pragma unroll 1
                for(int rr = 0; rr < kGradRows / 4; rr++)
                {
                    const int r = wave * (kGradRows / 4) + rr;
                    if(y0 + r >= L.h)
                        break;
                    h8 A[NA];
#pragma unroll
                    for(int i = 0; i < NA; i++)
                        A[i] = *reinterpret_cast<const h8*>(dzt + (i * 16 + l16) * kDCh + r * kGradCols + 8 * g);
#pragma unroll
                    for(int c = 0; c < CT; c++)
#pragma unroll
                        for(int ky = 0; ky < 3; ky++)
                        {
                            const _Float16* xp = xt + (c * 16 + l16) * kXCh + (r + ky) * kXRow + 8 + 8 * g;
                            const u4 m = *reinterpret_cast<const u4*>(xp);
                            const uint32_t lo = *reinterpret_cast<const uint32_t*>(xp - 2), hi = *reinterpret_cast<const uint32_t*>(xp + 8);
                            const uint32_t s0 = __builtin_amdgcn_alignbit(m.x, lo, 16), s1 = __builtin_amdgcn_alignbit(m.y, m.x, 16);
                            const uint32_t s2 = __builtin_amdgcn_alignbit(m.z, m.y, 16), s3 = __builtin_amdgcn_alignbit(m.w, m.z, 16);
                            const uint32_t s4 = __builtin_amdgcn_alignbit(hi, m.w, 16);
                            const h8 B0 = __builtin_bit_cast(h8, (u4{s0, s1, s2, s3})); // pixels p - 1
                            const h8 B1 = __builtin_bit_cast(h8, m);
                            const h8 B2 = __builtin_bit_cast(h8, (u4{s1, s2, s3, s4})); // pixels p + 1
#pragma unroll
                            for(int i = 0; i < NA; i++)
                            {
                                acc[i][c][ky * 3 + 0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i], B0, acc[i][c][ky * 3 + 0], 0, 0, 0);
                                acc[i][c][ky * 3 + 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i], B1, acc[i][c][ky * 3 + 1], 0, 0, 0);
                                acc[i][c][ky * 3 + 2] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[i], B2, acc[i][c][ky * 3 + 2], 0, 0, 0);
                            }
                        }
                }
            }
            // the four waves' sums, one wave after the other; the reads of 36 elements are in flight
            // together (a read, its wait and the write behind it one by one: loss and gradient of 8 images of
            // 128x128 768 us, 688 us this way)
            float* red = reinterpret_cast<float*>(lds);
            __syncthreads();
            if(wave == 0)
            {
#pragma unroll
                for(int i = 0; i < NA; i++)
#pragma unroll
                    for(int c = 0; c < CT; c++)
#pragma unroll
                        for(int t = 0; t < 9; t++)
#pragma unroll
                            for(int r = 0; r < 4; r++)
                                red[((i * CT + c) * 9 + t) * 256 + r * 64 + lane] = acc[i][c][t][r];
            }
#pragma unroll 1
            for(int w = 1; w < 4; w++)
            {
                __syncthreads();
                if(wave == w)
                {
#pragma unroll
                    for(int i = 0; i < NA; i++)
#pragma unroll
                        for(int c = 0; c < CT; c++)
                        {
                            float* d = red + (i * CT + c) * 9 * 256 + lane;
                            float v[36];
#pragma unroll
                            for(int k = 0; k < 36; k++)
                                v[k] = d[k * 64];
#pragma unroll
                            for(int k = 0; k < 36; k++)
                                d[k * 64] = v[k] + acc[i][c][k >> 2][k & 3];
                        }
                }
            }
            __syncthreads();
            float* out = L.partial + (size_t(blockIdx.y) * gridDim.x + blockIdx.x) * size_t(NT * 256);
            for(int i = tid; i < NT * 256; i += 256)
                out[i] = red[i];
            if(blockIdx.y != 0)
                return;
            __syncthreads();
#pragma unroll
            for(int e = 0; e < 8; e++)
                red[e * 256 + tid] = bsum[e];
            __syncthreads();
            if(tid < COUT)
            {
                float s = 0.0f;
                for(int j = tid / 8; j < 256; j += DG)
                    s += red[(tid & 7) * 256 + j];
                L.partialBias[size_t(blockIdx.x) * COUT + tid] = s;
            }
        }

        // 16-channel input blocks per workgroup of a layer
        constexpr int grad_ct(int cin, int cout)
        {
            return cout == 16 ? (cin == 48 ? 3 : 1) : (cout == 32 ? (cin == 16 ? 1 : 2) : 1);
        }

        template<int COUT, int CT>
        hipError_t grad_launch(const GradArgs& a, const GradShape& s, hipStream_t st)
        {
            constexpr size_t operands = (size_t(CT) * 16 * kXCh + size_t(COUT) * kDCh) * sizeof(_Float16);
            constexpr size_t sums = size_t(COUT / 16) * CT * 9 * 256 * sizeof(float);
            constexpr size_t lds = operands > sums ? operands : sums;
            static_assert(lds <= 64 * 1024 && sums >= 8 * 256 * sizeof(float), "LDS of a gradient workgroup");
            hipLaunchKernelGGL((conv_grad_kernel<COUT, CT>), dim3(unsigned(s.splits), unsigned(s.groups)), dim3(256), lds, st, a);
            return hipGetLastError();
        }

        struct SumArgs
        {
            GradLayer L[kGradMaxLayers];
            GradShape s[kGradMaxLayers];
            int first[kGradMaxLayers + 1]; // first block of each layer
            int layers;
        };

        // One workgroup per 64 elements of an accumulator tile (and one per layer for the biases): the
        // four waves each add a quarter of the splits.
        __global__ __launch_bounds__(256) void grad_sum_kernel(const SumArgs a)
        {
            int l = 0;
            while(l + 1 < a.layers && int(blockIdx.x) >= a.first[l + 1])
                l++;
            const GradLayer& L = a.L[l];
            const GradShape& s = a.s[l];
            const int b = int(blockIdx.x) - a.first[l], lane = int(threadIdx.x) & 63, wave = int(threadIdx.x) >> 6;
            const int ct = s.ct, nt = (L.cout / 16) * ct * 9;
            const int s0 = s.splits * wave / 4, s1 = s.splits * (wave + 1) / 4;
            const bool bias = b == s.groups * nt * 4;
            float v = 0.0f;
            const int group = bias ? 0 : b / (nt * 4), e = bias ? 0 : b - group * (nt * 4);
            if(!bias)
            {
                const float* p = L.partial + size_t(group) * s.splits * size_t(nt * 256) + size_t(e) * 64 + lane;
#pragma unroll 8
                for(int k = s0; k < s1; k++)
                    v += p[size_t(k) * size_t(nt * 256)];
            }
            else if(lane < L.cout)
                for(int k = s0; k < s1; k++)
                    v += L.partialBias[size_t(k) * L.cout + lane];
            __shared__ float red[256];
            red[threadIdx.x] = v;
            __syncthreads();
            if(wave != 0)
                return;
            v = (red[lane] + red[64 + lane]) + (red[128 + lane] + red[192 + lane]);
            if(bias)
            {
                if(lane < L.cout)
                    L.db[lane] = v;
                return;
            }
            const int t = e >> 2, r = e & 3; // accumulator tile and its row within the lane's four
            const int tap = t % 9, c = (t / 9) % ct, i = t / (9 * ct);
            const int co = i * 16 + 4 * (lane >> 4) + r, ci = (group * ct + c) * 16 + (lane & 15);
            if(ci < L.cin)
                L.dw[(size_t(co) * 9 + tap) * L.cin + ci] = v;
        }
    } // namespace

    GradShape grad_shape(int cin, int cout, int n, int h, int w)
    {
        GradShape s{};
        s.ct = grad_ct(cin, cout);
        s.groups = (cin + 16 * s.ct - 1) / (16 * s.ct);
        const int64_t tiles = int64_t((w + kGradCols - 1) / kGradCols) * ((h + kGradRows - 1) / kGradRows) * n;
        // about one workgroup per CU, two where the partial sums are small
        const int64_t target = (cout == 16 ? 512 : 256) / s.groups;
        s.splits = int(std::max<int64_t>(1, std::min(tiles, target)));
        s.partial = size_t(s.groups) * s.splits * size_t(cout / 16) * s.ct * 9 * 256;
        return s;
    }

    hipError_t launch_conv_grad(const GradLayer& L, hipStream_t s)
    {
        if(L.cin % 8 || L.ca % 8 || L.ca > L.cin || (L.ca > 0 && !L.up) || (L.up && (L.h % 2 || L.w % 2))
           || (L.dyMode == kDySkipAndPool && (L.h % 2 || L.w % 2 || !L.gPool)) || L.gStride % 4 || L.gOff % 4)
            return hipErrorInvalidValue;
        if(L.n <= 0 || L.h <= 0 || L.w <= 0)
            return hipErrorInvalidValue;
        GradArgs a{};
        a.L = L;
        a.tilesX = (L.w + kGradCols - 1) / kGradCols;
        a.tilesY = (L.h + kGradRows - 1) / kGradRows;
        const int64_t tiles = int64_t(a.tilesX) * a.tilesY * L.n;
        if(tiles > 0x3fffffff)
            return hipErrorInvalidValue;
        a.numTiles = int(tiles);
        const GradShape sh = grad_shape(L.cin, L.cout, L.n, L.h, L.w);
        if(L.cout == 16)
            return sh.ct == 3 ? grad_launch<16, 3>(a, sh, s) : grad_launch<16, 1>(a, sh, s);
        if(L.cout == 32)
            return sh.ct == 2 ? grad_launch<32, 2>(a, sh, s) : grad_launch<32, 1>(a, sh, s);
        if(L.cout == 64)
            return grad_launch<64, 1>(a, sh, s);
        return hipErrorInvalidValue;
    }

    hipError_t launch_grad_sum(const GradLayer* layers, int count, hipStream_t s)
    {
        if(count < 1 || count > kGradMaxLayers)
            return hipErrorInvalidValue;
        SumArgs a{};
        a.layers = count;
        for(int l = 0; l < count; l++)
        {
            a.L[l] = layers[l];
            a.s[l] = grad_shape(layers[l].cin, layers[l].cout, layers[l].n, layers[l].h, layers[l].w);
            a.first[l + 1] = a.first[l] + a.s[l].groups * (layers[l].cout / 16) * a.s[l].ct * 9 * 4 + 1;
        }
        hipLaunchKernelGGL(grad_sum_kernel, dim3(unsigned(a.first[count])), dim3(256), 0, s, a);
        return hipGetLastError();
    }
} // namespace isaac_hip
