// Learned occlusion pass: U-Net kernels on gfx950 (forward, backward, Adam).
//
// Convolutions are implicit GEMMs on the matrix cores (v_mfma_f32_16x16x32_f16, below);
// the weight gradients are in aonet_grad.hip.
#include "aonet.hpp"

#include <cfloat>

namespace isaac_hip
{
    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
    typedef float f4 __attribute__((ext_vector_type(4)));

    // ------------------------------------------------------------------ convolution
    // Forward layers (and, with GRAD, their backward data) run on v_mfma_f32_16x16x32_f16 (gfx950): lane l supplies
    //   A row l % 16 (output channel), k = 8*(l / 16) .. +7
    //   B col l % 16 (pixel),          k = 8*(l / 16) .. +7
    // and receives D rows 4*(l / 16) .. +3 of column l % 16.  Cin is a multiple of 8,
    // so a lane's eight k are eight consecutive channels of one tap: one 16-byte load
    // each.  Layer shapes are template parameters, so the tap / channel of every
    // K-chunk is a compile-time expression of the lane's group.
    typedef _Float16 h8 __attribute__((ext_vector_type(8)));

    __device__ inline f4 mfma32(h8 a, h8 b, f4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }

    // LDS pixel stride (halves) of a patch with CIN channels: an odd number of
    // 16-byte units, so 16 consecutive pixels of one 16-byte read hit 16 different
    // bank groups
    template<int CIN>
    constexpr int patch_stride()
    {
        return ((CIN / 8) % 2) ? CIN : CIN + 8;
    }

    // Patch staging in two halves, global loads into registers and LDS stores, so
    // a persistent workgroup loads tile t+1 while it computes tile t.  A thread
    // owns one 16-byte channel unit of one patch column (of RU = 66*CIN/8 per row)
    // and walks rows; when a row has fewer than 256 units, G = 256/RU thread groups
    // split the rows.
    template<int CIN, int CA, int PROWS>
    struct PatchStager
    {
        static constexpr int CS = CIN - CA, U = CIN / 8, PS = patch_stride<CIN>(), RU = 66 * U;
        static constexpr int G = RU >= 256 ? 1 : 256 / RU; // row groups
        static constexpr int CI = (RU + 255) / 256; // unit iterations per thread
        static constexpr int RPG = (PROWS + G - 1) / G; // rows per group
        int grp;
        int col[CI], ch[CI];
        bool uok[CI];
        h8 v[CI][RPG];

        __device__ inline void init()
        {
            const int t = int(threadIdx.x);
            grp = RU >= 256 ? 0 : t / RU;
            const int u0 = RU >= 256 ? t : t - grp * RU;
#pragma unroll
            for(int ci = 0; ci < CI; ci++)
            {
                const int u = u0 + ci * 256;
                uok[ci] = (RU >= 256) ? (u < RU) : (grp < G);
                col[ci] = u / U;
                ch[ci] = (u - col[ci] * U) * 8;
            }
        }

        __device__ inline void load(const _Float16* __restrict__ x, const _Float16* __restrict__ up, int n, int h, int w, int y0, int x0)
        {
#pragma unroll
            for(int ci = 0; ci < CI; ci++)
            {
                const int xx = x0 + col[ci] - 1;
                const bool xin = uok[ci] && xx >= 0 && xx < w;
                const bool fromUp = CA > 0 && ch[ci] < CA;
                const _Float16* base;
                size_t rs;
                if(fromUp)
                {
                    base = up + (size_t(n) * size_t(h / 2) * size_t(w / 2) + size_t(xx >= 0 ? xx / 2 : 0)) * CA + ch[ci];
                    rs = size_t(w / 2) * CA;
                }
                else
                {
                    base = x + (size_t(n) * size_t(h) * size_t(w) + size_t(xx >= 0 ? xx : 0)) * CS + (ch[ci] - CA);
                    rs = size_t(w) * CS;
                }
#pragma unroll
                for(int k = 0; k < RPG; k++)
                {
                    const int r = grp + k * G;
                    const int yy = y0 + r - 1;
                    v[ci][k] = h8{0, 0, 0, 0, 0, 0, 0, 0};
                    if(xin && r < PROWS && yy >= 0 && yy < h)
                        v[ci][k] = *reinterpret_cast<const h8*>(base + size_t(fromUp ? yy / 2 : yy) * rs);
                }
            }
        }

        __device__ inline void store(_Float16* patch) const
        {
#pragma unroll
            for(int ci = 0; ci < CI; ci++)
#pragma unroll
                for(int k = 0; k < RPG; k++)
                {
                    const int r = grp + k * G;
                    if(uok[ci] && r < PROWS)
                        *reinterpret_cast<h8*>(patch + (r * 66 + col[ci]) * PS + ch[ci]) = v[ci][k];
                }
        }
    };

    // LDS of a forward layer: the weights when all of them fit beside a one-row
    // patch in the 160 KiB of a CU (one row of KP + 8 halves per output channel: an
    // odd number of 16-byte units, so the 16 rows of a fragment read hit 16 bank
    // groups), then the (ROWS + 2) x 66-pixel input patch
    template<int CIN, int COUT>
    struct FwdLds
    {
        static constexpr int KP = (9 * CIN + 31) / 32 * 32;
        static constexpr int WS = KP + 8;
        static constexpr size_t patch(int rows)
        {
            return size_t((rows + 2) * 66) * patch_stride<CIN>() * sizeof(_Float16);
        }
        static constexpr size_t weights = size_t(COUT) * WS * sizeof(_Float16);
        static constexpr bool WLDS = weights + patch(1) <= size_t(160) * 1024;
        static constexpr size_t bytes(int rows)
        {
            return patch(rows) + (WLDS ? weights : 0);
        }
    };

    // Persistent forward layer: workgroup b computes tiles b, b + grid, ... of ROWS
    // rows x 64 pixels.  The four waves split the 16-channel output blocks first
    // (COUT 64: one block per wave; COUT 32: two blocks x two 32-pixel halves;
    // COUT 16: four 16-pixel columns): a wave owns one block in NPC 16-pixel columns
    // x ROWS rows, so each weight fragment feeds NPC * ROWS MFMAs.  Weights come from
    // LDS (loaded once per workgroup) or, when they do not fit, from global memory
    // PD chunks ahead of the MFMAs.
    // GRAD: y is FP32 without bias and ReLU, and workgroups with blockIdx.y = s compute the
    // 16-channel blocks s * COUT .. of a.couts output channels.
    template<int CIN, int COUT, int CA, int ROWS, bool GRAD = false>
    __global__ __launch_bounds__(256) void conv_fwd_kernel(const ConvArgs a, int tilesX, int tilesY, int numTiles)
    {
        using L = FwdLds<CIN, COUT>;
        constexpr int K = 9 * CIN, KP = L::KP, NCH = KP / 32, NCB = COUT / 16;
        constexpr int PS = patch_stride<CIN>();
        constexpr int WCB = NCB < 4 ? NCB : 4; // waves along output-channel blocks
        constexpr int NPC = WCB; // 16-pixel columns per wave
        static_assert(NCB == WCB, "one output-channel block per wave");
        constexpr bool WLDS = L::WLDS;
        constexpr int PD = WLDS ? 1 : (NCH < 8 ? NCH : 8);
        extern __shared__ _Float16 lds[];
        _Float16* wl = lds;
        _Float16* patch = lds + (WLDS ? COUT * L::WS : 0);
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int cb = wave % WCB, pc0 = (wave / WCB) * NPC;
        const int g = lane >> 4;
        const int tpi = tilesX * tilesY;
        auto coords = [&](int t, int& n, int& y0, int& x0) {
            n = t / tpi;
            const int r = t - n * tpi;
            const int by = r / tilesX;
            y0 = by * ROWS;
            x0 = (r - by * tilesX) * 64;
        };
        PatchStager<CIN, CA, ROWS + 2> st;
        st.init();
        const _Float16* wsrc = GRAD ? a.w + size_t(blockIdx.y) * COUT * KP : a.w;
        int t = int(blockIdx.x), n, y0, x0;
        coords(t, n, y0, x0);
        if constexpr(WLDS)
        {
            // all weights into LDS once (requested together with the first patch)
            constexpr int WU = COUT * KP / 8, WIT = (WU + 255) / 256;
            h8 wv[WIT];
#pragma unroll
            for(int it = 0; it < WIT; it++)
            {
                const int u = int(threadIdx.x) + it * 256;
                if(WU % 256 == 0 || u < WU)
                    wv[it] = *reinterpret_cast<const h8*>(wsrc + size_t(u) * 8);
            }
            st.load(a.x, a.up, n, a.h, a.w_, y0, x0);
#pragma unroll
            for(int it = 0; it < WIT; it++)
            {
                const int u = int(threadIdx.x) + it * 256;
                if(WU % 256 == 0 || u < WU)
                {
                    const int row = u / (KP / 8), k = (u - row * (KP / 8)) * 8;
                    *reinterpret_cast<h8*>(wl + row * L::WS + k) = wv[it];
                }
            }
        }
        else
            st.load(a.x, a.up, n, a.h, a.w_, y0, x0);
        const _Float16* wrow = wsrc + size_t(cb * 16 + (lane & 15)) * KP + 8 * g;
        _Float16* y = reinterpret_cast<_Float16*>(a.y);
        const int co = cb * 16 + 4 * g;
        float bias[4];
#pragma unroll
        for(int e = 0; e < 4; e++)
            bias[e] = GRAD ? 0.0f : a.bias[co + e];
        for(; t < numTiles; t += int(gridDim.x))
        {
            st.store(patch);
            __syncthreads();
            const int cn = n, cy0 = y0, cx0 = x0;
            if(t + int(gridDim.x) < numTiles)
            {
                coords(t + int(gridDim.x), n, y0, x0);
                st.load(a.x, a.up, n, a.h, a.w_, y0, x0);
            }
            h8 wq[PD];
            if constexpr(!WLDS)
            {
#pragma unroll
                for(int p = 0; p < PD; p++)
                    wq[p] = *reinterpret_cast<const h8*>(wrow + 32 * p);
            }
            f4 acc[ROWS][NPC];
#pragma unroll
            for(int r = 0; r < ROWS; r++)
#pragma unroll
                for(int q = 0; q < NPC; q++)
                    acc[r][q] = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for(int j = 0; j < NCH; j++)
            {
                h8 wa;
                if constexpr(WLDS)
                    wa = *reinterpret_cast<const h8*>(wl + (cb * 16 + (lane & 15)) * L::WS + 32 * j + 8 * g);
                else
                {
                    wa = wq[j % PD];
                    if(j + PD < NCH)
                        wq[j % PD] = *reinterpret_cast<const h8*>(wrow + 32 * (j + PD));
                }
                const int k0 = 32 * j + 8 * g;
                const int tap = k0 / CIN, ci = k0 - tap * CIN;
                const bool valid = k0 < K;
                const int ky = valid ? tap / 3 : 0, kx = valid ? tap - 3 * (tap / 3) : 0;
                const _Float16* pb = patch + (ky * 66 + pc0 * 16 + (lane & 15) + kx) * PS + ci;
#pragma unroll
                for(int r = 0; r < ROWS; r++)
#pragma unroll
                    for(int q = 0; q < NPC; q++)
                    {
                        h8 b = {0, 0, 0, 0, 0, 0, 0, 0};
                        if(valid)
                            b = *reinterpret_cast<const h8*>(pb + (r * 66 + q * 16) * PS);
                        acc[r][q] = mfma32(wa, b, acc[r][q]);
                    }
            }
            // epilogue per 16-pixel column q: bias + ReLU rounded to FP16 (the
            // activation), then optionally its 2x2 average pool (rows r-1, r of this
            // wave; x and x+1 in lanes l, l^1) and the 1x1 head (COUT 16: channels of
            // lane groups 1..3 gathered into group 0)
#pragma unroll
            for(int q = 0; q < NPC; q++)
            {
                const int x = cx0 + (pc0 + q) * 16 + (lane & 15);
                const bool xin = x < a.w_;
                h4 prev;
#pragma unroll
                for(int r = 0; r < ROWS; r++)
                {
                    const int yy = cy0 + r;
                    const bool in = xin && yy < a.h;
                    const size_t p = (size_t(cn) * a.h + yy) * a.w_ + x;
                    if constexpr(GRAD)
                    {
                        if(in)
                            *reinterpret_cast<f4*>(reinterpret_cast<float*>(a.y) + p * (size_t(gridDim.y) * COUT)
                                                   + size_t(blockIdx.y) * COUT + co) = acc[r][q];
                        continue;
                    }
                    h4 o;
#pragma unroll
                    for(int e = 0; e < 4; e++)
                    {
                        const float v = acc[r][q][e] + bias[e];
                        o[e] = _Float16(v > 0.0f ? v : 0.0f);
                    }
                    if(in && y)
                        *reinterpret_cast<h4*>(y + p * COUT + co) = o;
                    if((ROWS % 2) == 0 && a.pool && (r & 1))
                    {
                        const size_t p2 = (size_t(cn) * (a.h / 2) + yy / 2) * (a.w_ / 2) + x / 2;
                        h4 m;
#pragma unroll
                        for(int e = 0; e < 4; e++)
                        {
                            const float v00 = float(prev[e]), v10 = float(o[e]);
                            const float v01 = __shfl_xor(v00, 1), v11 = __shfl_xor(v10, 1);
                            m[e] = _Float16(((v00 + v01) + (v10 + v11)) * 0.25f);
                        }
                        if(in && (lane & 1) == 0)
                            *reinterpret_cast<h4*>(a.pool + p2 * COUT + co) = m;
                    }
                    if constexpr(COUT == 16)
                    {
                        if(a.head)
                        {
                            // channels 4g'..4g'+3 of this pixel from lane l + 16 g'
                            typedef uint32_t u2 __attribute__((ext_vector_type(2)));
                            const u2 bits = __builtin_bit_cast(u2, o);
                            h4 chv[4];
                            chv[0] = o;
#pragma unroll
                            for(int gg = 1; gg < 4; gg++)
                            {
                                u2 tt;
                                tt.x = __shfl_down(bits.x, 16 * gg);
                                tt.y = __shfl_down(bits.y, 16 * gg);
                                chv[gg] = __builtin_bit_cast(h4, tt);
                            }
                            if(g == 0 && x < a.imgW && yy < a.imgH)
                            {
                                float sum = a.headW[16];
#pragma unroll
                                for(int c4 = 0; c4 < 4; c4++)
#pragma unroll
                                    for(int e = 0; e < 4; e++)
                                        sum += float(chv[c4][e]) * a.headW[c4 * 4 + e];
                                a.head[(size_t(cn) * a.imgH + yy) * a.imgW + x] = sum < 0.0f ? 0.0f : (sum > 1.0f ? 1.0f : sum);
                            }
                        }
                    }
                    prev = o;
                }
            }
            __syncthreads();
        }
    }

    // compute units of the current device (cached per device index)
    static int device_cus()
    {
        static int cus[16] = {};
        int dev = 0;
        if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 16)
            return 256;
        if(cus[dev] == 0)
        {
            int v = 0;
            if(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0)
                v = 256;
            cus[dev] = v;
        }
        return cus[dev];
    }

    template<int CIN, int COUT, int CA, int ROWS, bool GRAD>
    hipError_t conv_fwd_launch(const ConvArgs& a, int slices, hipStream_t s)
    {
        const int tilesX = (a.w_ + 63) / 64, tilesY = (a.h + ROWS - 1) / ROWS;
        const int64_t numTiles = int64_t(tilesX) * tilesY * a.n;
        if(numTiles > int64_t(0x7fffffff))
            return hipErrorInvalidValue;
        const size_t lds = FwdLds<CIN, COUT>::bytes(ROWS);
        static int perCu = 0; // resident workgroups per CU (same for every gfx950 device)
        if(perCu == 0)
        {
            int v = 0;
            if(hipOccupancyMaxActiveBlocksPerMultiprocessor(&v, conv_fwd_kernel<CIN, COUT, CA, ROWS, GRAD>, 256, lds) != hipSuccess || v <= 0)
                v = 1;
            perCu = v;
        }
        const int64_t grid = std::min<int64_t>(numTiles, (int64_t(device_cus()) * perCu + slices - 1) / slices);
        hipLaunchKernelGGL((conv_fwd_kernel<CIN, COUT, CA, ROWS, GRAD>), dim3(unsigned(grid), unsigned(slices)), dim3(256), lds, s,
                           a, tilesX, tilesY, int(numTiles));
        return hipGetLastError();
    }

    // rows per tile: the most (of 8, 4, 2, 1) whose LDS leaves room for two
    // workgroups per CU and whose tiles cover every CU twice; else the most that fit
    // with a tile per CU; else the fewest that fit (a fused pool needs an even count).
    // A wave keeps at most 8 accumulator tiles (rows x its 16-pixel columns).
    template<int CIN, int COUT, int CA, bool GRAD = false>
    hipError_t conv_fwd_rows(const ConvArgs& a, size_t max_lds, hipStream_t s, int slices = 1)
    {
        using L = FwdLds<CIN, COUT>;
        constexpr int NPC = COUT / 16 < 4 ? COUT / 16 : 4;
        constexpr auto fits = [](int rows) { return L::bytes(rows) <= size_t(160) * 1024 && rows * NPC <= 8; };
        if(a.cin != CIN || a.ca != CA || a.kp != L::KP || (a.head && COUT != 16))
            return hipErrorInvalidValue;
        const bool pool = a.pool != nullptr;
        const int64_t cus = device_cus();
        const auto tiles = [&](int rows) { return int64_t((a.w_ + 63) / 64) * ((a.h + rows - 1) / rows) * a.n; };
        const auto ok = [&](int rows, size_t lim, int64_t minTiles) {
            return L::bytes(rows) <= lim && tiles(rows) >= minTiles && (!pool || rows % 2 == 0);
        };
        for(int pass = 0; pass < 3; pass++)
        {
            const size_t lim = pass == 0 ? max_lds / 2 : max_lds;
            const int64_t minTiles = pass == 0 ? 2 * cus : (pass == 1 ? cus : 0);
            if constexpr(fits(8))
                if(pass < 2 && ok(8, lim, minTiles))
                    return conv_fwd_launch<CIN, COUT, CA, 8, GRAD>(a, slices, s);
            if constexpr(fits(4))
                if(pass < 2 && ok(4, lim, minTiles))
                    return conv_fwd_launch<CIN, COUT, CA, 4, GRAD>(a, slices, s);
            if constexpr(fits(2))
                if(ok(2, lim, minTiles) && (pass < 2 || !ok(1, lim, 0)))
                    return conv_fwd_launch<CIN, COUT, CA, 2, GRAD>(a, slices, s);
            if constexpr(fits(1))
                if(ok(1, lim, minTiles))
                    return conv_fwd_launch<CIN, COUT, CA, 1, GRAD>(a, slices, s);
        }
        return hipErrorInvalidValue;
    }

    hipError_t launch_conv_fwd(const ConvArgs& a, int cout, size_t max_lds, hipStream_t s)
    {
        if((a.ca > 0 && !a.up) || ((a.up || a.pool) && (a.h % 2 || a.w_ % 2))
           || (a.head && (!a.headW || a.imgW > a.w_ || a.imgH > a.h)))
            return hipErrorInvalidValue;
        if(a.n == 0 || a.h == 0 || a.w_ == 0)
            return hipSuccess;
        const int cin = a.cin, ca = a.ca;
        if(cin == 8 && cout == 16 && ca == 0)
            return conv_fwd_rows<8, 16, 0>(a, max_lds, s);
        if(cin == 16 && cout == 16 && ca == 0)
            return conv_fwd_rows<16, 16, 0>(a, max_lds, s);
        if(cin == 16 && cout == 32 && ca == 0)
            return conv_fwd_rows<16, 32, 0>(a, max_lds, s);
        if(cin == 32 && cout == 32 && ca == 0)
            return conv_fwd_rows<32, 32, 0>(a, max_lds, s);
        if(cin == 32 && cout == 64 && ca == 0)
            return conv_fwd_rows<32, 64, 0>(a, max_lds, s);
        if(cin == 64 && cout == 64 && ca == 0)
            return conv_fwd_rows<64, 64, 0>(a, max_lds, s);
        if(cin == 128 && cout == 64 && ca == 64)
            return conv_fwd_rows<128, 64, 64>(a, max_lds, s);
        if(cin == 96 && cout == 32 && ca == 64)
            return conv_fwd_rows<96, 32, 64>(a, max_lds, s);
        if(cin == 48 && cout == 16 && ca == 32)
            return conv_fwd_rows<48, 16, 32>(a, max_lds, s);
        return hipErrorInvalidValue;
    }

    hipError_t launch_conv_bwd(const ConvArgs& a, int cout, size_t max_lds, hipStream_t s)
    {
        if(a.up || a.pool || a.head || a.ca != 0)
            return hipErrorInvalidValue;
        if(a.n == 0 || a.h == 0 || a.w_ == 0)
            return hipSuccess;
        if(a.cin == 16 && (cout == 16 || cout == 48))
            return conv_fwd_rows<16, 16, 0, true>(a, max_lds, s, cout / 16);
        if(a.cin == 32 && cout == 16)
            return conv_fwd_rows<32, 16, 0, true>(a, max_lds, s);
        if(a.cin == 32 && (cout == 32 || cout == 96))
            return conv_fwd_rows<32, 32, 0, true>(a, max_lds, s, cout / 32);
        if(a.cin == 64 && cout == 32)
            return conv_fwd_rows<64, 32, 0, true>(a, max_lds, s);
        if(a.cin == 64 && (cout == 64 || cout == 128))
            return conv_fwd_rows<64, 64, 0, true>(a, max_lds, s, cout / 64);
        return hipErrorInvalidValue;
    }

    // ------------------------------------------------------------------ elementwise
    static unsigned grid_for(int64_t count)
    {
        int64_t b = (count + 255) / 256;
        return unsigned(b > 8192 ? 8192 : (b < 1 ? 1 : b));
    }

    __global__ __launch_bounds__(256) void to_half_kernel(const float* __restrict__ f, _Float16* __restrict__ x, int64_t count)
    {
        for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += int64_t(gridDim.x) * blockDim.x)
            x[i] = _Float16(f[i]);
    }

    hipError_t launch_to_half(const float* f, _Float16* x, int64_t count, hipStream_t s)
    {
        if(count == 0)
            return hipSuccess;
        hipLaunchKernelGGL(to_half_kernel, dim3(grid_for(count)), dim3(256), 0, s, f, x, count);
        return hipGetLastError();
    }

    // ------------------------------------------------------------------ features and head
    __global__ __launch_bounds__(256) void features_kernel(const FeatureArgs a)
    {
        const int64_t count = int64_t(a.n) * a.h * a.w;
        for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += int64_t(gridDim.x) * blockDim.x)
        {
            const int xx = int(i % a.w), yy = int((i / a.w) % a.h);
            const int item = int(i / (int64_t(a.w) * a.h));
            const int gx = xx + (a.origin ? a.origin[2 * item] : 0), gy = yy + (a.origin ? a.origin[2 * item + 1] : 0);
            float d = FLT_MAX, nx = 0.f, ny = 0.f, nz = 0.f, t = 0.f;
            const float invScale = a.invScaleItem ? a.invScaleItem[item] : a.invScale;
            if(gx >= 0 && gx < a.imgW && gy >= 0 && gy < a.imgH)
            {
                const size_t p = size_t(item) * size_t(a.imgStride) + size_t(gy) * a.imgW + gx;
                d = a.depth[p];
                nx = a.normal[3 * p + 0];
                ny = a.normal[3 * p + 1];
                nz = a.normal[3 * p + 2];
                if(a.ao)
                    t = a.ao[p];
            }
            const bool bg = !(d < 3.0e38f);
            h4 lo, hi;
            lo[0] = _Float16(bg ? 0.0f : d * invScale);
            lo[1] = _Float16(bg ? 1.0f : 0.0f);
            lo[2] = _Float16(nx);
            lo[3] = _Float16(ny);
            hi[0] = _Float16(nz);
            hi[1] = hi[2] = hi[3] = _Float16(0.0f);
            *reinterpret_cast<h4*>(a.x + i * 8) = lo;
            *reinterpret_cast<h4*>(a.x + i * 8 + 4) = hi;
            if(a.target)
                a.target[i] = t;
        }
    }

    hipError_t launch_features(const FeatureArgs& a, hipStream_t s)
    {
        const int64_t count = int64_t(a.n) * a.h * a.w;
        if(count == 0)
            return hipSuccess;
        hipLaunchKernelGGL(features_kernel, dim3(grid_for(count)), dim3(256), 0, s, a);
        return hipGetLastError();
    }

    __device__ inline float head_dot(const _Float16* d0, const float* wh, int64_t p)
    {
        const h4* v = reinterpret_cast<const h4*>(d0 + p * 16);
        float s = wh[16];
#pragma unroll
        for(int q = 0; q < 4; q++)
        {
            const h4 u = v[q];
#pragma unroll
            for(int r = 0; r < 4; r++)
                s += float(u[r]) * wh[q * 4 + r];
        }
        return s;
    }

    __global__ __launch_bounds__(256) void head_train_kernel(
        const _Float16* d0,
        const float* wh,
        const float* target,
        float* loss,
        float* gwh,
        float* dd0,
        float* out,
        int64_t npx)
    {
        float gl = 0.0f, gw[17];
        for(int c = 0; c < 17; c++)
            gw[c] = 0.0f;
        for(int64_t p = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; p < npx; p += int64_t(gridDim.x) * blockDim.x)
        {
            const float o = head_dot(d0, wh, p);
            if(out)
                out[p] = o;
            const float e = o - target[p];
            const float dout = 2.0f * e;
            gl += e * e;
            const h4* v = reinterpret_cast<const h4*>(d0 + p * 16);
            for(int q = 0; q < 4; q++)
            {
                const h4 u = v[q];
                float4 o;
                o.x = dout * wh[q * 4 + 0];
                o.y = dout * wh[q * 4 + 1];
                o.z = dout * wh[q * 4 + 2];
                o.w = dout * wh[q * 4 + 3];
                reinterpret_cast<float4*>(dd0 + p * 16)[q] = o;
                for(int r = 0; r < 4; r++)
                    gw[q * 4 + r] += dout * float(u[r]);
            }
            gw[16] += dout;
        }
        __shared__ float red[18][256];
        red[0][threadIdx.x] = gl;
        for(int c = 0; c < 17; c++)
            red[c + 1][threadIdx.x] = gw[c];
        __syncthreads();
        for(int off = 128; off > 0; off >>= 1)
        {
            if(int(threadIdx.x) < off)
                for(int c = 0; c < 18; c++)
                    red[c][threadIdx.x] += red[c][threadIdx.x + off];
            __syncthreads();
        }
        if(threadIdx.x == 0)
            atomicAdd(loss, red[0][0]);
        if(threadIdx.x >= 1 && threadIdx.x < 18)
            atomicAdd(gwh + threadIdx.x - 1, red[threadIdx.x][0]);
    }

    hipError_t launch_head_train(
        const _Float16* d0,
        const float* wh,
        const float* target,
        float* loss,
        float* gwh,
        float* dd0,
        float* out,
        int64_t npx,
        hipStream_t s)
    {
        if(npx == 0)
            return hipSuccess;
        int64_t blocks = (npx + 255) / 256;
        if(blocks > 2048)
            blocks = 2048;
        hipLaunchKernelGGL(head_train_kernel, dim3(unsigned(blocks)), dim3(256), 0, s, d0, wh, target, loss, gwh, dd0, out, npx);
        return hipGetLastError();
    }

    // ------------------------------------------------------------------ optimiser
    __global__ __launch_bounds__(256) void adam_kernel(
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
        float gscale)
    {
        for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < count; i += int64_t(gridDim.x) * blockDim.x)
        {
            const float gi = g[i] * gscale;
            const float mi = b1 * m[i] + (1.0f - b1) * gi;
            const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
            m[i] = mi;
            v[i] = vi;
            w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
        }
    }

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
        hipStream_t s)
    {
        if(count == 0)
            return hipSuccess;
        hipLaunchKernelGGL(adam_kernel, dim3(grid_for(count)), dim3(256), 0, s, w, g, m, v, count, lr, b1, b2, eps, c1, c2, gscale);
        return hipGetLastError();
    }

    // all layers in one launch (blockIdx.y): eleven launches took ten times as long
    struct PackArgs
    {
        PackLayer L[kGradMaxLayers];
    };

    __global__ __launch_bounds__(256) void pack_weights_kernel(const PackArgs a)
    {
        const PackLayer& L = a.L[blockIdx.y];
        const int K = 9 * L.cin, KB = 9 * L.cout;
        const int nf = L.cout * L.kp, nb = L.cin * L.kpb;
        for(int i = int(blockIdx.x * blockDim.x + threadIdx.x); i < nf + nb; i += int(gridDim.x * blockDim.x))
        {
            if(i < nf)
            {
                const int co = i / L.kp, k = i - co * L.kp;
                L.wf[i] = _Float16(k < K ? L.master[co * K + k] : 0.0f);
            }
            else
            {
                const int j = i - nf, ci = j / L.kpb, k = j - ci * L.kpb; // [ci][t][co]
                const int t = k / L.cout, co = k - t * L.cout;
                L.wb[j] = _Float16(k < KB ? L.master[(co * 9 + (8 - t)) * L.cin + ci] : 0.0f);
            }
        }
    }

    hipError_t launch_pack_weights(const PackLayer* layers, int count, hipStream_t s)
    {
        if(count < 1 || count > kGradMaxLayers)
            return hipErrorInvalidValue;
        PackArgs a{};
        for(int l = 0; l < count; l++)
            a.L[l] = layers[l];
        hipLaunchKernelGGL(pack_weights_kernel, dim3(128, unsigned(count)), dim3(256), 0, s, a);
        return hipGetLastError();
    }
} // namespace isaac_hip
