// gfx950 kernels of the per-rank render path (the combined form's march: march.hip).
//
//   classify_kernel        MergeToCombinedTextureKernel  lib/isaac/isaac_common_kernel.hpp:553-615,690-758
//   ssao_tiled_kernel      SSAOKernel (live 7x7 part)     lib/isaac/isaac_ssao_kernel.hpp:161-182
//                          (with the shading of its pixels fused in render modes 0, 1, 3)
//   shade_kernel           ShadingKernel + the volume pass's final blend
//                          lib/isaac/isaac_common_kernel.hpp:220-320, lib/isaac/isaac_volume_kernel.hpp:83-86
//
// The fusions keep the reference's quantisation points: every stage that the
// reference stores as RGBA8 in the G-buffer is rounded to RGBA8 in registers
// at the same point, so the fused kernels produce the stage sequence's bytes.
//
// Launch shape: 256-thread workgroups = four wave64s, each wave an 8x8 pixel
// tile (16x16 pixels per workgroup), so the 64 rays of a wave sample
// neighbouring voxels; the march deals its tiles to the 8 XCDs (each with its
// own L2) in super-tiles or bands (march_tile), and can run one-wave workgroups.
#include "render_device.hpp"

namespace isaac_hip
{
#define DITHER_TABLE(type, name, n) __constant__ type name[n]
#include "dither_tables.inc"
#undef DITHER_TABLE

    // ------------------------------------------------------------------ functor chain
    // pow stays out of line: inlined, its ~70 instructions per component and
    // functor slot made up most of the code of the marches that evaluate the
    // chain per sample (rarely used, and the call is only taken for it).
    __device__ __noinline__ float chain_pow(float a, float b)
    {
        return powf(a, b);
    }

    // f2(f1(f0(v,p0),p1),p2).x with the feature dimension propagating
    // (lib/isaac/isaac_functor_chain.hpp:96-108, lib/isaac/isaac_functors.hpp:42-183).
    __device__ inline float apply_chain(const ChainDesc& c, float v0, float v1, float v2, float v3, int n)
    {
        float v[4] = {v0, v1, v2, v3};
#pragma unroll
        for(int k = 0; k < kMaxFunctors; k++)
        {
            const int op = c.op[k];
            if(op == OP_ADD)
            {
#pragma unroll
                for(int i = 0; i < 4; i++)
                    if(i < n)
                        v[i] = v[i] + c.p[k][i];
            }
            else if(op == OP_MUL)
            {
#pragma unroll
                for(int i = 0; i < 4; i++)
                    if(i < n)
                        v[i] = v[i] * c.p[k][i];
            }
            else if(op == OP_LENGTH)
            {
                float d;
                if(n == 1)
                    d = v[0] * v[0];
                else if(n == 2)
                    d = v[0] * v[0] + v[1] * v[1];
                else if(n == 3)
                    d = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
                else
                    d = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
                v[0] = sqrtf(d);
                n = 1;
            }
            else if(op == OP_POW)
            {
#pragma unroll
                for(int i = 0; i < 4; i++)
                    if(i < n)
                        v[i] = chain_pow(v[i], c.p[k][i]);
            }
            else if(op == OP_SUM)
            {
                float s = 0.0f;
#pragma unroll
                for(int i = 0; i < 4; i++)
                    if(i < n)
                        s = s + v[i];
                v[0] = s;
                n = 1;
            }
        }
        return v[0];
    }

    // x / d for a divisor fixed per launch, with r = RN(1/d) computed once on the
    // host: x*r plus one fma residual correction (Markstein's correction), three
    // instructions instead of the correctly rounded division sequence.  Equal to the
    // IEEE quotient for finite operands away from overflow and underflow
    // (tests/cpp/divq_check.c: 0 of 2e8 seeded quotients differ, a quarter of them
    // next to rounding boundaries; for d = 255 every x in [0, 256],
    // tests/cpp/div255_check.c).
    __device__ inline float div_by(float x, float d, float r)
    {
        const float q0 = x * r;
        const float e = __builtin_fmaf(-q0, d, x);
        return __builtin_fmaf(e, r, q0);
    }

    __device__ inline int tf_index(float v, int T)
    {
        return tf_index_of(v * float(T), T);
    }

    // ------------------------------------------------------------------ classification
    __device__ inline uint32_t dither_b4(int mode, int x, int y, int z, float r, float g, float b, float a)
    {
        if(mode == 0)
        {
            return unorm8(r) | (unorm8(g) << 8) | (unorm8(b) << 16) | (unorm8(a) << 24);
        }
        // threshold of the mode's mask (applyDither3D, lib/isaac/isaac_dither_kernel.hpp:20-323):
        // 1 ordered 4^3, 2 blue noise 4^3, 3 blue noise 8^3, any other mode blue noise 16^3
        float d;
        if(mode == 1)
            d = float(kDitherOrdered4[(x & 3) + (y & 3) * 4 + (z & 3) * 16]) / 64.0f;
        else if(mode == 2)
            d = float(kDitherBlue4[(x & 3) + (y & 3) * 4 + (z & 3) * 16]) / 64.0f;
        else if(mode == 3)
            d = float(kDitherBlue8[(x & 7) + (y & 7) * 8 + (z & 7) * 64]) / 512.0f;
        else
            d = float(kDitherBlue16[(x & 15) + (y & 15) * 16 + (z & 15) * 256]) / 4096.0f;
        auto q = [d](float v) -> uint32_t
        {
            float s = v * 255.0f;
            int i = (int) s;
            i += ((s - floorf(s)) > d) ? 1 : 0;
            return (uint32_t) iclamp(i, 0, 255);
        };
        return q(r) | (q(g) << 8) | (q(b) << 16) | (q(a) << 24);
    }

    // Marks the iso cells whose steps may read one of the voxels x0..x1 of row (y, z), which
    // holds an iso alpha byte >= 128 (ClassifyParams::isoCells).  Cell c serves the base texels
    // 8c..8c+7 with their + neighbours, and one voxel more on each side for the rounding of the
    // march's cell exits: voxels 8c-1..8c+9.  Every writer stores the same value, so plain
    // stores do; the value is the update's number, so nothing is cleared between updates.
    __device__ inline void mark_iso_cells(const ClassifyParams& P, int x0, int x1, int y, int z)
    {
        const int cx0 = max(0, (x0 - 2) >> kIsoCellShift), cx1 = min(P.ncx - 1, (x1 + 1) >> kIsoCellShift);
        const int cy0 = max(0, (y - 2) >> kIsoCellShift), cy1 = min(P.ncy - 1, (y + 1) >> kIsoCellShift);
        const int cz0 = max(0, (z - 2) >> kIsoCellShift), cz1 = min(P.ncz - 1, (z + 1) >> kIsoCellShift);
        for(int cz = cz0; cz <= cz1; cz++)
            for(int cy = cy0; cy <= cy1; cy++)
                for(int cx = cx0; cx <= cx1; cx++)
                    P.isoCells[(size_t(cz) * size_t(P.ncy) + size_t(cy)) * size_t(P.ncx) + size_t(cx)] = P.isoEpoch;
    }

    // One workgroup stages up to nLut transfer functions (T float4 each) in LDS
    // and then walks voxels with a grid-stride loop (x fastest, coalesced
    // source reads and texel writes).
    __global__ __launch_bounds__(256) void classify_kernel(const ClassifyParams P)
    {
        extern __shared__ float4 lds_lut[];
        const int T = P.T;
        for(int i = threadIdx.x; i < P.nLut * T; i += blockDim.x)
            lds_lut[i] = P.luts[i];
        __syncthreads();
        const int64_t stride = int64_t(gridDim.x) * blockDim.x;
        for(int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < P.nvox; idx += stride)
        {
            const uint32_t u = (uint32_t) idx;
            const uint32_t zq = fastdiv(u, P.divXY_mul, P.divXY_shift);
            const uint32_t rem = u - zq * uint32_t(P.X * P.Y);
            const uint32_t yq = fastdiv(rem, P.divX_mul, P.divX_shift);
            const int x = int(rem - yq * uint32_t(P.X)), y = int(yq), z = int(zq);
            float vr = 0.f, vg = 0.f, vb = 0.f, va = 0.f;
            float ir = 0.f, ig = 0.f, ib = 0.f, ia = 0.f;
            for(int s = 0; s < P.nsrc; s++)
            {
                const ClassifySource& S = P.src[s];
                if(!S.active)
                    continue;
                const float* e = S.data + (int64_t(x) * S.stride[0] + int64_t(y) * S.stride[1] + int64_t(z) * S.stride[2]) * S.dim;
                float c0 = e[0];
                float c1 = S.dim > 1 ? e[1] : 0.f;
                float c2 = S.dim > 2 ? e[2] : 0.f;
                float c3 = S.dim > 3 ? e[3] : 0.f;
                const float tv = apply_chain(S.chain, c0, c1, c2, c3, S.dim);
                const int li = tf_index(tv, T);
                const float4 col = (S.lutSlot < P.nLut) ? lds_lut[S.lutSlot * T + li] : P.luts[S.lutSlot * T + li];
                // field sources: alpha blended with the advection texture
                // (MergeAdvectionToCombinedTextureIterator, lib/isaac/isaac_common_kernel.hpp:655-656)
                float ca = col.w;
                if(S.adv)
                    ca = ca * div_by(float(S.adv[idx]), 255.0f, 1.0f / 255.0f);
                if(S.weight > 0.0f)
                {
                    float a = ca * S.weight;
                    vr = vr + col.x * a;
                    vg = vg + col.y * a;
                    vb = vb + col.z * a;
                    va = va + a;
                }
                if(S.iso > 0.0f)
                {
                    float a = div_by(ca, S.iso, S.invIso) * 0.5f;
                    if(ia < a)
                    {
                        ir = col.x;
                        ig = col.y;
                        ib = col.z;
                        ia = a;
                    }
                }
            }
            if(P.totalWeight != 0.0f)
            {
                vr = div_by(vr, P.totalWeight, P.invTotalWeight);
                vg = div_by(vg, P.totalWeight, P.invTotalWeight);
                vb = div_by(vb, P.totalWeight, P.invTotalWeight);
                va = div_by(va, P.totalWeight, P.invTotalWeight);
            }
            else
            {
                vr = vg = vb = va = 0.0f;
            }
            const uint32_t vol = dither_b4(P.ditherMode, x, y, z, vr, vg, vb, va);
            const uint32_t q0 = unorm8(ir), q1 = unorm8(ig), q2 = unorm8(ib), q3 = unorm8(ia);
            P.vol[idx] = vol;
            if(P.iso)
            {
                P.iso[idx] = q0 | (q1 << 8) | (q2 << 16) | (q3 << 24);
                if(q3 >= 128u)
                    mark_iso_cells(P, x, x, y, z);
            }
        }
    }

    // non-persistent source -> functor-applied float texture incl. guard
    // (UpdatePersistendTextureKernel, lib/isaac/isaac_common_kernel.hpp:432-451)
    __global__ __launch_bounds__(256) void persistent_copy_kernel(
        const float* src,
        int64_t sx,
        int64_t sy,
        int64_t sz,
        int dim,
        ChainDesc chain,
        int gX,
        int gY,
        int gZ,
        int guard,
        float* dst)
    {
        const int64_t n = int64_t(gX) * gY * gZ;
        for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
        {
            int x = int(i % gX), y = int((i / gX) % gY), z = int(i / (int64_t(gX) * gY));
            int cx = x - guard, cy = y - guard, cz = z - guard;
            const float* e = src + (int64_t(cx) * sx + int64_t(cy) * sy + int64_t(cz) * sz) * dim;
            float c0 = e[0], c1 = dim > 1 ? e[1] : 0.f, c2 = dim > 2 ? e[2] : 0.f, c3 = dim > 3 ? e[3] : 0.f;
            dst[i] = apply_chain(chain, c0, c1, c2, c3, dim);
        }
    }

    // ------------------------------------------------------------------ SSAO
    __device__ __attribute__((always_inline)) inline void ssao_body(const FrameParams& F, uint32_t tile)
    {
        int px, py;
        if(!tile_pixel_at(F, tile, px, py))
            return;
        const float ref = F.depth[size_t(py) * F.W + px];
        float occ = 0.0f;
#pragma unroll
        for(int i = -3; i <= 3; ++i)
        {
            const int sx = iclamp(px + i * 10, 0, F.W - 1);
#pragma unroll
            for(int j = -3; j <= 3; ++j)
            {
                const int sy = iclamp(py + j * 10, 0, F.H - 1);
                if(F.depth[size_t(sy) * F.W + sx] < ref)
                    occ = occ + 1.0f;
            }
        }
        F.ao[size_t(py) * F.W + px] = gclamp(occ / 42.0f, 0.0f, 1.0f);
    }

    // ssao_body's count with the depth taps from LDS: a workgroup takes a 64x32 block
    // of the viewport and stages the 124x92 depth region around it (the 30-pixel reach
    // of the 7x7 taps at a stride of 10), each region texel read at its framebuffer-
    // clamped position -- so region[px + 10 i - x0 + 30] is the clamped tap itself and
    // the 49 taps are LDS reads at fixed offsets.  The count is exact (at most 49
    // increments of 1), so the occlusion equals ssao_body's.
    constexpr int kSsaoBW = 64, kSsaoBH = 32, kSsaoReach = 30;
    constexpr int kSsaoRW = kSsaoBW + 2 * kSsaoReach, kSsaoRH = kSsaoBH + 2 * kSsaoReach; // 124 x 92
    // SHADE: the block also shades its pixels with the occlusion term it just formed (render
    // modes that leave the depth buffer alone, so no block changes a depth another one reads)
    // the G-buffer values the shading of one pixel reads (besides occlusion and depth)
    struct ShadeIn
    {
        uint32_t cb;
        F3 normal;
        float4 v;
    };

    __device__ __attribute__((always_inline)) inline ShadeIn shade_load(const FrameParams& F, size_t p);
    __device__ __attribute__((always_inline)) inline void shade_finish(const FrameParams& F, int px, int py, const ShadeIn& in,
                                                                      float ao, float depth);

    template<bool SHADE>
    __global__ __launch_bounds__(256) void ssao_tiled_kernel(const FrameParams F)
    {
        __shared__ float region[kSsaoRW * kSsaoRH];
        const int nbX = (F.vx1 - F.vx0 + kSsaoBW - 1) / kSsaoBW;
        const int x0 = F.vx0 + int(blockIdx.x % uint32_t(nbX)) * kSsaoBW;
        const int y0 = F.vy0 + int(blockIdx.x / uint32_t(nbX)) * kSsaoBH;
        // staging: thread t loads column t % 124 of rows t / 124 + 2 k (248 threads)
        const int col = int(threadIdx.x) % kSsaoRW, r0 = int(threadIdx.x) / kSsaoRW;
        if(r0 < 2)
        {
            const int gx = iclamp(x0 - kSsaoReach + col, 0, F.W - 1);
            const float* src = F.depth + gx;
#pragma unroll 4
            for(int r = r0; r < kSsaoRH; r += 2)
            {
                const int gy = iclamp(y0 - kSsaoReach + r, 0, F.H - 1);
                region[r * kSsaoRW + col] = src[size_t(gy) * F.W];
            }
        }
        __syncthreads();
#pragma unroll
        for(int k = 0; k < kSsaoBW * kSsaoBH / 256; k++)
        {
            const int q = int(threadIdx.x) + 256 * k;
            const int px = x0 + (q & (kSsaoBW - 1)), py = y0 + q / kSsaoBW;
            if(px >= F.vx1 || py >= F.vy1)
                continue;
            // (SHADE: this pixel's G-buffer values are requested before its taps are counted)
            ShadeIn in;
            if(SHADE)
                in = shade_load(F, size_t(py) * size_t(F.W) + size_t(px));
            // the tap (-3, -3) of this pixel; every tap is a fixed offset from it
            const float* t0 = region + (py - y0) * kSsaoRW + (px - x0);
            const float ref = t0[kSsaoReach * kSsaoRW + kSsaoReach];
            float occ = 0.0f;
#pragma unroll
            for(int i = 0; i < 7; ++i)
#pragma unroll
                for(int j = 0; j < 7; ++j)
                    if(t0[(j * 10) * kSsaoRW + i * 10] < ref)
                        occ = occ + 1.0f;
            const float ao = gclamp(occ / 42.0f, 0.0f, 1.0f);
            F.ao[size_t(py) * F.W + px] = ao;
            if(SHADE)
                shade_finish(F, px, py, in, ao, ref);
        }
    }

    // ------------------------------------------------------------------ shading + blend
    // ShadingKernel (lib/isaac/isaac_common_kernel.hpp:220-320), then the volume
    // pass's final blend color + (1 - color.a) * solid
    // (lib/isaac/isaac_volume_kernel.hpp:83-86) for pixels whose volume pass ran.
    __device__ __attribute__((always_inline)) inline ShadeIn shade_load(const FrameParams& F, size_t p)
    {
        ShadeIn in;
        in.cb = F.color[p];
        in.normal = f3(F.normal[3 * p + 0], F.normal[3 * p + 1], F.normal[3 * p + 2]);
        in.v = F.volColor[p];
        return in;
    }

    // one pixel, given its G-buffer values, occlusion term and depth
    __device__ __attribute__((always_inline)) inline void shade_finish(const FrameParams& F, int px, int py, const ShadeIn& in,
                                                                      float ao, float depth)
    {
        const size_t p = size_t(py) * size_t(F.W) + size_t(px);
        const uint32_t cb = in.cb;
        F4 color = F4{div255(float(cb & 0xffu)), div255(float((cb >> 8) & 0xffu)), div255(float((cb >> 16) & 0xffu)),
                      div255(float(cb >> 24))};
        const F3 normal = in.normal;
        const float aoStrength = 1.0f - ao;
        const int mode = F.renderMode;
        uint32_t solid = cb;
        bool depthChanged = false;
        if(mode == 7)
            color = F4{F.rankHue[0], F.rankHue[1], F.rankHue[2], color.w};
        if(mode < 3 || mode == 7)
        {
            const Ray ray = pixel_to_ray(F, px, py);
            const F3 lightDir = f3(-ray.dir.x, -ray.dir.y, -ray.dir.z);
            float lightFactor = fabsf(dot3(normal, lightDir));
            const F3 half = normalize3(add(lightDir, lightDir));
            float spec = dot3(normal, half);
            const float s2 = spec * spec;
            spec = s2 * s2;
            spec = spec * 0.5f;
            if(mode == 1)
                spec = 0.0f;
            const float w = F.aoWeight;
            const float aoF = (1.0f - w) + w * aoStrength;
            lightFactor = lightFactor + aoF;
            lightFactor = lightFactor * 0.5f;
            solid = to_byte4(gmin(color.x * lightFactor + spec, 1.0f), gmin(color.y * lightFactor + spec, 1.0f),
                             gmin(color.z * lightFactor + spec, 1.0f), color.w);
            if(mode == 2 || mode == 7)
            {
                depth = 0.0f;
                depthChanged = true;
            }
        }
        else if(mode == 3)
            solid = to_byte4(F.bg[0], F.bg[1], F.bg[2], color.w);
        else if(mode == 4)
        {
            solid = to_byte4(normal.x * 0.5f + 0.5f, normal.y * 0.5f + 0.5f, normal.z * 0.5f + 0.5f, color.w);
            depth = 0.0f;
            depthChanged = true;
        }
        else if(mode == 5)
        {
            const float d = depth / F.maxGlobalSizeScaled;
            solid = to_byte4(d, d, d, color.w);
            depth = 0.0f;
            depthChanged = true;
        }
        else if(mode == 6)
        {
            const float w = F.aoWeight;
            const float aoF = (1.0f - w) + w * aoStrength;
            solid = to_byte4(aoF, aoF, aoF, color.w);
            depth = 0.0f;
            depthChanged = true;
        }
        else if(mode == 8)
        {
            solid = to_byte4(F.rankHue[0], F.rankHue[1], F.rankHue[2], 1.0f);
            depth = 0.0f;
            depthChanged = true;
        }
        uint32_t out = solid;
        const float4 v = in.v;
        const float sr = div255(float(solid & 0xffu)), sg = div255(float((solid >> 8) & 0xffu));
        const float sb = div255(float((solid >> 16) & 0xffu)), sa = div255(float(solid >> 24));
        float4 fo = make_float4(sr, sg, sb, sa);
        if(v.w >= 0.0f)
        {
            const float om = 1.0f - v.w;
            fo = make_float4(v.x + om * sr, v.y + om * sg, v.z + om * sb, v.w + om * sa);
            out = to_byte4(fo.x, fo.y, fo.z, fo.w);
        }
        if(F.outFloat)
            F.outFloat[p] = make_float4(gclamp(fo.x, 0.f, 1.f), gclamp(fo.y, 0.f, 1.f), gclamp(fo.z, 0.f, 1.f), gclamp(fo.w, 0.f, 1.f));
        F.color[p] = out;
        if(depthChanged)
            F.depth[p] = depth;
    }

    __device__ __attribute__((always_inline)) inline void shade_body(const FrameParams& F, uint32_t tile)
    {
        int px, py;
        if(!tile_pixel_at(F, tile, px, py))
            return;
        const size_t p = size_t(py) * size_t(F.W) + size_t(px);
        shade_finish(F, px, py, shade_load(F, p), F.aoEnabled ? F.ao[p] : 0.0f, F.depth[p]);
    }

    __global__ __launch_bounds__(256) void shade_kernel(const FrameParams F)
    {
        shade_body(F, xcd_tile(F, blockIdx.x));
    }

    // ------------------------------------------------------------------ precision form
    // Field bricks (FP32 / FP16 / BF16 + FP32 scale) rendered with
    // post-classification: interpolate the raw field, then functor chain and
    // transfer function per sample (the semantics of the reference's legacy
    // renderer, lib/isaac/isaac_volume_kernel.hpp:101-168), blended across
    // sources as the classification pass does (lib/isaac/isaac_common_kernel.hpp:574-612)
    // but without the RGBA8 quantisation.  The ray setup (pixelToRay + clipRay)
    // runs in binary64; interpolation and compositing accumulate in binary32.

    struct RayD
    {
        double dir[3], start[3];
        double startDepth, endDepth;
        bool isClipped;
        double clipN[3];
    };

    __device__ inline bool ray_setup_d(const FrameParams& F, const PostParams& Q, int px, int py, RayD& r)
    {
        const double vx = double(px) / double(F.fbW) * 2.0 - 1.0;
        const double vy = double(py) / double(F.fbH) * 2.0 - 1.0;
        double s[4], e[4];
        for(int k = 0; k < 4; k++)
        {
            const double s0 = Q.invd[0 * 4 + k] * vx + Q.invd[1 * 4 + k] * vy;
            s[k] = s0 + (Q.invd[3 * 4 + k] - Q.invd[2 * 4 + k]);
            e[k] = s0 + (Q.invd[3 * 4 + k] + Q.invd[2 * 4 + k]);
        }
        double d[3], len2 = 0.0;
        for(int k = 0; k < 3; k++)
        {
            r.start[k] = s[k] / s[3] * Q.maxSized;
            d[k] = e[k] / e[3] * Q.maxSized - r.start[k];
            len2 += d[k] * d[k];
        }
        const double il = 1.0 / sqrt(len2);
        double bmin[3], bmax[3];
        for(int k = 0; k < 3; k++)
        {
            r.dir[k] = d[k] * il;
            r.start[k] += double(F.off[k]);
            bmin[k] = (double(F.bbMin[k]) - r.start[k]) / r.dir[k];
            bmax[k] = (double(F.bbMax[k]) - r.start[k]) / r.dir[k];
            if(bmax[k] < bmin[k])
            {
                const double t = bmax[k];
                bmax[k] = bmin[k];
                bmin[k] = t;
            }
            r.clipN[k] = 0.0;
        }
        r.isClipped = false;
        r.startDepth = fmax(bmin[0], fmax(bmin[1], bmin[2]));
        r.endDepth = fmin(bmax[0], fmin(bmax[1], bmax[2]));
        for(int k = 0; k < 3; k++)
        {
            const double sgn = (r.dir[k] > 0.0) ? 1.0 : ((r.dir[k] < 0.0) ? -1.0 : 0.0);
            if(bmin[k] == r.startDepth && ((F.outerLow[k] && sgn + 1.0 != 0.0) || (F.outerHigh[k] && sgn - 1.0 != 0.0)))
            {
                r.isClipped = true;
                r.clipN[k] = sgn;
            }
        }
        for(int i = 0; i < F.nclip; i++)
        {
            double dn = 0.0, pn = 0.0, sn = 0.0;
            for(int k = 0; k < 3; k++)
            {
                dn += r.dir[k] * double(F.cnorm[i][k]);
                pn += Q.cposd[i][k] * double(F.cnorm[i][k]);
                sn += r.start[k] * double(F.cnorm[i][k]);
            }
            const double t = (pn - sn) / dn;
            if(dn > 0.0)
            {
                if(r.endDepth < t)
                    return false;
                if(r.startDepth <= t)
                {
                    for(int k = 0; k < 3; k++)
                        r.clipN[k] = double(F.cnorm[i][k]);
                    r.isClipped = true;
                    r.startDepth = t;
                }
            }
            else
            {
                if(r.startDepth > t)
                    return false;
                if(r.endDepth > t)
                    r.endDepth = t;
            }
        }
        r.startDepth = fmax(r.startDepth, double(kZNear));
        return !(r.startDepth > r.endDepth || isinf(r.startDepth) || isinf(r.endDepth));
    }

    __device__ inline float half_lo(uint32_t v)
    {
        return __half2float(__ushort_as_half((unsigned short) (v & 0xffffu)));
    }
    __device__ inline float half_hi(uint32_t v)
    {
        return __half2float(__ushort_as_half((unsigned short) (v >> 16)));
    }

    // Tap geometry of one sample position, shared by every source (all sources
    // of a rank have the local box's brick grid).  Sampler LINEAR|NEAREST with
    // CLAMP addressing (lib/isaac/isaac_texture.hpp:182-259): the taps of a sample
    // all come from the brick holding its clamped (x0, y0, z0) tap; where x1 = x0
    // (clamped at the edge) the second element of each pair gets weight 0.
    struct BrickTaps
    {
        uint32_t brick; // brick index
        uint32_t i00, i10, i01, i11; // pair index in a component block of rows (y0,z0) (y1,z0) (y0,z1) (y1,z1)
        // trilinear weights of the corners (x, y, z) = 000 001 010 011 100 101 110 111,
        // shared by every component of every source at this position; where both x
        // taps are texel x0 (CLAMP at the x edge) the x1 corners weigh 0
        float w[8];
    };

    template<bool LINEAR>
    __device__ inline BrickTaps brick_taps(const PostParams& Q, int X, int Y, int Z, float px, float py, float pz)
    {
        BrickTaps t;
        if(!LINEAR)
        {
            const uint32_t x = iclamp(int(px), 0, X - 1), y = iclamp(int(py), 0, Y - 1), z = iclamp(int(pz), 0, Z - 1);
            t.brick = ((z >> 3) * uint32_t(Q.nby) + (y >> 3)) * uint32_t(Q.nbx) + (x >> 3);
            t.i00 = ((z & 7) * 9 + (y & 7)) * 8 + (x & 7);
            t.i10 = t.i01 = t.i11 = t.i00;
            return t;
        }
        const float cx = px - 0.5f, cy = py - 0.5f, cz = pz - 0.5f;
        const float flx = floorf(cx), fly = floorf(cy), flz = floorf(cz);
        const int bx = int(flx), by = int(fly), bz = int(flz);
        const uint32_t x0 = iclamp(bx, 0, X - 1), x1 = iclamp(bx + 1, 0, X - 1);
        const uint32_t y0 = iclamp(by, 0, Y - 1), y1 = iclamp(by + 1, 0, Y - 1);
        const uint32_t z0 = iclamp(bz, 0, Z - 1), z1 = iclamp(bz + 1, 0, Z - 1);
        const uint32_t Bx = x0 >> 3, By = y0 >> 3, Bz = z0 >> 3;
        const uint32_t lx = x0 - (Bx << 3);
        const uint32_t ly0 = y0 - (By << 3), ly1 = y1 - (By << 3);
        const uint32_t lz0 = z0 - (Bz << 3), lz1 = z1 - (Bz << 3);
        t.brick = (Bz * uint32_t(Q.nby) + By) * uint32_t(Q.nbx) + Bx;
        t.i00 = lx + (lz0 * 9 + ly0) * 8;
        t.i10 = lx + (lz0 * 9 + ly1) * 8;
        t.i01 = lx + (lz1 * 9 + ly0) * 8;
        t.i11 = lx + (lz1 * 9 + ly1) * 8;
        const float fx = x1 == x0 ? 0.0f : cx - flx, fy = cy - fly, fz = cz - flz;
        const float ox = 1.0f - fx, oy = 1.0f - fy, oz = 1.0f - fz;
        const float w00 = oy * oz, w01 = oy * fz, w10 = fy * oz, w11 = fy * fz;
        t.w[0] = ox * w00;
        t.w[1] = ox * w01;
        t.w[2] = ox * w10;
        t.w[3] = ox * w11;
        t.w[4] = fx * w00;
        t.w[5] = fx * w01;
        t.w[6] = fx * w10;
        t.w[7] = fx * w11;
        return t;
    }

    // the DIM pairs of one pair row (all components of a source side by side):
    // lo[c] = v_c[x], hi[c] = v_c[x+1], still divided by the brick scale.  One
    // struct load per row, which the compiler emits as one wide global load.
    template<int N>
    struct Words
    {
        uint32_t w[N];
    };

    // 32-bit words of one pair row: 2 per component in FP32, 1 (two 16-bit halves) otherwise
    template<int DT, int DIM>
    constexpr int row_words()
    {
        return DT == kDtF32 ? 2 * DIM : DIM;
    }

    // The raw words of one source's sample: its 1 (NEAREST) or 4 (LINEAR) pair
    // rows and its brick scales, sized for 4 components.  Fetching is split
    // from interpolation so that the rows of every source of a sample are
    // requested before the first of them is used.
    template<int DT>
    struct SlotRaw
    {
        uint32_t r[4][row_words<DT, 4>()];
        uint32_t sc[4];
    };

    template<int DT, bool LINEAR, int DIM>
    __device__ inline void slot_fetch_dim(const BrickSource& S, const BrickTaps& t, SlotRaw<DT>& R)
    {
        constexpr int W = row_words<DT, DIM>();
        const Words<W>* rows = reinterpret_cast<const Words<W>*>(S.data) + t.brick * uint32_t(kBrickPairs);
        const uint32_t idx[4] = {t.i00, t.i10, t.i01, t.i11};
#pragma unroll
        for(int k = 0; k < (LINEAR ? 4 : 1); k++)
        {
            const Words<W> a = rows[idx[k]];
#pragma unroll
            for(int w = 0; w < W; w++)
                R.r[k][w] = a.w[w];
        }
        const Words<DIM> sc = reinterpret_cast<const Words<DIM>*>(S.scale)[t.brick];
#pragma unroll
        for(int c = 0; c < DIM; c++)
            R.sc[c] = sc.w[c];
    }

    template<int DT, bool LINEAR>
    __device__ __attribute__((always_inline)) inline void slot_fetch(const BrickSource& S, const BrickTaps& t, SlotRaw<DT>& R)
    {
        switch(S.dim)
        {
        case 1: slot_fetch_dim<DT, LINEAR, 1>(S, t, R); break;
        case 2: slot_fetch_dim<DT, LINEAR, 2>(S, t, R); break;
        case 3: slot_fetch_dim<DT, LINEAR, 3>(S, t, R); break;
        default: slot_fetch_dim<DT, LINEAR, 4>(S, t, R); break;
        }
    }

    // lo[c] = v_c[x], hi[c] = v_c[x+1] of one fetched row (still divided by the brick scale)
    template<int DT, int DIM>
    __device__ inline void decode_row(const uint32_t* w, float lo[DIM], float hi[DIM])
    {
#pragma unroll
        for(int c = 0; c < DIM; c++)
        {
            if constexpr(DT == kDtF32)
            {
                lo[c] = __uint_as_float(w[2 * c]);
                hi[c] = __uint_as_float(w[2 * c + 1]);
            }
            else if constexpr(DT == kDtF16)
            {
                lo[c] = half_lo(w[c]);
                hi[c] = half_hi(w[c]);
            }
            else
            {
                lo[c] = __uint_as_float(w[c] << 16);
                hi[c] = __uint_as_float(w[c] & 0xffff0000u);
            }
        }
    }

    // raw sample of every component of one source with DIM components (v[c], c < DIM)
    template<int DT, bool LINEAR, int DIM>
    __device__ inline void slot_interp(const SlotRaw<DT>& R, const BrickTaps& t, float v[4])
    {
        if(!LINEAR)
        {
            float a[DIM], b[DIM];
            decode_row<DT, DIM>(R.r[0], a, b);
#pragma unroll
            for(int c = 0; c < DIM; c++)
                v[c] = a[c] * __uint_as_float(R.sc[c]);
            return;
        }
        float d000[DIM], d100[DIM], d010[DIM], d110[DIM], d001[DIM], d101[DIM], d011[DIM], d111[DIM];
        decode_row<DT, DIM>(R.r[0], d000, d100);
        decode_row<DT, DIM>(R.r[1], d010, d110);
        decode_row<DT, DIM>(R.r[2], d001, d101);
        decode_row<DT, DIM>(R.r[3], d011, d111);
        // sum of the corners times their weights (one multiply and seven fmas per
        // component), then the brick scale; equal to the nested lerps in exact arithmetic
#pragma unroll
        for(int c = 0; c < DIM; c++)
        {
            float a = d000[c] * t.w[0];
            a = __builtin_fmaf(d001[c], t.w[1], a);
            a = __builtin_fmaf(d010[c], t.w[2], a);
            a = __builtin_fmaf(d011[c], t.w[3], a);
            a = __builtin_fmaf(d100[c], t.w[4], a);
            a = __builtin_fmaf(d101[c], t.w[5], a);
            a = __builtin_fmaf(d110[c], t.w[6], a);
            a = __builtin_fmaf(d111[c], t.w[7], a);
            v[c] = a * __uint_as_float(R.sc[c]);
        }
    }

    // the functor-chain value of one source's sample, dispatched on its component
    // count (fetch and interpolation in the same case: one source at a time)
    template<int DT, bool LINEAR, int DIM>
    __device__ inline void slot_sample(const BrickSource& S, const BrickTaps& t, float v[4])
    {
        SlotRaw<DT> R;
        slot_fetch_dim<DT, LINEAR, DIM>(S, t, R);
        slot_interp<DT, LINEAR, DIM>(R, t, v);
    }

    template<int DT, bool LINEAR>
    __device__ __attribute__((always_inline)) inline float brick_value(const BrickSource& S, const BrickTaps& t)
    {
        float v[4] = {0.f, 0.f, 0.f, 0.f};
        switch(S.dim)
        {
        case 1: slot_sample<DT, LINEAR, 1>(S, t, v); break;
        case 2: slot_sample<DT, LINEAR, 2>(S, t, v); break;
        case 3: slot_sample<DT, LINEAR, 3>(S, t, v); break;
        default: slot_sample<DT, LINEAR, 4>(S, t, v); break;
        }
        // one chain per source slot, with the component count as a value
        return apply_chain(S.chain, v[0], v[1], v[2], v[3], S.dim);
    }

    // Source signature: the component counts of the enabled sources in slot
    // order, as base-5 digits (slot 0 lowest), 0 = resolved at run time.  A
    // march compiled for one signature fetches the rows of all its sources
    // before interpolating any of them, so their latencies overlap.
    constexpr bool sig_natural(int sig)
    {
        return sig >= kSigNatural;
    }

    constexpr int sig_count(int sig)
    {
        int n = 0;
        for(sig %= kSigNatural; sig > 0; sig /= 5)
            n++;
        return n;
    }

    constexpr int sig_dim(int sig, int slot)
    {
        sig %= kSigNatural;
        for(int i = 0; i < slot; i++)
            sig /= 5;
        return sig % 5;
    }

    // the natural chain's value of a D-component sample: the value itself, or the length
    // with apply_chain's association ((v0 v0 + v1 v1) + v2 v2)
    template<int D>
    __device__ inline float natural_value(const float (&v)[4])
    {
        if constexpr(D == 1)
            return v[0];
        else if constexpr(D == 2)
            return sqrtf(v[0] * v[0] + v[1] * v[1]);
        else if constexpr(D == 3)
            return sqrtf(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        else
            return sqrtf((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]));
    }

    template<int DT, bool LINEAR, int SIG, int S>
    __device__ __attribute__((always_inline)) inline void sig_fetch(const PostParams& Q, const BrickTaps& t, SlotRaw<DT>* R)
    {
        if constexpr(S < sig_count(SIG))
        {
            slot_fetch_dim<DT, LINEAR, sig_dim(SIG, S)>(Q.src[S], t, R[S]);
            sig_fetch<DT, LINEAR, SIG, S + 1>(Q, t, R);
        }
    }

    struct PostSample
    {
        float r, g, b, a; // premultiplied, normalised volume colour
        float ir, ig, ib, ia; // iso colour and alpha (alpha / threshold * 0.5, maximum over sources)
    };

    // one source's classified sample into the running sums (weights in slot order)
    __device__ __attribute__((always_inline)) inline void post_accumulate(PostSample& o, const BrickSource& S, const float4 col)
    {
        if(S.weight > 0.0f)
        {
            const float a = col.w * S.weight;
            o.r = o.r + col.x * a;
            o.g = o.g + col.y * a;
            o.b = o.b + col.z * a;
            o.a = o.a + a;
        }
        if(S.iso > 0.0f)
        {
            const float a = col.w * S.isoScale;
            if(o.ia < a)
            {
                o.ir = col.x;
                o.ig = col.y;
                o.ib = col.z;
                o.ia = a;
            }
        }
    }

    template<int DT, bool LINEAR, int SIG, int S>
    __device__ __attribute__((always_inline)) inline void sig_classify(
        const PostParams& Q, const float4* lut, const BrickTaps& t, const SlotRaw<DT>* R, PostSample& o)
    {
        if constexpr(S < sig_count(SIG))
        {
            constexpr int D = sig_dim(SIG, S);
            float v[4] = {0.f, 0.f, 0.f, 0.f};
            slot_interp<DT, LINEAR, D>(R[S], t, v);
            const float tv = sig_natural(SIG) ? natural_value<D>(v) : apply_chain(Q.src[S].chain, v[0], v[1], v[2], v[3], D);
            post_accumulate(o, Q.src[S], lut[S * Q.T + tf_index(tv, Q.T)]);
            sig_classify<DT, LINEAR, SIG, S + 1>(Q, lut, t, R, o);
        }
    }

    template<int DT, bool LINEAR, int SIG>
    __device__ __attribute__((always_inline)) inline PostSample post_classify(const PostParams& Q, const float4* lut, int X, int Y, int Z, float px, float py, float pz)
    {
        const BrickTaps t = brick_taps<LINEAR>(Q, X, Y, Z, px, py, pz);
        PostSample o{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if constexpr(SIG != 0)
        {
            SlotRaw<DT> R[sig_count(SIG)];
            sig_fetch<DT, LINEAR, SIG, 0>(Q, t, R);
            sig_classify<DT, LINEAR, SIG, 0>(Q, lut, t, R, o);
        }
        else
        {
            // unrolled over the source slots so every parameter-block index is constant
#pragma unroll
            for(int s = 0; s < kMaxBrickSources; s++)
            {
                if(s >= Q.nsrc)
                    break;
                const BrickSource& S = Q.src[s];
                const float tv = brick_value<DT, LINEAR>(S, t);
                post_accumulate(o, S, lut[s * Q.T + tf_index(tv, Q.T)]);
            }
        }
        // invTotalWeight = 1 / (sum of volume-source weights), 0 when that sum is 0
        o.r = o.r * Q.invTotalWeight;
        o.g = o.g * Q.invTotalWeight;
        o.b = o.b * Q.invTotalWeight;
        o.a = o.a * Q.invTotalWeight;
        return o;
    }

    // Post-classification march over field bricks.  Same pass structure as
    // march_kernel (clear, particle DDA, one traversal serving iso and volume,
    // G-buffer + premultiplied volume colour out); sample positions
    // startU + stepVec*i with startSteps / end steps taken from the binary64 ray.
    // the enabled sources' transfer functions, staged in LDS in source order
    __device__ inline void stage_luts(float4* lds_lut, const PostParams& Q)
    {
#pragma unroll
        for(int j = 0; j < kMaxBrickSources; j++)
        {
            if(j >= Q.nsrc)
                break;
            const float4* src = Q.luts + size_t(Q.src[j].lutSlot) * Q.T;
            for(int i = threadIdx.x; i < Q.T; i += blockDim.x)
                lds_lut[j * Q.T + i] = src[i];
        }
    }

    template<int DT, bool LINEAR, bool COUNT, int SIG = 0>
    __device__ __attribute__((always_inline)) inline void brick_march_body(
        const FrameParams& F,
        const PostParams& Q,
        const ParticleParams& PP,
        const float4* lut,
        uint32_t tile)
    {
        int px, py;
        const bool valid = tile_pixel_at(F, tile, px, py);
        unsigned long long nVol = 0, nIso = 0, nIsoHits = 0, nVolRays = 0, nIsoRays = 0;
        unsigned long long nCells = 0, nTests = 0, nPartRays = 0, nSteps = 0;
        if(valid)
        {
            const size_t p = size_t(py) * size_t(F.W) + size_t(px);
            uint32_t color = F.bgClear;
            F3 normal = f3(0.f, 0.f, 0.f);
            float depth = FLT_MAX;
            float4 vcol = make_float4(0.f, 0.f, 0.f, -1.f);
            RayD rd;
            const bool inside = ray_setup_d(F, Q, px, py, rd);
            Ray ray;
            ray.dir = f3(float(rd.dir[0]), float(rd.dir[1]), float(rd.dir[2]));
            ray.start = f3(float(rd.start[0]), float(rd.start[1]), float(rd.start[2]));
            ray.startDepth = float(rd.startDepth);
            ray.endDepth = float(rd.endDepth);
            ray.isClipped = rd.isClipped;
            ray.clipN = f3(float(rd.clipN[0]), float(rd.clipN[1]), float(rd.clipN[2]));
            if(inside && PP.nsrc > 0)
            {
                nPartRays++;
                particle_dda<COUNT>(PP, ray, color, depth, normal, nCells, nTests);
            }
            const int mode = F.renderMode;
            const bool depthZeroed = mode == 2 || (mode >= 4 && mode <= 8);
            if(inside)
            {
                const double endD = fmin(rd.endDepth, double(depth));
                bool isoOn = F.isoEnabled && endD > rd.startDepth;
                bool volBlend = F.volumeEnabled && !depthZeroed && endD > rd.startDepth;
                if(isoOn || volBlend)
                {
                    const F3 sc = f3(F.scale[0], F.scale[1], F.scale[2]);
                    const double ex = rd.dir[0] / double(sc.x), ey = rd.dir[1] / double(sc.y), ez = rd.dir[2] / double(sc.z);
                    const double stepUd = double(F.step)
                        * (sqrt(rd.dir[0] * rd.dir[0] + rd.dir[1] * rd.dir[1] + rd.dir[2] * rd.dir[2]) / sqrt(ex * ex + ey * ey + ez * ez));
                    const float stepU = float(stepUd);
                    const float factor = stepU / F.minSize * 2.0f * F.totalWeightAll;
                    const int startSteps = int(ceil(rd.startDepth / stepUd));
                    const int endIso = int(floor(endD / stepUd));
                    int endVol = endIso;
                    const F3 stepVec = divv(muls(ray.dir, stepU), sc);
                    const F3 startU = divv(ray.start, sc);
                    if(isoOn)
                        nIsoRays++;
                    float cr = 0.f, cg = 0.f, cb = 0.f, ca = 0.f;
                    float oldValue = 0.0f;
                    // traversal state as step bounds, not flags (no lane masks carried by the
                    // loop): the iso test runs while i <= isoEnd, the volume while i <= volEnd,
                    // either set below every step to switch it off; hitStep is the hit's step
                    const int off = -0x7fffffff;
                    int isoEnd = isoOn ? endIso : off;
                    int volEnd = volBlend ? endVol : off;
                    int hitStep = -1;
                    for(int i = startSteps;; i++)
                    {
                        if(i > (isoEnd > volEnd ? isoEnd : volEnd))
                            break;
                        if(COUNT)
                            nSteps++;
                        const float fi = float(i);
                        const PostSample sm = post_classify<DT, LINEAR, SIG>(
                            Q, lut, F.X, F.Y, F.Z, startU.x + stepVec.x * fi, startU.y + stepVec.y * fi, startU.z + stepVec.z * fi);
                        if(i <= isoEnd)
                        {
                            const float value = gmin(sm.ia, 1.0f);
                            if(COUNT)
                                nIso++;
                            const float tmp = oldValue;
                            oldValue = value;
                            if(value >= 0.5f)
                            {
                                const bool first = ray.isClipped && i == startSteps;
                                depth = first ? ray.startDepth : fi * stepU + stepU * (0.5f - tmp) / (value - tmp);
                                hitStep = i;
                                isoEnd = off;
                                if(COUNT)
                                    nIsoHits++;
                                // the volume pass ends at min(clip end, iso depth)
                                const double ve = fmin(rd.endDepth, double(depth));
                                if(!(ve > rd.startDepth))
                                    volEnd = off;
                                else if(volEnd != off)
                                    volEnd = int(floor(ve / stepUd));
                            }
                        }
                        if(i <= volEnd)
                        {
                            if(COUNT)
                                nVol++;
                            const float w = 1.0f - ca;
                            cr = cr + w * (sm.r * factor);
                            cg = cg + w * (sm.g * factor);
                            cb = cb + w * (sm.b * factor);
                            ca = ca + w * (sm.a * factor);
                            if(ca > 0.99f)
                                volEnd = off;
                        }
                    }
                    const bool isoHit = hitStep >= 0;
                    const bool isoFirst = isoHit && ray.isClipped && hitStep == startSteps;
                    // a hit at or before the ray's start leaves no volume segment to blend
                    if(isoHit && !(fmin(rd.endDepth, double(depth)) > rd.startDepth))
                        volBlend = false;
                    if(isoHit)
                    {
                        const F3 pu = divv(add(ray.start, muls(ray.dir, depth)), sc);
                        // hit colour, then the six central-difference samples of the iso value
                        // (one loop, so the per-sample classification is inlined once)
                        float hr = 0.f, hg = 0.f, hb = 0.f;
                        F3 g = f3(0.f, 0.f, 0.f);
#pragma unroll 1
                        for(int d = -1; d < 6; d++)
                        {
                            const float sx = d == 0 ? 1.0f : (d == 1 ? -1.0f : 0.0f);
                            const float sy = d == 2 ? 1.0f : (d == 3 ? -1.0f : 0.0f);
                            const float sz = d == 4 ? 1.0f : (d == 5 ? -1.0f : 0.0f);
                            const PostSample h = post_classify<DT, LINEAR, SIG>(Q, lut, F.X, F.Y, F.Z, pu.x + sx, pu.y + sy, pu.z + sz);
                            const float v = gmin(h.ia, 1.0f);
                            if(d < 0)
                            {
                                hr = h.ir;
                                hg = h.ig;
                                hb = h.ib;
                            }
                            else if(d == 0)
                                g.x = v;
                            else if(d == 1)
                                g.x = g.x - v;
                            else if(d == 2)
                                g.y = v;
                            else if(d == 3)
                                g.y = g.y - v;
                            else if(d == 4)
                                g.z = v;
                            else
                                g.z = g.z - v;
                        }
                        float gl = len3(g);
                        if(isoFirst || gl == 0.0f)
                        {
                            g = ray.clipN;
                            gl = 1.0f;
                        }
                        normal = f3(-g.x / gl, -g.y / gl, -g.z / gl);
                        color = to_byte4(hr, hg, hb, 1.0f);
                    }
                    if(volBlend)
                    {
                        nVolRays++;
                        vcol = make_float4(cr, cg, cb, ca);
                    }
                }
            }
            F.color[p] = color;
            F.depth[p] = depth;
            F.normal[3 * p + 0] = normal.x;
            F.normal[3 * p + 1] = normal.y;
            F.normal[3 * p + 2] = normal.z;
            F.volColor[p] = vcol;
            if(!F.aoEnabled)
                F.ao[p] = 0.0f;
        }
        if(COUNT)
        {
            block_count_add(F.counters + 0, nVol);
            block_count_add(F.counters + 1, nIso);
            block_count_add(F.counters + 2, nIsoHits);
            block_count_add(F.counters + 3, nCells);
            block_count_add(F.counters + 4, nTests);
            block_count_add(F.counters + 5, nVolRays);
            block_count_add(F.counters + 6, nIsoRays);
            block_count_add(F.counters + 7, nPartRays);
            block_count_add(F.counters + 8, nSteps);
            // the wave runs the traversal loop as long as its longest lane
            int wm = int(nSteps);
            for(int off = 32; off > 0; off >>= 1)
                wm = max(wm, __shfl_xor(wm, off, 64));
            block_count_add(F.counters + 9, (threadIdx.x & 63u) == 0 ? (unsigned long long) wm : 0ull);
        }
    }

    template<int DT, bool LINEAR, bool COUNT>
    __global__ __launch_bounds__(256) void brick_march_kernel(const FrameParams F, const PostParams Q, const ParticleParams PP)
    {
        extern __shared__ float4 lds_lut[];
        stage_luts(lds_lut, Q);
        __syncthreads();
        brick_march_body<DT, LINEAR, COUNT>(F, Q, PP, lds_lut, march_tile(F));
    }

    // trilinear march compiled for one source signature (see sig_count)
    template<int DT, int SIG>
    __global__ __launch_bounds__(256) void brick_march_sig_kernel(const FrameParams F, const PostParams Q, const ParticleParams PP)
    {
        extern __shared__ float4 lds_lut[];
        stage_luts(lds_lut, Q);
        __syncthreads();
        brick_march_body<DT, true, false, SIG>(F, Q, PP, lds_lut, march_tile(F));
    }

    // ------------------------------------------------------------------ batched form
    // One persistent launch over many frames (sub-volume x view): workgroups pop
    // chunks of 16x16 tiles from a global counter until the work is exhausted
    // (every workgroup reaches the exit when the counter passes the last chunk).
    // Frames share the transfer functions (staged once per workgroup).
    template<int DT, bool LINEAR, int SIG = 0>
    __global__ __launch_bounds__(256) void batch_march_kernel(const BatchParams B)
    {
        extern __shared__ float4 lds_lut[];
        __shared__ uint32_t s_work;
        stage_luts(lds_lut, B.posts[0]);
        for(;;)
        {
            __syncthreads();
            if(threadIdx.x == 0)
                s_work = atomicAdd(B.counter, 1u);
            __syncthreads();
            // uniform across the workgroup: keep the work index in a scalar register so
            // the frame's parameter blocks are read with scalar loads
            const uint32_t t0 = uint32_t(__builtin_amdgcn_readfirstlane(int(s_work))) * uint32_t(B.chunk);
            if(t0 >= B.ntiles)
                break;
            const uint32_t t1 = min(t0 + uint32_t(B.chunk), B.ntiles);
            // frame of tile t0: largest i with tileStart[i] <= t0
            int lo = 0, hi = B.nframes - 1;
            while(lo < hi)
            {
                const int mid = (lo + hi + 1) >> 1;
                if(B.tileStart[mid] <= t0)
                    lo = mid;
                else
                    hi = mid - 1;
            }
            int item = __builtin_amdgcn_readfirstlane(lo);
            for(uint32_t t = t0; t < t1; t++)
            {
                while(t >= B.tileStart[item + 1])
                    item++;
                item = __builtin_amdgcn_readfirstlane(item);
                brick_march_body<DT, LINEAR, false, SIG>(B.frames[item], B.posts[item], B.parts[item], lds_lut, t - B.tileStart[item]);
            }
        }
    }

    // per-frame passes of the batch: grid (tiles of the largest frame, frames)
    __global__ __launch_bounds__(256) void batch_ssao_kernel(const FrameParams* frames)
    {
        const FrameParams& F = frames[blockIdx.y];
        if(F.aoEnabled)
            ssao_body(F, blockIdx.x);
    }

    __global__ __launch_bounds__(256) void batch_shade_kernel(const FrameParams* frames)
    {
        shade_body(frames[blockIdx.y], blockIdx.x);
    }


    // per brick and component: scale = max |v| over the 9^3 region (1 if all zero)
    __device__ inline uint32_t to_bf16_rne(float f)
    {
        const uint32_t u = __float_as_uint(f);
        if((u & 0x7f800000u) == 0x7f800000u)
            return (u >> 16) | ((u & 0xffffu) ? 0x40u : 0u); // inf / nan
        return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
    }

    // One workgroup per brick: the brick's 9^3 region (x, y, z clamped to the local
    // box) of all DIM components is read once into LDS; wave c < DIM reduces the
    // max |v| of component c (the brick scale: 1 when the region is all zero or the
    // form is FP32); then every thread writes pairs (v[x], v[x+1]) of the region,
    // divided by the scale and rounded for 16-bit forms.  Output element
    // (brick*648 + pair)*DIM + c, pair = (lz*9 + ly)*8 + lx.
    template<int DT, int DIM>
    __global__ __launch_bounds__(256) void brick_build_kernel(
        const float* src,
        int64_t sx,
        int64_t sy,
        int64_t sz,
        int X,
        int Y,
        int Z,
        int nbx,
        int nby,
        float* scale,
        void* out)
    {
        __shared__ float reg[729 * DIM];
        __shared__ float sc[DIM], rc[DIM];
        __shared__ int64_t rowOff[81]; // element offset of region row (ly, lz), x = 0
        const int64_t brick = blockIdx.x;
        const int Bx = int(brick % nbx), By = int((brick / nbx) % nby), Bz = int(brick / (int64_t(nbx) * nby));
        if(threadIdx.x < 81)
        {
            const int lz = int(threadIdx.x) / 9, ly = int(threadIdx.x) - lz * 9;
            const int y = min(By * 8 + ly, Y - 1), z = min(Bz * 8 + lz, Z - 1);
            rowOff[threadIdx.x] = (int64_t(y) * sy + int64_t(z) * sz) * DIM;
        }
        __syncthreads();
        const int x0 = Bx * 8, xLast = X - 1 - x0; // last local x inside the box
        const int64_t sxD = sx * DIM;
        for(int i = threadIdx.x; i < 729 * DIM; i += 256)
        {
            const int vox = i / DIM, c = i - vox * DIM;
            const int row = vox / 9, lx = vox - row * 9;
            const int x = x0 + min(lx, xLast);
            reg[i] = src[rowOff[row] + int64_t(x) * sxD + c];
        }
        __syncthreads();
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        if(wave < DIM)
        {
            float m = 0.0f;
            if(DT != kDtF32)
                for(int vox = lane; vox < 729; vox += 64)
                    m = fmaxf(m, fabsf(reg[vox * DIM + wave]));
            for(int off = 32; off > 0; off >>= 1)
                m = fmaxf(m, __shfl_xor(m, off));
            const float s = m > 0.0f ? m : 1.0f;
            if(lane == 0)
            {
                sc[wave] = s;
                // RN(1/s) for the quotients, 0 where s is outside [2^-60, 2^60] (there
                // the quotients take the IEEE division)
                rc[wave] = (s >= 0x1p-60f && s <= 0x1p+60f) ? 1.0f / s : 0.0f;
                scale[brick * DIM + wave] = s;
            }
        }
        __syncthreads();
        for(int e = threadIdx.x; e < kBrickPairs * DIM; e += 256)
        {
            const int pair = e / DIM, c = e - pair * DIM;
            const int vox0 = (pair >> 3) * 9 + (pair & 7);
            const float v0 = reg[vox0 * DIM + c], v1 = reg[(vox0 + 1) * DIM + c];
            const int64_t i = brick * (kBrickPairs * DIM) + e;
            if(DT == kDtF32)
                reinterpret_cast<float2*>(out)[i] = make_float2(v0, v1);
            else
            {
                // v / s as x*r plus one fma residual step (div_by), with v's sign (the
                // residual step turns -0 into +0): the IEEE quotient for |v| <= s with s in
                // [2^-60, 2^60]; for BF16, whose range keeps tiny quotients, only where
                // |v| >= 2^-60 (the residual stays normal)
                const float s = sc[c], r = rc[c];
                auto quot = [&](float v) {
                    const bool fast = r != 0.0f && (DT == kDtF16 || fabsf(v) >= 0x1p-60f);
                    return fast ? copysignf(div_by(v, s, r), v) : v / s;
                };
                const float q0 = quot(v0), q1 = quot(v1);
                uint32_t w;
                if(DT == kDtF16)
                    w = uint32_t(__half_as_ushort(__float2half_rn(q0))) | (uint32_t(__half_as_ushort(__float2half_rn(q1))) << 16);
                else
                    w = to_bf16_rne(q0) | (to_bf16_rne(q1) << 16);
                reinterpret_cast<uint32_t*>(out)[i] = w;
            }
        }
    }

    template<int DT>
    hipError_t launch_brick_build(
        const float* src, const int64_t stride[3], int dim, int X, int Y, int Z, int nbx, int nby, int64_t nbricks, float* scale,
        void* out, hipStream_t s)
    {
        const dim3 grid = dim3(static_cast<unsigned>(nbricks)), block = dim3(256);
        switch(dim)
        {
        case 1: hipLaunchKernelGGL((brick_build_kernel<DT, 1>), grid, block, 0, s, src, stride[0], stride[1], stride[2], X, Y, Z, nbx, nby, scale, out); break;
        case 2: hipLaunchKernelGGL((brick_build_kernel<DT, 2>), grid, block, 0, s, src, stride[0], stride[1], stride[2], X, Y, Z, nbx, nby, scale, out); break;
        case 3: hipLaunchKernelGGL((brick_build_kernel<DT, 3>), grid, block, 0, s, src, stride[0], stride[1], stride[2], X, Y, Z, nbx, nby, scale, out); break;
        case 4: hipLaunchKernelGGL((brick_build_kernel<DT, 4>), grid, block, 0, s, src, stride[0], stride[1], stride[2], X, Y, Z, nbx, nby, scale, out); break;
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }

    hipError_t launch_bricks(
        const float* src,
        const int64_t stride[3],
        int dim,
        int X,
        int Y,
        int Z,
        int dtype,
        float* scale,
        void* out,
        hipStream_t s)
    {
        const int nbx = (X + 7) / 8, nby = (Y + 7) / 8, nbz = (Z + 7) / 8;
        const int64_t nbricks = int64_t(nbx) * nby * nbz;
        if(nbricks == 0)
            return hipSuccess;
        if(nbricks > int64_t(0x7fffffff))
            return hipErrorInvalidValue;
        if(dtype == kDtF32)
            return launch_brick_build<kDtF32>(src, stride, dim, X, Y, Z, nbx, nby, nbricks, scale, out, s);
        if(dtype == kDtF16)
            return launch_brick_build<kDtF16>(src, stride, dim, X, Y, Z, nbx, nby, nbricks, scale, out, s);
        return launch_brick_build<kDtBf16>(src, stride, dim, X, Y, Z, nbx, nby, nbricks, scale, out, s);
    }

    static_assert(sizeof(FrameParams) + sizeof(PostParams) + sizeof(ParticleParams) <= 4096, "kernel argument block");

    // a source's chain is its natural one: no operations for a scalar source, one
    // `length` (then nothing) for a vector source
    bool natural_chain(const ChainDesc& c, int dim)
    {
        for(int k = 0; k < kMaxFunctors; k++)
        {
            const int want = (k == 0 && dim > 1) ? OP_LENGTH : OP_IDEM;
            if(c.op[k] != want)
                return false;
        }
        return true;
    }

    bool natural_chains(const PostParams& Q)
    {
        for(int i = 0; i < Q.nsrc; i++)
            if(!natural_chain(Q.src[i].chain, Q.src[i].dim))
                return false;
        return true;
    }

    int post_signature(const PostParams& Q)
    {
        int sig = 0;
        for(int i = Q.nsrc - 1; i >= 0; i--)
            sig = sig * 5 + Q.src[i].dim;
        return Q.nsrc > 0 ? sig : -1;
    }

    hipError_t launch_brick_march(const FrameParams& F, const PostParams& Q, const ParticleParams& PP, bool counting, hipStream_t s)
    {
        const unsigned nb = march_grid(F);
        if(nb == 0)
            return hipSuccess;
        const dim3 grid(nb), block(256);
        const size_t lds = size_t(Q.nsrc) * Q.T * sizeof(float4);
        if(F.linear && !counting)
        {
            // signatures with a compiled march: density (1), vector (3), and pairs of them
            const int sig = post_signature(Q);
            const int v = Q.dtype * 8 + (sig == 1 ? 0 : sig == 3 ? 1 : sig == 6 ? 2 : sig == 8 ? 3 : sig == 16 ? 4 : 7);
            const bool natural = natural_chains(Q);
            switch(v)
            {
#define ISAAC_SIG_CASE(dt, k, sg)                                                                                       \
    case dt * 8 + k:                                                                                                    \
        if(natural)                                                                                                     \
            hipLaunchKernelGGL((brick_march_sig_kernel<dt, sg + kSigNatural>), grid, block, lds, s, F, Q, PP);          \
        else                                                                                                            \
            hipLaunchKernelGGL((brick_march_sig_kernel<dt, sg>), grid, block, lds, s, F, Q, PP);                        \
        return hipGetLastError();
                ISAAC_SIG_CASE(0, 0, 1)
                ISAAC_SIG_CASE(0, 1, 3)
                ISAAC_SIG_CASE(0, 2, 6)
                ISAAC_SIG_CASE(0, 3, 8)
                ISAAC_SIG_CASE(0, 4, 16)
                ISAAC_SIG_CASE(1, 0, 1)
                ISAAC_SIG_CASE(1, 1, 3)
                ISAAC_SIG_CASE(1, 2, 6)
                ISAAC_SIG_CASE(1, 3, 8)
                ISAAC_SIG_CASE(1, 4, 16)
                ISAAC_SIG_CASE(2, 0, 1)
                ISAAC_SIG_CASE(2, 1, 3)
                ISAAC_SIG_CASE(2, 2, 6)
                ISAAC_SIG_CASE(2, 3, 8)
                ISAAC_SIG_CASE(2, 4, 16)
#undef ISAAC_SIG_CASE
            default: break;
            }
        }
        const int v = (Q.dtype * 4) | (F.linear ? 2 : 0) | (counting ? 1 : 0);
        switch(v)
        {
        case 0: hipLaunchKernelGGL((brick_march_kernel<0, false, false>), grid, block, lds, s, F, Q, PP); break;
        case 1: hipLaunchKernelGGL((brick_march_kernel<0, false, true>), grid, block, lds, s, F, Q, PP); break;
        case 2: hipLaunchKernelGGL((brick_march_kernel<0, true, false>), grid, block, lds, s, F, Q, PP); break;
        case 3: hipLaunchKernelGGL((brick_march_kernel<0, true, true>), grid, block, lds, s, F, Q, PP); break;
        case 4: hipLaunchKernelGGL((brick_march_kernel<1, false, false>), grid, block, lds, s, F, Q, PP); break;
        case 5: hipLaunchKernelGGL((brick_march_kernel<1, false, true>), grid, block, lds, s, F, Q, PP); break;
        case 6: hipLaunchKernelGGL((brick_march_kernel<1, true, false>), grid, block, lds, s, F, Q, PP); break;
        case 7: hipLaunchKernelGGL((brick_march_kernel<1, true, true>), grid, block, lds, s, F, Q, PP); break;
        case 8: hipLaunchKernelGGL((brick_march_kernel<2, false, false>), grid, block, lds, s, F, Q, PP); break;
        case 9: hipLaunchKernelGGL((brick_march_kernel<2, false, true>), grid, block, lds, s, F, Q, PP); break;
        case 10: hipLaunchKernelGGL((brick_march_kernel<2, true, false>), grid, block, lds, s, F, Q, PP); break;
        default: hipLaunchKernelGGL((brick_march_kernel<2, true, true>), grid, block, lds, s, F, Q, PP); break;
        }
        return hipGetLastError();
    }

    hipError_t launch_batch_march(const BatchParams& B, int dtype, bool linear, int sig, size_t lds, int grid, hipStream_t s)
    {
        if(B.nframes <= 0 || grid <= 0)
            return hipSuccess;
        const bool natural = sig_natural(sig);
        sig %= kSigNatural;
        if(linear && (sig == 1 || sig == 3 || sig == 16))
        {
            const int k = dtype * 3 + (sig == 1 ? 0 : sig == 3 ? 1 : 2);
            switch(k)
            {
#define ISAAC_SIG_CASE(dt, j, sg)                                                                                       \
    case dt * 3 + j:                                                                                                    \
        if(natural)                                                                                                     \
            hipLaunchKernelGGL((batch_march_kernel<dt, true, sg + kSigNatural>), dim3(grid), dim3(256), lds, s, B);     \
        else                                                                                                            \
            hipLaunchKernelGGL((batch_march_kernel<dt, true, sg>), dim3(grid), dim3(256), lds, s, B);                   \
        return hipGetLastError();
                ISAAC_SIG_CASE(0, 0, 1)
                ISAAC_SIG_CASE(0, 1, 3)
                ISAAC_SIG_CASE(0, 2, 16)
                ISAAC_SIG_CASE(1, 0, 1)
                ISAAC_SIG_CASE(1, 1, 3)
                ISAAC_SIG_CASE(1, 2, 16)
                ISAAC_SIG_CASE(2, 0, 1)
                ISAAC_SIG_CASE(2, 1, 3)
                ISAAC_SIG_CASE(2, 2, 16)
#undef ISAAC_SIG_CASE
            default: break;
            }
        }
        const int v = dtype * 2 + (linear ? 1 : 0);
        switch(v)
        {
        case 0: hipLaunchKernelGGL((batch_march_kernel<0, false>), dim3(grid), dim3(256), lds, s, B); break;
        case 1: hipLaunchKernelGGL((batch_march_kernel<0, true>), dim3(grid), dim3(256), lds, s, B); break;
        case 2: hipLaunchKernelGGL((batch_march_kernel<1, false>), dim3(grid), dim3(256), lds, s, B); break;
        case 3: hipLaunchKernelGGL((batch_march_kernel<1, true>), dim3(grid), dim3(256), lds, s, B); break;
        case 4: hipLaunchKernelGGL((batch_march_kernel<2, false>), dim3(grid), dim3(256), lds, s, B); break;
        default: hipLaunchKernelGGL((batch_march_kernel<2, true>), dim3(grid), dim3(256), lds, s, B); break;
        }
        return hipGetLastError();
    }

    hipError_t launch_batch_ssao(const FrameParams* frames, int nframes, int maxTiles, hipStream_t s)
    {
        if(nframes <= 0 || maxTiles <= 0)
            return hipSuccess;
        hipLaunchKernelGGL(batch_ssao_kernel, dim3(unsigned(maxTiles), unsigned(nframes)), dim3(256), 0, s, frames);
        return hipGetLastError();
    }

    hipError_t launch_batch_shade(const FrameParams* frames, int nframes, int maxTiles, hipStream_t s)
    {
        if(nframes <= 0 || maxTiles <= 0)
            return hipSuccess;
        hipLaunchKernelGGL(batch_shade_kernel, dim3(unsigned(maxTiles), unsigned(nframes)), dim3(256), 0, s, frames);
        return hipGetLastError();
    }

    // ------------------------------------------------------------------ launchers
    // the 4 voxels of quad q (x, y, z of its first voxel): every source's components,
    // f[s][k * D + c] for voxel k, component c (16-byte loads)
    template<int SIG>
    __device__ __attribute__((always_inline)) inline void cls_fetch(
        const ClassifyParams& P, int64_t q, float (&f)[sig_count(SIG)][16], int& x, int& y, int& z)
    {
        constexpr int N = sig_count(SIG);
        const uint32_t u = uint32_t(q) << 2;
        const uint32_t zq = fastdiv(u, P.divXY_mul, P.divXY_shift);
        const uint32_t rem = u - zq * uint32_t(P.X * P.Y);
        const uint32_t yq = fastdiv(rem, P.divX_mul, P.divX_shift);
        x = int(rem - yq * uint32_t(P.X));
        y = int(yq);
        z = int(zq);
#pragma unroll
        for(int s = 0; s < N; s++)
        {
            const int D = sig_dim(SIG, s);
            const ClassifySource& S = P.src[s];
            const float4* e = reinterpret_cast<const float4*>(
                S.data + (int64_t(x) + int64_t(y) * S.stride[1] + int64_t(z) * S.stride[2]) * D);
#pragma unroll
            for(int j = 0; j < D; j++)
            {
                const float4 w = e[j];
                f[s][4 * j + 0] = w.x;
                f[s][4 * j + 1] = w.y;
                f[s][4 * j + 2] = w.z;
                f[s][4 * j + 3] = w.w;
            }
        }
    }

    // classification of one fetched quad, its 4 texels stored with one 16-byte store per texture
    template<int SIG>
    __device__ __attribute__((always_inline)) inline void cls_emit(
        const ClassifyParams& P, const float4* lds_lut, const float (&f)[sig_count(SIG)][16], int x, int y, int z, int64_t q)
    {
        constexpr int N = sig_count(SIG);
        const int T = P.T;
        const uint32_t u = uint32_t(q) << 2;
        uint32_t vol[4], iso[4];
#pragma unroll
        for(int k = 0; k < 4; k++)
        {
            float vr = 0.f, vg = 0.f, vb = 0.f, va = 0.f;
            float ir = 0.f, ig = 0.f, ib = 0.f, ia = 0.f;
#pragma unroll
            for(int s = 0; s < N; s++)
            {
                const int D = sig_dim(SIG, s);
                const ClassifySource& S = P.src[s];
                const float c0 = f[s][k * D];
                const float c1 = D > 1 ? f[s][k * D + 1] : 0.f;
                const float c2 = D > 2 ? f[s][k * D + 2] : 0.f;
                // natural chains (identity, or one `length`) evaluated inline, in the
                // interpreter's order, instead of interpreting the chain per voxel
                const float tv = sig_natural(SIG) ? (D == 1 ? c0 : sqrtf(c0 * c0 + c1 * c1 + c2 * c2))
                                                  : apply_chain(S.chain, c0, c1, c2, 0.f, D);
                const float4 col = lds_lut[S.lutSlot * T + tf_index(tv, T)];
                const float ca = col.w;
                if(S.weight > 0.0f)
                {
                    float a = ca * S.weight;
                    vr = vr + col.x * a;
                    vg = vg + col.y * a;
                    vb = vb + col.z * a;
                    va = va + a;
                }
                if(S.iso > 0.0f)
                {
                    float a = div_by(ca, S.iso, S.invIso) * 0.5f;
                    if(ia < a)
                    {
                        ir = col.x;
                        ig = col.y;
                        ib = col.z;
                        ia = a;
                    }
                }
            }
            if(P.totalWeight != 0.0f)
            {
                vr = div_by(vr, P.totalWeight, P.invTotalWeight);
                vg = div_by(vg, P.totalWeight, P.invTotalWeight);
                vb = div_by(vb, P.totalWeight, P.invTotalWeight);
                va = div_by(va, P.totalWeight, P.invTotalWeight);
            }
            else
            {
                vr = vg = vb = va = 0.0f;
            }
            vol[k] = dither_b4(P.ditherMode, x + k, y, z, vr, vg, vb, va);
            const uint32_t q0 = unorm8(ir), q1 = unorm8(ig), q2 = unorm8(ib), q3 = unorm8(ia);
            iso[k] = q0 | (q1 << 8) | (q2 << 16) | (q3 << 24);
        }
        *reinterpret_cast<uint4*>(P.vol + u) = make_uint4(vol[0], vol[1], vol[2], vol[3]);
        if(P.iso)
        {
            *reinterpret_cast<uint4*>(P.iso + u) = make_uint4(iso[0], iso[1], iso[2], iso[3]);
            if(((iso[0] | iso[1] | iso[2] | iso[3]) >> 31) != 0u)
                mark_iso_cells(P, x, x + 3, y, z);
        }
    }

    // Classification compiled for the signature of its active sources (component
    // counts 1 or 3, at most two sources, all transfer functions in LDS, x-contiguous
    // sources with rows of a multiple of 4 voxels, no advection texture): each
    // thread classifies 4 consecutive voxels of a row per iteration (every source's
    // values in 16-byte loads; requesting the next quad's values before classifying the
    // current one held 32 more VGPRs, 90 against 71, and was 11 % slower than the
    // occupancy that frees) and stores the 4 texels with one 16-byte store per texture.  Same
    // arithmetic, in the same order, as classify_kernel.  Workgroups of 512 threads:
    // eight waves share one LDS copy of the transfer functions, which halves the
    // staging reads against 256-thread workgroups and lets 8 waves per SIMD be
    // resident with two 1024-entry functions (32 KB per workgroup).
    template<int SIG>
    __global__ __launch_bounds__(512) void classify_sig_kernel(const ClassifyParams P)
    {
        extern __shared__ float4 lds_lut[];
        for(int i = threadIdx.x; i < P.nLut * P.T; i += blockDim.x)
            lds_lut[i] = P.luts[i];
        __syncthreads();
        constexpr int N = sig_count(SIG);
        const int64_t nq = P.nvox >> 2;
        const int64_t stride = int64_t(gridDim.x) * blockDim.x;
        int64_t q = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
        if(q >= nq)
            return;
        for(; q < nq; q += stride)
        {
            float f[N][16];
            int x, y, z;
            cls_fetch<SIG>(P, q, f, x, y, z);
            cls_emit<SIG>(P, lds_lut, f, x, y, z, q);
        }
    }


    // signature of the active sources for classify_sig_kernel, 0 when the generic kernel applies;
    // Pc receives the active sources in slot order
    int classify_signature(const ClassifyParams& P, ClassifyParams& Pc)
    {
        if(P.X % 4 != 0 || ((reinterpret_cast<uintptr_t>(P.vol) | reinterpret_cast<uintptr_t>(P.iso)) & 15u) != 0)
            return 0;
        Pc = P;
        int n = 0, sig = 0, w = 1;
        for(int s = 0; s < P.nsrc; s++)
        {
            const ClassifySource& S = P.src[s];
            if(!S.active)
                continue;
            if(n == 2 || (S.dim != 1 && S.dim != 3) || S.adv || S.lutSlot >= P.nLut || S.stride[0] != 1 || S.stride[1] % 4 != 0
               || S.stride[2] % 4 != 0 || (reinterpret_cast<uintptr_t>(S.data) & 15u) != 0)
                return 0;
            Pc.src[n++] = S;
            sig += S.dim * w;
            w *= 5;
        }
        Pc.nsrc = n;
        return n > 0 ? sig : 0;
    }

    hipError_t launch_classify(const ClassifyParams& P, hipStream_t s)
    {
        if(P.nvox <= 0)
            return hipSuccess;
        const size_t lds = size_t(P.nLut) * P.T * sizeof(float4);
        ClassifyParams Pc;
        const int sig = classify_signature(P, Pc);
        if(sig)
        {
            int64_t blocks = (P.nvox / 4 + 511) / 512;
            if(blocks > 2048)
                blocks = 2048;
            const dim3 grid = dim3(unsigned(blocks)), block(512);
            bool natural = true;
            for(int k = 0; k < Pc.nsrc; k++)
                natural = natural && natural_chain(Pc.src[k].chain, Pc.src[k].dim);
#define ISAAC_CLS_SIG(sg)                                                                                            \
    case sg:                                                                                                         \
        if(natural)                                                                                                  \
            hipLaunchKernelGGL((classify_sig_kernel<sg + kSigNatural>), grid, block, lds, s, Pc);                     \
        else                                                                                                         \
            hipLaunchKernelGGL((classify_sig_kernel<sg>), grid, block, lds, s, Pc);                                   \
        return hipGetLastError();
            switch(sig)
            {
                ISAAC_CLS_SIG(1)
                ISAAC_CLS_SIG(3)
                ISAAC_CLS_SIG(6)
                ISAAC_CLS_SIG(8)
                ISAAC_CLS_SIG(16)
                ISAAC_CLS_SIG(18)
            default: break;
            }
#undef ISAAC_CLS_SIG
        }
        int64_t blocks = (P.nvox + 255) / 256;
        if(blocks > 4096)
            blocks = 4096;
        hipLaunchKernelGGL(classify_kernel, dim3(unsigned(blocks)), dim3(256), lds, s, P);
        return hipGetLastError();
    }

    // ------------------------------------------------------------------ field-source advection
    // halton (lib/isaac/isaac_helper.hpp:57-69)
    __device__ inline float halton(uint32_t index, uint32_t base)
    {
        float result = 0.0f, f = 1.0f;
        while(index > 0)
        {
            f = f / float(base);
            result = result + f * float(index % base);
            index = index / base;
        }
        return result;
    }

    // HaltonSeedingKernel (lib/isaac/isaac_common_kernel.hpp:334-348): point i = 1..count
    // at (halton(i,3), halton(i,5), halton(i,7)) * size, truncated, set to 1 (one
    // thread per point; points that land on one voxel all store 1)
    __global__ __launch_bounds__(256) void halton_seed_kernel(float* noise, int X, int Y, int Z, uint32_t count)
    {
        for(uint32_t i = blockIdx.x * blockDim.x + threadIdx.x + 1; i <= count; i += gridDim.x * blockDim.x)
        {
            const int x = int(float(X) * halton(i, 3)), y = int(float(Y) * halton(i, 5)), z = int(float(Z) * halton(i, 7));
            noise[(size_t(z) * Y + y) * X + x] = 1.0f;
        }
    }

    // Sampler<LINEAR, REPEAT> on a guard-less float texture (lib/isaac/isaac_texture.hpp:182-259)
    __device__ inline int wrap(int c, int n)
    {
        return (n + (c % n)) % n;
    }

    __device__ inline float sample_repeat(const float* t, int X, int Y, int Z, float px, float py, float pz)
    {
        const float cx = px - 0.5f, cy = py - 0.5f, cz = pz - 0.5f;
        const float flx = floorf(cx), fly = floorf(cy), flz = floorf(cz);
        const float fx = cx - flx, fy = cy - fly, fz = cz - flz;
        const int x0 = int(flx), y0 = int(fly), z0 = int(flz);
        auto v = [&](int dx, int dy, int dz) {
            return t[(size_t(wrap(z0 + dz, Z)) * Y + wrap(y0 + dy, Y)) * X + wrap(x0 + dx, X)];
        };
        const float oz = 1.0f - fz, oy = 1.0f - fy, ox = 1.0f - fx;
        const float a0 = v(0, 0, 0) * oz + v(0, 0, 1) * fz, a1 = v(0, 1, 0) * oz + v(0, 1, 1) * fz;
        const float A = a0 * oy + a1 * fy;
        const float b0 = v(1, 0, 0) * oz + v(1, 0, 1) * fz, b1 = v(1, 1, 0) * oz + v(1, 1, 1) * fz;
        const float B = b0 * oy + b1 * fy;
        return A * ox + B * fx;
    }

    // GaussBlur7Kernel (lib/isaac/isaac_common_kernel.hpp:381-411) along one axis
    // sample position coord + mask * k / scale, as the reference evaluates it
    __global__ __launch_bounds__(256) void gauss7_kernel(const float* src, float* dst, int X, int Y, int Z, float3 mask, float3 scale)
    {
        const float w[4] = {64.0f, 40.5f, 10.0f, 1.0f};
        const uint32_t n = uint32_t(X) * uint32_t(Y) * uint32_t(Z);
        for(uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        {
            const int x = int(i % uint32_t(X)), y = int((i / uint32_t(X)) % uint32_t(Y)), z = int(i / (uint32_t(X) * uint32_t(Y)));
            float r = 0.0f;
            for(int k = -3; k < 4; k++)
            {
                const float px = float(x) + mask.x * float(k) / scale.x, py = float(y) + mask.y * float(k) / scale.y,
                            pz = float(z) + mask.z * float(k) / scale.z;
                r = r + sample_repeat(src, X, Y, Z, px, py, pz) * w[k < 0 ? -k : k];
            }
            dst[i] = r / 167.0f;
        }
    }

    // MultiplyClampKernel (lib/isaac/isaac_common_kernel.hpp:413-429)
    __global__ __launch_bounds__(256) void multiply_clamp_kernel(const float* src, float* dst, int64_t n, float value, float lo, float hi)
    {
        for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
            dst[i] = fminf(fmaxf(src[i] * value, lo), hi);
    }

    hipError_t launch_noise(float* noise, float* tmp, int X, int Y, int Z, const float scale[3], uint32_t seedPoints, hipStream_t s)
    {
        const int64_t n = int64_t(X) * Y * Z;
        if(n <= 0)
            return hipSuccess;
        if(n >= (int64_t(1) << 32))
            return hipErrorInvalidValue;
        const unsigned grid = unsigned(std::min<int64_t>((n + 255) / 256, 8192));
        const float3 sc = make_float3(scale[0], scale[1], scale[2]);
        hipError_t e = launch_fill_u32(reinterpret_cast<uint32_t*>(noise), 0u, size_t(n), s);
        if(e != hipSuccess)
            return e;
        if(seedPoints > 0)
            hipLaunchKernelGGL(halton_seed_kernel, dim3(std::min<uint32_t>((seedPoints + 255) / 256, 4096)), dim3(256), 0, s,
                               noise, X, Y, Z, seedPoints);
        // three separable passes noise -> tmp (x) -> noise (y) -> tmp (z), then noise = clamp(tmp * 30, 0, 1)
        hipLaunchKernelGGL(gauss7_kernel, dim3(grid), dim3(256), 0, s, (const float*) noise, tmp, X, Y, Z, make_float3(1.0f, 0.0f, 0.0f), sc);
        hipLaunchKernelGGL(gauss7_kernel, dim3(grid), dim3(256), 0, s, (const float*) tmp, noise, X, Y, Z, make_float3(0.0f, 1.0f, 0.0f), sc);
        hipLaunchKernelGGL(gauss7_kernel, dim3(grid), dim3(256), 0, s, (const float*) noise, tmp, X, Y, Z, make_float3(0.0f, 0.0f, 1.0f), sc);
        hipLaunchKernelGGL(multiply_clamp_kernel, dim3(grid), dim3(256), 0, s, (const float*) tmp, noise, n, 30.0f, 0.0f, 1.0f);
        return hipGetLastError();
    }

    // Sampler<LINEAR, VALUE> on a byte texture whose guard (and beyond) reads 0
    __device__ inline float sample_bytes_zero(const uint8_t* t, int X, int Y, int Z, float px, float py, float pz)
    {
        const float cx = px - 0.5f, cy = py - 0.5f, cz = pz - 0.5f;
        const float flx = floorf(cx), fly = floorf(cy), flz = floorf(cz);
        const float fx = cx - flx, fy = cy - fly, fz = cz - flz;
        const int x0 = int(flx), y0 = int(fly), z0 = int(flz);
        auto v = [&](int dx, int dy, int dz) {
            const int x = x0 + dx, y = y0 + dy, z = z0 + dz;
            if(x < 0 || y < 0 || z < 0 || x >= X || y >= Y || z >= Z)
                return 0.0f;
            return float(t[(size_t(z) * Y + y) * X + x]);
        };
        const float oz = 1.0f - fz, oy = 1.0f - fy, ox = 1.0f - fx;
        const float a0 = v(0, 0, 0) * oz + v(0, 0, 1) * fz, a1 = v(0, 1, 0) * oz + v(0, 1, 1) * fz;
        const float A = a0 * oy + a1 * fy;
        const float b0 = v(1, 0, 0) * oz + v(1, 0, 1) * fz, b1 = v(1, 1, 0) * oz + v(1, 1, 1) * fz;
        const float B = b0 * oy + b1 * fy;
        return A * ox + B * fx;
    }

    // GenerateAdvectionTextureKernel (lib/isaac/isaac_common_kernel.hpp:500-550): the
    // unit field direction moves the history back by stepSize / scale; the noise seeds
    // where the seeding window is open; blended value dithered with the 16^3 mask
    __global__ __launch_bounds__(256) void advect_kernel(const AdvectParams P)
    {
        const uint32_t n = uint32_t(P.X) * uint32_t(P.Y) * uint32_t(P.Z);
        for(uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        {
            const int x = int(i % uint32_t(P.X)), y = int((i / uint32_t(P.X)) % uint32_t(P.Y)), z = int(i / (uint32_t(P.X) * uint32_t(P.Y)));
            const float* e = P.field + (int64_t(x) * P.stride[0] + int64_t(y) * P.stride[1] + int64_t(z) * P.stride[2]) * 3;
            float vx = e[0], vy = e[1], vz = e[2];
            float len = sqrtf((vx * vx + vy * vy) + vz * vz);
            len = (len < FLT_MIN) ? FLT_MIN : len;
            vx = vx / len;
            vy = vy / len;
            vz = vz / len;
            const float ox = vx * P.stepSize / P.scale[0], oy = vy * P.stepSize / P.scale[1], oz = vz * P.stepSize / P.scale[2];
            const float px = (float(x) + 0.5f) - ox, py = (float(y) + 0.5f) - oy, pz = (float(z) + 0.5f) - oz;
            const float history = sample_bytes_zero(P.history, P.X, P.Y, P.Z, px, py, pz) / 255.0f;
            const float noise = P.seeding ? P.noise[i] : 0.0f;
            const float v = noise + history * P.historyWeight * (1.0f - noise);
            P.out[i] = uint8_t(dither_b4(5, x, y, z, v, 0.f, 0.f, 0.f) & 0xffu);
        }
    }

    hipError_t launch_advect(const AdvectParams& P, hipStream_t s)
    {
        const int64_t n = int64_t(P.X) * P.Y * P.Z;
        if(n <= 0)
            return hipSuccess;
        if(n >= (int64_t(1) << 32))
            return hipErrorInvalidValue;
        hipLaunchKernelGGL(advect_kernel, dim3(unsigned(std::min<int64_t>((n + 255) / 256, 8192))), dim3(256), 0, s, P);
        return hipGetLastError();
    }

    // ------------------------------------------------------------------ min/max request
    // MinMaxKernel (lib/isaac/isaac_min_max_kernel.hpp:22-57) as a grid-stride
    // reduction over the voxels; the visiting-order key of voxel (x, y, z) is
    // (x + y*X) * Z + z + 1 (columns in the host loop's order, z inside a column).
    __global__ __launch_bounds__(256) void min_max_volume_kernel(const MinMaxVolumeParams P, MinMaxPartial* partials)
    {
        MinMaxPartial a{FLT_MAX, -FLT_MAX, 0, 0};
        const int64_t stride = int64_t(gridDim.x) * blockDim.x;
        for(int64_t idx = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; idx < P.nvox; idx += stride)
        {
            const uint32_t u = (uint32_t) idx;
            const uint32_t zq = fastdiv(u, P.divXY_mul, P.divXY_shift);
            const uint32_t rem = u - zq * uint32_t(P.X * P.Y);
            const uint32_t yq = fastdiv(rem, P.divX_mul, P.divX_shift);
            const int x = int(rem - yq * uint32_t(P.X)), y = int(yq), z = int(zq);
            const float* e = P.data + (int64_t(x) * P.stride[0] + int64_t(y) * P.stride[1] + int64_t(z) * P.stride[2]) * P.dim;
            float v = e[0];
            if(P.applyChain)
                v = apply_chain(P.chain, e[0], P.dim > 1 ? e[1] : 0.f, P.dim > 2 ? e[2] : 0.f, P.dim > 3 ? e[3] : 0.f, P.dim);
            const uint64_t key = (uint64_t(x) + uint64_t(y) * uint64_t(P.X)) * uint64_t(P.Z) + uint64_t(z) + 1;
            mm_take_min(a.vmin, a.kmin, v, key);
            mm_take_max(a.vmax, a.kmax, v, key);
        }
        a = mm_block_reduce(a);
        if(threadIdx.x == 0)
            partials[blockIdx.x] = a;
    }

    __global__ __launch_bounds__(256) void min_max_final_kernel(const MinMaxPartial* partials, int count, float2* out)
    {
        MinMaxPartial a{FLT_MAX, -FLT_MAX, 0, 0};
        for(int i = threadIdx.x; i < count; i += blockDim.x)
        {
            mm_take_min(a.vmin, a.kmin, partials[i].vmin, partials[i].kmin);
            mm_take_max(a.vmax, a.kmax, partials[i].vmax, partials[i].kmax);
        }
        a = mm_block_reduce(a);
        if(threadIdx.x == 0)
            *out = make_float2(a.vmin, a.vmax);
    }

    hipError_t launch_min_max_final(const MinMaxPartial* partials, int count, float2* out, hipStream_t s)
    {
        hipLaunchKernelGGL(min_max_final_kernel, dim3(1), dim3(256), 0, s, partials, count, out);
        return hipGetLastError();
    }

    hipError_t launch_min_max_volume(const MinMaxVolumeParams& P, MinMaxPartial* partials, float2* out, hipStream_t s)
    {
        if(P.nvox <= 0 || P.nvox >= (int64_t(1) << 32))
            return hipErrorInvalidValue;
        const int groups = int(std::min<int64_t>((P.nvox + 255) / 256, kMinMaxGroups));
        hipLaunchKernelGGL(min_max_volume_kernel, dim3(groups), dim3(256), 0, s, P, partials);
        hipError_t e = hipGetLastError();
        return e != hipSuccess ? e : launch_min_max_final(partials, groups, out, s);
    }

    hipError_t launch_persistent_copy(
        const float* src,
        const int64_t stride[3],
        int dim,
        const ChainDesc& chain,
        int gX,
        int gY,
        int gZ,
        int guard,
        float* dst,
        hipStream_t s)
    {
        int64_t n = int64_t(gX) * gY * gZ;
        int64_t blocks = (n + 255) / 256;
        if(blocks > 4096)
            blocks = 4096;
        if(blocks < 1)
            return hipSuccess;
        hipLaunchKernelGGL(
            persistent_copy_kernel, dim3(unsigned(blocks)), dim3(256), 0, s, src, stride[0], stride[1], stride[2], dim,
            chain, gX, gY, gZ, guard, dst);
        return hipGetLastError();
    }

    // The combined texture with both texels of a voxel side by side, for readers of the
    // textures (the march reads the two separately); iso == nullptr: iso texels of 0.
    __global__ __launch_bounds__(256) void interleave_kernel(const uint32_t* __restrict__ vol, const uint32_t* __restrict__ iso,
                                                             uint2* __restrict__ out, int64_t n)
    {
        for(int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += int64_t(gridDim.x) * blockDim.x)
            out[i] = make_uint2(vol[i], iso ? iso[i] : 0u);
    }

    hipError_t launch_interleave(const uint32_t* vol, const uint32_t* iso, uint2* out, int64_t n, hipStream_t s)
    {
        if(n <= 0)
            return hipSuccess;
        const int64_t blocks = std::min<int64_t>((n + 255) / 256, 4096);
        hipLaunchKernelGGL(interleave_kernel, dim3(unsigned(blocks)), dim3(256), 0, s, vol, iso, out, n);
        return hipGetLastError();
    }

    bool ssao_shades(const FrameParams& F)
    {
        // render modes 0, 1 and 3 leave the depth buffer as the march wrote it
        return F.aoEnabled && (F.renderMode == 0 || F.renderMode == 1 || F.renderMode == 3);
    }

    hipError_t launch_ssao(const FrameParams& F, hipStream_t s, bool shade)
    {
        const unsigned bw = unsigned(F.vx1 - F.vx0 + kSsaoBW - 1) / kSsaoBW;
        const unsigned bh = unsigned(F.vy1 - F.vy0 + kSsaoBH - 1) / kSsaoBH;
        if(bw * bh == 0)
            return hipSuccess;
        if(shade)
            hipLaunchKernelGGL(ssao_tiled_kernel<true>, dim3(bw * bh), dim3(256), 0, s, F);
        else
            hipLaunchKernelGGL(ssao_tiled_kernel<false>, dim3(bw * bh), dim3(256), 0, s, F);
        return hipGetLastError();
    }

    hipError_t launch_shade(const FrameParams& F, hipStream_t s)
    {
        const unsigned nb = unsigned(F.tilesX) * unsigned(F.tilesY);
        if(nb == 0)
            return hipSuccess;
        hipLaunchKernelGGL(shade_kernel, dim3(nb), dim3(256), 0, s, F);
        return hipGetLastError();
    }
} // namespace isaac_hip
