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
