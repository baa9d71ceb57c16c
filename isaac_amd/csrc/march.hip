// The combined form's march on gfx950: clear, particles, iso-surface and volume of a
// pixel in one traversal of its ray
//   march_kernel           ClearBufferKernel + ParticleRenderKernel + CombinedIsoRenderKernel +
//                          the march of CombinedVolumeRenderKernel, fused per pixel
//                          lib/isaac/isaac_common_kernel.hpp:195-217, lib/isaac/isaac_particle_kernel.hpp:117-260,
//                          lib/isaac/isaac_iso_kernel.hpp:25-128, lib/isaac/isaac_volume_kernel.hpp:23-82
#include "render_device.hpp"

namespace isaac_hip
{
    // ------------------------------------------------------------------ texture sampling
    // Texels: the combined volume and iso RGBA8 are two textures of one layout (x fastest,
    // one word per voxel, one word of padding at the end), so the march's gathers move 4 bytes
    // per corner and read the iso texture only where a cell of it can hold a surface.
    // Two adjacent texels come from one 8-byte load (4-byte aligned).
    typedef uint32_t TexPair __attribute__((ext_vector_type(2), aligned(4)));

    // The 8 taps of one sample position of the iso texture (or the single NEAREST tap): tap k
    // holds voxel (x0 + (k>>2), y0 + ((k>>1)&1), z0 + (k&1)), clamped.  Sampler<LINEAR|NEAREST,
    // CLAMP> addressing (lib/isaac/isaac_texture.hpp:182-259); every coordinate is clamped into
    // the texture, so a fetch at any position is in bounds.
    struct Taps
    {
        uint32_t t[8];
        float fx, fy, fz;
    };

    template<bool LINEAR>
    __device__ inline void fetch_taps(const FrameParams& F, float px, float py, float pz, Taps& T)
    {
        const uint32_t* __restrict__ tex = F.iso;
        const int X = F.X, Y = F.Y, Z = F.Z;
        auto index = [&](uint32_t x, uint32_t y, uint32_t z) { return x + uint32_t(X) * (y + uint32_t(Y) * z); };
        if(!LINEAR)
        {
            const uint32_t x = iclamp(int(px), 0, X - 1), y = iclamp(int(py), 0, Y - 1), z = iclamp(int(pz), 0, Z - 1);
            T.t[0] = tex[index(x, y, z)];
            T.fx = T.fy = T.fz = 0.0f;
            return;
        }
        const float cx = px - 0.5f, cy = py - 0.5f, cz = pz - 0.5f;
        const float flx = floorf(cx), fly = floorf(cy), flz = floorf(cz);
        T.fx = cx - flx;
        T.fy = cy - fly;
        T.fz = cz - flz;
        const int bx = int(flx), by = int(fly), bz = int(flz);
        const uint32_t x0 = iclamp(bx, 0, X - 1), x1 = iclamp(bx + 1, 0, X - 1);
        const uint32_t y0 = iclamp(by, 0, Y - 1), y1 = iclamp(by + 1, 0, Y - 1);
        const uint32_t z0 = iclamp(bz, 0, Z - 1), z1 = iclamp(bz + 1, 0, Z - 1);
        // texels x0 and x0+1 are adjacent: one load per (y, z) row; at the x edge (x1 == x0)
        // the second texel (the next row's first, or the padding) is replaced by the first
        const TexPair p00 = *reinterpret_cast<const TexPair*>(tex + index(x0, y0, z0));
        const TexPair p01 = *reinterpret_cast<const TexPair*>(tex + index(x0, y0, z1));
        const TexPair p10 = *reinterpret_cast<const TexPair*>(tex + index(x0, y1, z0));
        const TexPair p11 = *reinterpret_cast<const TexPair*>(tex + index(x0, y1, z1));
        const bool dup = x1 == x0;
        T.t[0] = p00.x;
        T.t[1] = p01.x;
        T.t[2] = p10.x;
        T.t[3] = p11.x;
        T.t[4] = dup ? p00.x : p00.y;
        T.t[5] = dup ? p01.x : p01.y;
        T.t[6] = dup ? p10.x : p10.y;
        T.t[7] = dup ? p11.x : p11.y;
    }

    // one normalised channel: trilinear of the bytes (z innermost, x outermost,
    // lib/isaac/isaac_helper.hpp:124-144), then / 255
    template<bool LINEAR>
    __device__ inline float channel(const Taps& T, int sh)
    {
        auto d = [&](int k) { return float((T.t[k] >> sh) & 0xffu); };
        if(!LINEAR)
            return div255(d(0));
        const float oz = 1.0f - T.fz, oy = 1.0f - T.fy, ox = 1.0f - T.fx;
        const float a0 = d(0) * oz + d(1) * T.fz, a1 = d(2) * oz + d(3) * T.fz;
        const float A = a0 * oy + a1 * T.fy;
        const float b0 = d(4) * oz + d(5) * T.fz, b1 = d(6) * oz + d(7) * T.fz;
        const float B = b0 * oy + b1 * T.fy;
        return div255(A * ox + B * T.fx);
    }

    template<bool LINEAR>
    __device__ inline float iso_alpha_at(const FrameParams& F, float px, float py, float pz)
    {
        Taps T;
        fetch_taps<LINEAR>(F, px, py, pz, T);
        return channel<LINEAR>(T, 24);
    }

    // ------------------------------------------------------------------ march sampling
    // The march's per-step samples weigh the eight texels once per position: each
    // channel is sum_k byte_k * w_k (one multiply and seven fmas) with the corner
    // weights w_k = wx * wy * wz, instead of seven lerps per channel, and at the x
    // edge (both x taps on texel x0, CLAMP) the first texel takes weight 1 instead of
    // the texels being swapped.  In exact arithmetic this is the reference's trilinear
    // (lib/isaac/isaac_helper.hpp:124-144); in binary32 the result differs from its
    // nested lerps by rounding only.
    //
    // Where a sample lies: the byte (OFF32) or texel offset of its row pairs and the fractions.
    // A row pair is texels x0 and x0 + 1; rows are (y0, z0), (y0, z1), (y1, z0), (y1, z1).
    struct Place
    {
        uint32_t o00, o01, o10, o11;
        float fx, fy, fz;
    };

    // The corner sums take a texel's bytes as binary32 denormals, without conversions: the byte
    // in bits 0..7 of a word is b * 2^-149 as a float, in bits 8..15 b * 2^-141, in bits 16..23
    // b * 2^-133 (the byte in bits 24..31 is shifted down).  One mask and one fma per byte, both
    // at twice the rate of v_cvt_f32_ubyte (and of v_fma_mix_f32, which would take them as
    // binary16).  The corner weights carry a factor of 2^100, so that the products are normal
    // numbers; powers of two change no rounding, and the scales below take them out again.
    constexpr float kWeightScale = 0x1p100f; // on every corner weight
    constexpr float kByteScale = 0x1p49f; // a sum of bytes in bits 0..7: 2^(149 - 100)

    struct Weights
    {
        float w[8]; // k = 4 x + 2 y + z (x outermost, as the reference's lerps nest), times kWeightScale
    };

    __device__ inline Weights corner_weights(float fx, float fy, float fz)
    {
        Weights W;
        const float sz = fz * kWeightScale;
        const float ox = 1.0f - fx, oy = 1.0f - fy, oz = kWeightScale - sz;
        const float w00 = oy * oz, w01 = oy * sz, w10 = fy * oz, w11 = fy * sz;
        W.w[0] = ox * w00;
        W.w[1] = ox * w01;
        W.w[2] = ox * w10;
        W.w[3] = ox * w11;
        W.w[4] = fx * w00;
        W.w[5] = fx * w01;
        W.w[6] = fx * w10;
        W.w[7] = fx * w11;
        return W;
    }

    // any position c (for LINEAR the position minus 0.5, the texel centres' offset; for NEAREST
    // the position itself), clamped into the texture
    template<bool LINEAR>
    __device__ inline Place place_of(const FrameParams& F, uint32_t XY, float cx, float cy, float cz)
    {
        Place p;
        const int X = F.X, Y = F.Y, Z = F.Z;
        if(!LINEAR)
        {
            const uint32_t x = iclamp(int(cx), 0, X - 1), y = iclamp(int(cy), 0, Y - 1), z = iclamp(int(cz), 0, Z - 1);
            p.o00 = p.o01 = p.o10 = p.o11 = x + uint32_t(X) * y + XY * z;
            p.fx = p.fy = p.fz = 0.0f;
            return p;
        }
        const float flx = floorf(cx), fly = floorf(cy), flz = floorf(cz);
        const int bx = int(flx), by = int(fly), bz = int(flz);
        // taps x0 and x0 + 1 come from one load; where both are x0 (bx < 0 or bx >= X - 1)
        // the second gets weight 0
        const bool xin = uint32_t(bx) < uint32_t(X - 1);
        p.fx = xin ? cx - flx : 0.0f;
        p.fy = cy - fly;
        p.fz = cz - flz;
        const uint32_t x0 = iclamp(bx, 0, X - 1), y0 = iclamp(by, 0, Y - 1), z0 = iclamp(bz, 0, Z - 1);
        // rows y + 1 and z + 1: the next row / slice, or the same one at a clamped edge
        const uint32_t dy = uint32_t(by) < uint32_t(Y - 1) ? uint32_t(X) : 0u;
        const uint32_t dz = uint32_t(bz) < uint32_t(Z - 1) ? XY : 0u;
        p.o00 = x0 + __umul24(y0, uint32_t(X)) + z0 * XY;
        p.o01 = p.o00 + dz;
        p.o10 = p.o00 + dy;
        p.o11 = p.o10 + dz;
        return p;
    }

    // the 8 texels of a place (one for NEAREST).  OFF32: the texture spans < 4 GiB, so the loads
    // take a 32-bit byte offset from its (uniform) base instead of a 64-bit address per lane.
    template<bool LINEAR, bool OFF32>
    __device__ inline void fetch_place(const uint32_t* __restrict__ tex, const Place& p, uint32_t t[8])
    {
        if(!LINEAR)
        {
            t[0] = tex[p.o00];
            return;
        }
        auto pair = [&](uint32_t o) -> TexPair
        {
            if constexpr(OFF32)
                return *reinterpret_cast<const TexPair*>(reinterpret_cast<const char*>(tex) + (o << 2));
            else
                return *reinterpret_cast<const TexPair*>(tex + o);
        };
        const TexPair p00 = pair(p.o00), p01 = pair(p.o01), p10 = pair(p.o10), p11 = pair(p.o11);
        t[0] = p00.x;
        t[1] = p01.x;
        t[2] = p10.x;
        t[3] = p11.x;
        t[4] = p00.y;
        t[5] = p01.y;
        t[6] = p10.y;
        t[7] = p11.y;
    }

    // the iso alpha of a sample in byte units (0..255)
    template<bool LINEAR>
    __device__ inline float iso_sum(const uint32_t t[8], const Weights& W)
    {
        if(!LINEAR)
            return float(t[0] >> 24);
        float v = __uint_as_float(t[0] >> 24) * W.w[0];
#pragma unroll
        for(int k = 1; k < 8; k++)
            v = __builtin_fmaf(__uint_as_float(t[k] >> 24), W.w[k], v);
        return v * kByteScale;
    }

    // The volume RGBA of a sample, each channel the corner sum of its bytes: r and a in units of
    // 1 / kByteScale, g of 2^8 / kByteScale and b of 2^16 / kByteScale (bytes for NEAREST).
    template<bool LINEAR>
    __device__ inline float4 vol_sums(const uint32_t t[8], const Weights& W)
    {
        if(!LINEAR)
            return make_float4(float(t[0] & 0xffu), float((t[0] >> 8) & 0xffu), float((t[0] >> 16) & 0xffu), float(t[0] >> 24));
        float4 v = make_float4(__uint_as_float(t[0] & 0xffu) * W.w[0], __uint_as_float(t[0] & 0xff00u) * W.w[0],
                               __uint_as_float(t[0] & 0xff0000u) * W.w[0], __uint_as_float(t[0] >> 24) * W.w[0]);
#pragma unroll
        for(int k = 1; k < 8; k++)
        {
            v.x = __builtin_fmaf(__uint_as_float(t[k] & 0xffu), W.w[k], v.x);
            v.y = __builtin_fmaf(__uint_as_float(t[k] & 0xff00u), W.w[k], v.y);
            v.z = __builtin_fmaf(__uint_as_float(t[k] & 0xff0000u), W.w[k], v.z);
            v.w = __builtin_fmaf(__uint_as_float(t[k] >> 24), W.w[k], v.w);
        }
        return v;
    }

    // ------------------------------------------------------------------ fused march
    // One pass per pixel: clear, particle DDA, then ONE traversal of the ray that
    // serves both the iso march (CombinedIsoRenderKernel) and the volume march
    // (CombinedVolumeRenderKernel).  Both reference kernels sample the same
    // positions startU + stepVec*i from the same startSteps; the volume stops at
    // floor(min(clipEnd, depth)/step) where depth is the particle/iso depth, so
    // the iso decision at step i is made before the volume consumes step i.  The
    // premultiplied volume colour goes to volColor and is blended over the shaded
    // solid colour by shade_kernel after SSAO, which keeps the reference's pass
    // order (particles, iso, SSAO, shading, volume) for every pixel.

    // the accumulated volume colour of a ray; for the trilinear sampler g carries a factor of
    // 2^8 and b of 2^16 (vol_sums), taken out at the end of the ray
    struct VolAcc
    {
        float r, g, b, a;
    };

    __device__ inline void composite(VolAcc& c, const float4 v, float vscale)
    {
        const float w = (1.0f - c.a) * vscale;
        c.r = c.r + w * v.x;
        c.g = c.g + w * v.y;
        c.b = c.b + w * v.z;
        c.a = c.a + w * v.w;
    }

    // steps a ray takes in a box: sample i lies at c + v * i (one fma per axis)
    struct StepLine
    {
        F3 c, v;
        __device__ inline F3 at(float k) const
        {
            return f3(__builtin_fmaf(v.x, k, c.x), __builtin_fmaf(v.y, k, c.y), __builtin_fmaf(v.z, k, c.z));
        }
    };

    // The steps i0..i1 of the line whose samples lie inside [0, X-1) x [0, Y-1) x [0, Z-1), i.e.
    // whose eight corners need no clamp.  The estimate from the slabs is checked at both ends
    // with the march's own arithmetic; an fma is monotonic in i, so every step between them is
    // inside too.  i1 < i0 where there are none.
    __device__ inline void interior_steps(const FrameParams& F, const StepLine& L, int first, int last, int& i0, int& i1)
    {
        float lo = float(first), hi = float(last);
        auto slab = [&](float c, float v, int n)
        {
            // (an axis without movement divides by 0: the bounds are infinite, or NaN, which fmin and
            // fmax drop; the check of the ends covers it)
            const float a = (0.0f - c) / v, b = (float(n - 1) - c) / v;
            lo = fmaxf(lo, fminf(a, b));
            hi = fminf(hi, fmaxf(a, b));
        };
        slab(L.c.x, L.v.x, F.X);
        slab(L.c.y, L.v.y, F.Y);
        slab(L.c.z, L.v.z, F.Z);
        i0 = 0;
        i1 = -1;
        if(!(lo <= hi)) // NaN bounds too
            return;
        const int j0 = max(first, int(ceilf(lo))), j1 = min(last, int(floorf(hi)));
        auto inside = [&](int i)
        {
            const F3 p = L.at(float(i));
            return p.x >= 0.0f && p.x < float(F.X - 1) && p.y >= 0.0f && p.y < float(F.Y - 1) && p.z >= 0.0f
                && p.z < float(F.Z - 1);
        };
        // the slab bounds may be off by a rounding: one step in at each end is enough
        const int k0 = inside(j0) ? j0 : j0 + 1, k1 = inside(j1) ? j1 : j1 - 1;
        if(k0 <= k1 && inside(k0) && inside(k1))
        {
            i0 = k0;
            i1 = k1;
        }
    }

    // The steps between which the line can read an iso alpha byte >= 128: the ray walks through
    // the iso cells (8^3 base texels each, marked by the classification) and notes the first step
    // in a marked one and the last.  from > to where there is none.  Walked for the whole ray before
    // the march, when all lanes of a wave walk together: lanes leave cells at different steps, so a
    // walk from cell to cell inside the march would make each lane wait for all the others' walks.
    //
    // A ray that starts in LEAD marked cells in a row is in data whose surface is everywhere
    // (noise about the threshold, a box opaque from its face on), and has most likely met it before
    // the walk would end: it is not walked on, every step is tested.  Measured on MI355X at 960x540,
    // march of 192^3 voxels all above the threshold, trilinear / nearest: 38 / 36 us walked to the end,
    // 31 / 20 us with 16 and 3 cells (the test at every step that the walk replaced: 24 / 17); uniform noise
    // about the threshold 112 / 53 -> 108 / 38 us (101 / 36).  Fewer cells would gain the trilinear march
    // more there (8: 28 us, 3: 25 us), but rays that run along a surface from a clipping plane start in as
    // many and test in vain: of eleven 256^3 production frames one goes from 604 to 657 us with 8, others
    // from 3 on, none with 12 or 16; anywhere along the ray 4 in a row take all of them from 610 to
    // 659 us.  A test of the nearest march is one load beside another, and takes its frames from 620 to
    // 622 us at most.  The count is kept where a cell is marked only: every instruction on the path of the
    // others, or a loop of its own for the first cells, costs frames with a surface 1-3 %.
    template<int LEAD>
    __device__ inline void iso_steps(const FrameParams& F, const StepLine& L, int first, int last, int& from, int& to)
    {
        const F3 inv = f3(1.0f / L.v.x, 1.0f / L.v.y, 1.0f / L.v.z);
        const float lastF = float(last);
        from = 0x7fffffff;
        to = first - 1;
        int lead = 0; // marked cells in a row from the ray's start (below 0 behind a gap)
        for(float k = float(first); k <= lastF;)
        {
            const F3 p = L.at(k);
            const int cx = iclamp(int(floorf(p.x)), 0, F.X - 1) >> kIsoCellShift;
            const int cy = iclamp(int(floorf(p.y)), 0, F.Y - 1) >> kIsoCellShift;
            const int cz = iclamp(int(floorf(p.z)), 0, F.Z - 1) >> kIsoCellShift;
            const uint32_t mark = F.isoCells[uint32_t(cx) + uint32_t(F.ncx) * (uint32_t(cy) + uint32_t(F.ncy) * uint32_t(cz))];
            // the last step before the ray leaves the cell's slabs; texels are clamped, so the first and
            // last cell of an axis reach beyond the texture and a ray never leaves them outwards (nor
            // any cell along an axis it does not move on)
            auto exit = [](int cell, float c, float v, float r, int n)
            {
                const int next = v > 0.0f ? cell + 1 : cell;
                const bool inner = v != 0.0f && next > 0 && (next << kIsoCellShift) < n;
                return inner ? (float(next << kIsoCellShift) - c) * r : FLT_MAX;
            };
            const float t = fminf(fminf(exit(cx, L.c.x, L.v.x, inv.x, F.X), exit(cy, L.c.y, L.v.y, inv.y, F.Y)),
                                  exit(cz, L.c.z, L.v.z, inv.z, F.Z));
            float end = floorf(fmaxf(fminf(t, lastF), k));
            if(mark == F.isoEpoch)
            {
                const int start = int(k);
                lead = start == to + 1 ? lead + 1 : -0x40000000;
                if(lead == LEAD)
                    end = lastF;
                from = min(from, start);
                to = int(end); // (last where end is lastF: both are below 2^23)
            }
            k = end + 1.0f;
        }
    }

    template<bool LINEAR, bool COUNT, bool OFF32>
    __device__ __attribute__((always_inline)) inline void march_body(const FrameParams& F, const ParticleParams& PP)
    {
        int px, py;
        const bool valid = tile_pixel_at(F, march_tile(F), march_wave(F), px, py);
        unsigned long long nCells = 0, nTests = 0, nIso = 0, nIsoHits = 0, nIsoRays = 0, nPartRays = 0;
        unsigned long long nVol = 0, nVolRays = 0, nSteps = 0;
        if(valid)
        {
            const size_t p = size_t(py) * size_t(F.W) + size_t(px);
            uint32_t color = F.bgClear;
            F3 normal = f3(0.f, 0.f, 0.f);
            float depth = FLT_MAX;
            float4 vcol = make_float4(0.f, 0.f, 0.f, -1.f);
            Ray ray = pixel_to_ray(F, px, py);
            const bool inside = clip_ray(F, ray);
            // ---- particles
            if(inside && PP.nsrc > 0)
            {
                nPartRays++;
                particle_dda<COUNT>(PP, ray, color, depth, normal, nCells, nTests);
            }
            // ---- iso + volume, one traversal
            const int mode = F.renderMode;
            // ShadingKernel zeroes the depth in these modes, so the volume pass never blends there
            const bool depthZeroed = mode == 2 || (mode >= 4 && mode <= 8);
            if(inside)
            {
                const float endAfterParticles = gmin(ray.endDepth, depth);
                bool isoOn = F.isoEnabled && endAfterParticles > ray.startDepth;
                bool volBlend = F.volumeEnabled && !depthZeroed && endAfterParticles > ray.startDepth;
                if(isoOn || volBlend)
                {
                    const F3 sc = f3(F.scale[0], F.scale[1], F.scale[2]);
                    const float stepU = F.step * (len3(ray.dir) / len3(divv(ray.dir, sc)));
                    const float factor = stepU / F.minSize * 2.0f * F.totalWeightAll;
                    const int startSteps = int(ceilf(ray.startDepth / stepU));
                    const int endIso = int(floorf(endAfterParticles / stepU));
                    const F3 stepVec = divv(muls(ray.dir, stepU), sc);
                    const F3 startU = divv(ray.start, sc);
                    if(isoOn)
                        nIsoRays++;
                    VolAcc acc{0.f, 0.f, 0.f, 0.f};
                    // The traversal state is kept in plain numbers rather than flags, so the loops
                    // carry no lane masks: the iso test runs while isoFrom <= i <= isoEnd and the
                    // volume while i <= volEnd (set below the first step to switch it off); hitStep
                    // is the step of the iso hit (-1: none); oldValue is the iso sum of step oldStep,
                    // the last one formed; blendW is the volume colour's w marker (0: the volume
                    // pass blends, -1: it does not).
                    const int off = -0x7fffffff;
                    int isoFrom = 0x7fffffff, isoEnd = off;
                    int volEnd = volBlend ? endIso : off;
                    int hitStep = -1;
                    float blendW = volBlend ? 0.0f : -1.0f;
                    if(startSteps <= endIso)
                    {
                        // volume samples times factor / 255
                        const float vscale = factor * (1.0f / 255.0f) * (LINEAR ? kByteScale : 1.0f);
                        const uint32_t XY = uint32_t(F.X) * uint32_t(F.Y);
                        // sample k at startC + stepVec * k, shifted by the texel centres' -0.5 for
                        // the trilinear sampler
                        const float sh = LINEAR ? 0.5f : 0.0f;
                        const StepLine L{f3(startU.x - sh, startU.y - sh, startU.z - sh), stepVec};
                        // step numbers that are exact as floats, in the loops that count in floats
                        const bool exact = endIso < (1 << 23);
                        int in0 = 0, in1 = -1;
                        if(LINEAR && !COUNT && volBlend && exact)
                            interior_steps(F, L, startSteps, endIso, in0, in1);
                        if(isoOn)
                        {
                            if(COUNT || !exact) // (the counting march tests every step, as the reference does)
                            {
                                isoFrom = startSteps;
                                isoEnd = endIso;
                            }
                            else
                                iso_steps<LINEAR ? 16 : 3>(F, L, startSteps, endIso, isoFrom, isoEnd);
                        }
                        float oldValue = 0.0f; // (0 before the first step)
                        int oldStep = startSteps - 1;
                        auto place = [&](int i)
                        {
                            const F3 c = L.at(float(i));
                            return place_of<LINEAR>(F, XY, c.x, c.y, c.z);
                        };
                        // the iso test of step i, whose corners have the texels t and the weights W
                        auto iso_test = [&](int i, const uint32_t t[8], const Weights& W) __attribute__((always_inline))
                        {
                            if(COUNT)
                                nIso++;
                            // the iso alpha in byte units; alpha >= 0.5 is a sum >= 127.5, which needs an
                            // alpha byte >= 128 (the corner weights sum to 1 up to a few ulps, so eight
                            // bytes <= 127 stay below 127.1): without one the sum is not formed, and
                            // formed again from the step's corners if the next step hits
                            uint32_t any = t[0];
                            if(LINEAR)
                            {
#pragma unroll
                                for(int j = 1; j < 8; j++)
                                    any |= t[j];
                            }
                            if((any >> 31) == 0u)
                                return;
                            const float sum = iso_sum<LINEAR>(t, W);
                            if(sum >= 127.5f)
                            {
                                float before = oldValue;
                                if(oldStep != i - 1)
                                {
                                    const Place pp = place(i - 1);
                                    uint32_t tp[8];
                                    fetch_place<LINEAR, OFF32>(F.iso, pp, tp);
                                    before = iso_sum<LINEAR>(tp, corner_weights(pp.fx, pp.fy, pp.fz));
                                }
                                const bool first = ray.isClipped && i == startSteps;
                                const float tt = float(i) * stepU;
                                const float value = div255(sum), tmp = div255(before);
                                // colour and gradient at the hit are sampled after the loop
                                hitStep = i;
                                depth = first ? ray.startDepth : tt + stepU * (0.5f - tmp) / (value - tmp);
                                if(COUNT)
                                    nIsoHits++;
                                isoEnd = off;
                                // the volume pass ends at min(clip end, iso depth)
                                const float ve = gmin(ray.endDepth, depth);
                                if(!(ve > ray.startDepth))
                                {
                                    volEnd = off;
                                    blendW = -1.0f;
                                }
                                else if(volEnd != off)
                                    volEnd = int(floorf(ve / stepU));
                            }
                            oldValue = sum;
                            oldStep = i;
                        };
                        // The steps in front of the interior ones, the interior ones, and the steps
                        // after them: three loops in turn, so that no lane runs the interior while
                        // its neighbours still wait to reach theirs.
                        int i = startSteps;
#pragma unroll 1
                        for(int part = 0; part < 2; part++)
                        {
                            const int head = part == 0 && in0 <= in1 ? in0 - 1 : 0x7fffffff;
                            while(i <= min(max(isoEnd, volEnd), head))
                            {
                                if(COUNT)
                                    nSteps++;
                                const Place pl = place(i);
                                const Weights W = corner_weights(pl.fx, pl.fy, pl.fz);
                                // (nearest, which has no request ahead: both textures' texels are requested before the
                                // first is looked at, march of 181x127x203 voxels at 1283x719 176 -> 168 us; the trilinear
                                // march, whose interior steps have one, holds 8 more VGPRs for nothing)
                                uint32_t tv[8];
                                if(!LINEAR && i <= volEnd)
                                    fetch_place<LINEAR, OFF32>(F.vol, pl, tv);
                                if(i >= isoFrom && i <= isoEnd)
                                {
                                    uint32_t t[8];
                                    fetch_place<LINEAR, OFF32>(F.iso, pl, t);
                                    iso_test(i, t, W);
                                }
                                if(i <= volEnd)
                                {
                                    if(COUNT)
                                        nVol++;
                                    if(LINEAR)
                                        fetch_place<LINEAR, OFF32>(F.vol, pl, tv);
                                    composite(acc, vol_sums<LINEAR>(tv, W), vscale);
                                    if(acc.a > 0.99f)
                                        volEnd = off;
                                }
                                i++;
                                // without volume, on to the steps that can meet the surface
                                if(i > volEnd)
                                    i = max(i, isoFrom);
                            }
                            if constexpr(!LINEAR || COUNT)
                                break;
                            else if(part == 0)
                            {
                                // The interior steps that the volume takes (no clamps).  VALU issue bounds
                                // this loop: 32 masks and 32 fmas, 16 for the corner weights, 12 for
                                // position and offset, 10 to composite.  The four row pairs share one
                                // offset register (their distances go into four uniform base
                                // addresses).  The next step's pairs are requested before this step's
                                // are summed, two buffers in turn.
                                struct Sample
                                {
                                    TexPair p[4];
                                    uint32_t o;
                                    float fx, fy, fz;
                                };
                                const size_t r01 = size_t(XY) * 4u, r10 = size_t(F.X) * 4u;
                                auto rows = [&](const uint32_t* tex, Sample& s) __attribute__((always_inline))
                                {
                                    const char* b = reinterpret_cast<const char*>(tex);
                                    const size_t o = OFF32 ? size_t(s.o) : size_t(s.o) << 2;
                                    s.p[0] = *reinterpret_cast<const TexPair*>(b + o);
                                    s.p[1] = *reinterpret_cast<const TexPair*>(b + r01 + o);
                                    s.p[2] = *reinterpret_cast<const TexPair*>(b + r10 + o);
                                    s.p[3] = *reinterpret_cast<const TexPair*>(b + r01 + r10 + o);
                                };
                                auto get = [&](float q, Sample& s) __attribute__((always_inline))
                                {
                                    const F3 c = L.at(q);
                                    // (c >= 0: its fraction is exact, and truncation is the floor)
                                    s.fx = __builtin_amdgcn_fractf(c.x);
                                    s.fy = __builtin_amdgcn_fractf(c.y);
                                    s.fz = __builtin_amdgcn_fractf(c.z);
                                    const uint32_t x = uint32_t(c.x), y = uint32_t(c.y), z = uint32_t(c.z);
                                    s.o = OFF32 ? (x + __umul24(y, uint32_t(F.X)) + __umul24(z, XY)) << 2 : x + y * uint32_t(F.X) + z * XY;
                                    rows(F.vol, s);
                                };
                                // step q from its sample: false where the loop ends
                                float e = float(min(volEnd, in1));
                                const float isoFromF = float(isoFrom);
                                float isoEndF = float(isoEnd);
                                auto use = [&](float q, const Sample& s) __attribute__((always_inline))
                                {
                                    const Weights W = corner_weights(s.fx, s.fy, s.fz);
                                    if(q >= isoFromF && q <= isoEndF)
                                    {
                                        Sample iso = s;
                                        rows(F.iso, iso);
                                        const uint32_t t[8] = {iso.p[0].x, iso.p[1].x, iso.p[2].x, iso.p[3].x,
                                                               iso.p[0].y, iso.p[1].y, iso.p[2].y, iso.p[3].y};
                                        iso_test(int(q), t, W);
                                        isoEndF = float(isoEnd);
                                        e = float(min(volEnd, in1));
                                        if(q > e)
                                            return false;
                                    }
                                    const uint32_t t[8] = {s.p[0].x, s.p[1].x, s.p[2].x, s.p[3].x, s.p[0].y, s.p[1].y, s.p[2].y, s.p[3].y};
                                    composite(acc, vol_sums<true>(t, W), vscale);
                                    if(acc.a > 0.99f)
                                    {
                                        volEnd = off;
                                        return false;
                                    }
                                    return q < e;
                                };
                                if(i <= min(volEnd, in1))
                                {
                                    float k = float(i);
                                    Sample s0, s1;
                                    get(k, s0);
                                    for(;;)
                                    {
                                        get(fminf(k + 1.0f, e), s1);
                                        if(!use(k, s0))
                                            break;
                                        k = k + 1.0f;
                                        get(fminf(k + 1.0f, e), s0);
                                        if(!use(k, s1))
                                            break;
                                        k = k + 1.0f;
                                    }
                                    i = int(k) + 1;
                                    if(i > volEnd)
                                        i = max(i, isoFrom);
                                }
                            }
                        }
                    }
                    const bool isoHit = hitStep >= 0;
                    const bool isoFirst = isoHit && ray.isClipped && hitStep == startSteps;
                    if(isoHit)
                    {
                        // hit colour and central-difference gradient of the iso alpha
                        // (lib/isaac/isaac_iso_kernel.hpp:97-119)
                        const F3 pu = divv(add(ray.start, muls(ray.dir, depth)), sc);
                        Taps h;
                        fetch_taps<LINEAR>(F, pu.x, pu.y, pu.z, h);
                        const float hr = channel<LINEAR>(h, 0), hg = channel<LINEAR>(h, 8);
                        const float hb = channel<LINEAR>(h, 16);
                        F3 g;
                        g.x = iso_alpha_at<LINEAR>(F, pu.x + 1.0f, pu.y, pu.z) - iso_alpha_at<LINEAR>(F, pu.x - 1.0f, pu.y, pu.z);
                        g.y = iso_alpha_at<LINEAR>(F, pu.x, pu.y + 1.0f, pu.z) - iso_alpha_at<LINEAR>(F, pu.x, pu.y - 1.0f, pu.z);
                        g.z = iso_alpha_at<LINEAR>(F, pu.x, pu.y, pu.z + 1.0f) - iso_alpha_at<LINEAR>(F, pu.x, pu.y, pu.z - 1.0f);
                        float gl = len3(g);
                        if(isoFirst || gl == 0.0f)
                        {
                            g = ray.clipN;
                            gl = 1.0f;
                        }
                        normal = f3(-g.x / gl, -g.y / gl, -g.z / gl);
                        color = to_byte4(hr, hg, hb, 1.0f);
                    }
                    if(blendW >= 0.0f)
                    {
                        nVolRays++;
                        vcol = LINEAR ? make_float4(acc.r, acc.g * 0x1p-8f, acc.b * 0x1p-16f, acc.a)
                                      : make_float4(acc.r, acc.g, acc.b, acc.a);
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
            unsigned long long* const cnt = F.counters + blockIdx.x % kCounterSets * kCounterStride;
            block_count_add(cnt + 0, nVol);
            block_count_add(cnt + 1, nIso);
            block_count_add(cnt + 2, nIsoHits);
            block_count_add(cnt + 3, nCells);
            block_count_add(cnt + 4, nTests);
            block_count_add(cnt + 5, nVolRays);
            block_count_add(cnt + 6, nIsoRays);
            block_count_add(cnt + 7, nPartRays);
            block_count_add(cnt + 8, nSteps);
            // the wave runs the traversal loop as long as its longest lane
            int wm = int(nSteps);
            for(int off = 32; off > 0; off >>= 1)
                wm = max(wm, __shfl_xor(wm, off, 64));
            block_count_add(cnt + 9, (threadIdx.x & 63u) == 0 ? (unsigned long long) wm : 0ull);
        }
    }

    // Workgroups of one wave by default (march_block), which any SIMD with a free slot takes: with
    // four waves a workgroup waits for four slots of one CU while its rays' lengths differ.  At
    // 88 VGPRs (5 waves per SIMD); held to 80 or 64 registers for 6 or 8 waves it spills and is slower.
    // Measured on MI355X (events around it), before (8-byte texels with both textures, byte conversions,
    // an iso sum test every step, four-wave workgroups) and after: 256^3 with iso-surface and 2 M particles
    // at 1920x1080 514 -> 370 us (volume in the middle of the frame) and 810 -> 730 us (filling it, 176 G
    // samples/s: the waves wait for gathers and the last ones run alone); 512^3 at 3840x2160 and step 0.25
    // 4730 -> 3720 us, 436 G samples/s, 354 cycles of a SIMD per 64 samples of which about 305 issue VALU
    // instructions; 64^3 at 512x512 82 -> 58 us.  Four-wave workgroups: 370, 805, 3735 and 58 us.  Without the
    // request ahead: 416, 733, 3990 and 73 us.
    template<bool LINEAR, bool COUNT, bool OFF32>
    __global__ __launch_bounds__(256) void march_kernel(const FrameParams F, const ParticleParams PP)
    {
        march_body<LINEAR, COUNT, OFF32>(F, PP);
    }

    template<bool LINEAR, bool OFF32>
    void launch_march_sampler(const FrameParams& F, const ParticleParams& PP, bool counting, dim3 grid, dim3 block, hipStream_t s)
    {
        if(counting)
            hipLaunchKernelGGL((march_kernel<LINEAR, true, OFF32>), grid, block, 0, s, F, PP);
        else
            hipLaunchKernelGGL((march_kernel<LINEAR, false, OFF32>), grid, block, 0, s, F, PP);
    }

    hipError_t launch_march(const FrameParams& F, const ParticleParams& PP, bool counting, hipStream_t s)
    {
        const unsigned nb = march_grid(F);
        if(nb == 0)
            return hipSuccess;
        // one-wave workgroups: 4 per logical workgroup, the logical grid rounded to 8
        const dim3 grid(F.waveGroups == 1 ? (nb + 7u) / 8u * 32u : nb), block(F.waveGroups == 1 ? 64 : 256);
        if(!F.linear) // (one texel per step: its load takes the texel index either way)
            launch_march_sampler<false, false>(F, PP, counting, grid, block, s);
        else if(F.texOff32)
            launch_march_sampler<true, true>(F, PP, counting, grid, block, s);
        else
            launch_march_sampler<true, false>(F, PP, counting, grid, block, s);
        return hipGetLastError();
    }
} // namespace isaac_hip
