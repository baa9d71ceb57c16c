// Device functions shared by the render kernels: ray setup, pixel tiles of the
// workgroups, the particle walk, byte scaling, functor chains, source signatures.
#pragma once

#include "kernels.hpp"

namespace isaac_hip
{
    // x / 255 in binary32 as x*r plus one fma residual correction, r = RN(1/255).
    // For every float x in [0, 256] this equals the IEEE quotient bit for bit
    // (tests/test_div255.py checks all 1,132,462,081 inputs); trilinear results
    // of RGBA8 texels always lie in [0, 255].  Three instructions instead of the
    // correctly rounded division sequence.
    __device__ inline float div255(float x)
    {
        const float r = 1.0f / 255.0f;
        const float q0 = x * r;
        const float e = __builtin_fmaf(-q0, 255.0f, x);
        return __builtin_fmaf(e, r, q0);
    }

    // ------------------------------------------------------------------ rays
    struct Ray
    {
        F3 dir, start;
        float startDepth, endDepth;
        bool isClipped;
        F3 clipN;
    };

    // pixelToRay (lib/isaac/isaac_common_kernel.hpp:51-92); glm mat4*vec4 = (m0*x+m1*y)+(m2*z+m3*w)
    __device__ inline Ray pixel_to_ray(const FrameParams& F, int px, int py)
    {
        const float vx = float(px) / F.fbW * 2.0f - 1.0f;
        const float vy = float(py) / F.fbH * 2.0f - 1.0f;
        float s[4], e[4];
#pragma unroll
        for(int r = 0; r < 4; r++)
        {
            const float a0 = F.inv[0 * 4 + r] * vx;
            const float a1 = F.inv[1 * 4 + r] * vy;
            const float s0 = a0 + a1;
            const float bs = F.inv[2 * 4 + r] * -1.0f;
            const float be = F.inv[2 * 4 + r] * 1.0f;
            const float a3 = F.inv[3 * 4 + r] * 1.0f;
            s[r] = s0 + (bs + a3);
            e[r] = s0 + (be + a3);
        }
        Ray ray;
        F3 st = f3(s[0] / s[3], s[1] / s[3], s[2] / s[3]);
        F3 en = f3(e[0] / e[3], e[1] / e[3], e[2] / e[3]);
        st = muls(st, F.maxSize);
        en = muls(en, F.maxSize);
        ray.dir = normalize3(sub(en, st));
        ray.start = st;
        ray.isClipped = false;
        ray.clipN = f3(0.f, 0.f, 0.f);
        ray.startDepth = 0.f;
        ray.endDepth = 0.f;
        return ray;
    }

    // clipRay (lib/isaac/isaac_common_kernel.hpp:94-193)
    __device__ inline bool clip_ray(const FrameParams& F, Ray& ray)
    {
        ray.start = add(ray.start, f3(F.off[0], F.off[1], F.off[2]));
        float bmin[3], bmax[3];
        const float st[3] = {ray.start.x, ray.start.y, ray.start.z};
        const float dr[3] = {ray.dir.x, ray.dir.y, ray.dir.z};
#pragma unroll
        for(int i = 0; i < 3; i++)
        {
            bmin[i] = (F.bbMin[i] - st[i]) / dr[i];
            bmax[i] = (F.bbMax[i] - st[i]) / dr[i];
            if(bmax[i] < bmin[i])
            {
                float t = bmax[i];
                bmax[i] = bmin[i];
                bmin[i] = t;
            }
        }
        ray.startDepth = gmax(bmin[0], gmax(bmin[1], bmin[2]));
        ray.endDepth = gmin(bmax[0], gmin(bmax[1], bmax[2]));
        float cn[3] = {0.f, 0.f, 0.f};
#pragma unroll
        for(int i = 0; i < 3; i++)
        {
            const float sgn = gsign(dr[i]);
            const bool lowOuter = F.outerLow[i] && (sgn + 1.0f) != 0.0f;
            const bool highOuter = F.outerHigh[i] && (sgn - 1.0f) != 0.0f;
            if(bmin[i] == ray.startDepth && (lowOuter || highOuter))
            {
                ray.isClipped = true;
                cn[i] = sgn;
            }
        }
        ray.clipN = f3(cn[0], cn[1], cn[2]);
        for(int i = 0; i < F.nclip; i++)
        {
            const F3 n = f3(F.cnorm[i][0], F.cnorm[i][1], F.cnorm[i][2]);
            const F3 p = f3(F.cpos[i][0], F.cpos[i][1], F.cpos[i][2]);
            const float d = dot3(ray.dir, n);
            const float depth = (dot3(p, n) - dot3(ray.start, n)) / d;
            if(d > 0.0f)
            {
                if(ray.endDepth < depth)
                    return false;
                if(ray.startDepth <= depth)
                {
                    ray.clipN = n;
                    ray.isClipped = true;
                    ray.startDepth = depth;
                }
            }
            else
            {
                if(ray.startDepth > depth)
                    return false;
                if(ray.endDepth > depth)
                    ray.endDepth = depth;
            }
        }
        ray.startDepth = gmax(ray.startDepth, kZNear);
        if(ray.startDepth > ray.endDepth || isinf(ray.startDepth) || isinf(ray.endDepth))
            return false;
        return true;
    }

    struct F4
    {
        float x, y, z, w;
    };

    // ------------------------------------------------------------------ pixel tiling
    // pixel of this lane in 16x16 tile b of the viewport (row-major tiles), whose 8x8 quarter
    // `wave` (0..3) its wave renders; false outside the viewport
    __device__ inline bool tile_pixel_at(const FrameParams& F, uint32_t b, uint32_t wave, int& px, int& py)
    {
        const uint32_t tx = b % uint32_t(F.tilesX), ty = b / uint32_t(F.tilesX);
        const uint32_t lane = threadIdx.x & 63u;
        px = F.vx0 + int(tx * 16u + (wave & 1u) * 8u + (lane & 7u));
        py = F.vy0 + int(ty * 16u + (wave >> 1) * 8u + (lane >> 3));
        return b < uint32_t(F.tilesX) * uint32_t(F.tilesY) && px < F.vx1 && py < F.vy1;
    }

    __device__ inline bool tile_pixel_at(const FrameParams& F, uint32_t b, int& px, int& py)
    {
        return tile_pixel_at(F, b, threadIdx.x >> 6, px, py);
    }

    // The march's workgroups: one 16x16 tile of 4 waves each, or (F.waveGroups == 1)
    // one wave each: workgroup b is then quarter (b / 8) % 4 of the tile of logical
    // workgroup (b / 32) * 8 + b % 8, and runs on the XCD b % 8 of that logical
    // workgroup, so the dealing of tiles to the XCDs is unchanged while the
    // dispatcher fills any SIMD with a free wave slot.
    __device__ inline uint32_t march_block(const FrameParams& F)
    {
        return F.waveGroups == 1 ? ((blockIdx.x >> 5) << 3) | (blockIdx.x & 7u) : blockIdx.x;
    }
    __device__ inline uint32_t march_wave(const FrameParams& F)
    {
        return F.waveGroups == 1 ? (blockIdx.x >> 3) & 3u : threadIdx.x >> 6;
    }

    __device__ inline uint32_t xcd_tile(const FrameParams& F, uint32_t b)
    {
        const uint32_t nb = uint32_t(F.tilesX) * uint32_t(F.tilesY);
        const uint32_t full = nb & ~7u;
        if(b < full)
            b = (b & 7u) * (full >> 3) + (b >> 3);
        return b;
    }

    // Super-tiles of SxS tiles (S = F.tileOrder: 2, 4, 8 or 16; 4 is 64x64 pixels)
    // dealt round-robin to the XCDs: workgroup b runs on XCD b % 8 and takes tile
    // (b / 8) % S^2 of that XCD's super-tile number (b / 8) / S^2.  Every XCD gets
    // super-tiles from all over the frame (balanced when the work is concentrated,
    // e.g. a volume in the middle of the frame) while the rays of one super-tile
    // share its L2.  Grid: march_grid workgroups; padding workgroups map to no tile.
    __device__ inline uint32_t supertile_tile(const FrameParams& F, uint32_t b)
    {
        const uint32_t S = uint32_t(F.tileOrder), sh = uint32_t(__ffs(int(S)) - 1);
        const uint32_t tX = uint32_t(F.tilesX), tY = uint32_t(F.tilesY);
        const uint32_t sx = (tX + S - 1u) >> sh, sy = (tY + S - 1u) >> sh;
        const uint32_t i = b >> 3;
        const uint32_t s = (b & 7u) + 8u * (i >> (2u * sh)), w = i & (S * S - 1u);
        if(s >= sx * sy)
            return 0xffffffffu;
        const uint32_t tx = ((s % sx) << sh) + (w & (S - 1u)), ty = ((s / sx) << sh) + (w >> sh);
        if(tx >= tX || ty >= tY)
            return 0xffffffffu;
        return ty * tX + tx;
    }

    __device__ inline uint32_t march_tile(const FrameParams& F)
    {
        const uint32_t b = march_block(F);
        return F.tileOrder != 0 ? supertile_tile(F, b) : xcd_tile(F, b);
    }

    __device__ inline void block_count_add(unsigned long long* dst, unsigned long long v)
    {
        __shared__ unsigned long long red[4];
        // wave reduction through DPP-free shuffles
        for(int off = 32; off > 0; off >>= 1)
            v += __shfl_down(v, off, 64);
        if((threadIdx.x & 63) == 0)
            red[threadIdx.x >> 6] = v;
        __syncthreads();
        if(threadIdx.x == 0)
        {
            unsigned long long s = 0;
            for(uint32_t w = 0; w < (blockDim.x >> 6); w++)
                s += red[w];
            if(s)
                atomicAdd(dst, s);
        }
        __syncthreads();
    }

    // ------------------------------------------------------------------ particles
    // ParticleRenderKernel (lib/isaac/isaac_particle_kernel.hpp:117-260): 3D-DDA over
    // the particle cell grid from the clipped ray start; the first cell holding a
    // visible sphere hit ends the walk (hit point of the nearest sphere in it).
    template<bool COUNT>
    __device__ inline void particle_dda(
        const ParticleParams& PP,
        const Ray& ray,
        uint32_t& color,
        float& depth,
        F3& normal,
        unsigned long long& nCells,
        unsigned long long& nTests)
    {
        const F3 ps = f3(PP.pscale[0], PP.pscale[1], PP.pscale[2]);
        const int ds[3] = {int(gsign(ray.dir.x)), int(gsign(ray.dir.y)), int(gsign(ray.dir.z))};
        const F3 cur = add(ray.start, muls(ray.dir, ray.startDepth));
        const F3 cdiv = divv(cur, ps);
        uint32_t cell[3];
        cell[0] = uint32_t(iclamp(int(cdiv.x), 0, PP.grid[0] - 1));
        cell[1] = uint32_t(iclamp(int(cdiv.y), 0, PP.grid[1] - 1));
        cell[2] = uint32_t(iclamp(int(cdiv.z), 0, PP.grid[2] - 1));
        const float rayLength = ray.endDepth - ray.startDepth;
        float tested = 0.0f;
        const float curA[3] = {cur.x, cur.y, cur.z};
        const float dA[3] = {ray.dir.x, ray.dir.y, ray.dir.z};
        const float psA[3] = {ps.x, ps.y, ps.z};
        float t[3], dt[3];
#pragma unroll
        for(int i = 0; i < 3; i++)
        {
            t[i] = ((float(cell[i]) + float(ds[i] > 0 ? ds[i] : 0)) * psA[i] - curA[i]) / dA[i];
            dt[i] = psA[i] / dA[i] * float(ds[i]);
            if(dA[i] == 0.0f)
                t[i] = FLT_MAX;
        }
        bool hit = false;
        float pdepth = FLT_MAX;
        float4 pcol = make_float4(0.f, 0.f, 0.f, 0.f);
        F3 pn = f3(0.f, 0.f, 0.f);
        const uint32_t gx = uint32_t(PP.grid[0]), gy = uint32_t(PP.grid[1]), gz = uint32_t(PP.grid[2]);
        auto inside = [&](const uint32_t (&c)[3]) { return c[0] < gx && c[1] < gy && c[2] < gz; };
        auto cell_id = [&](const uint32_t (&c)[3]) { return int(c[0] + gx * (c[1] + gy * c[2])); };
        // record ranges of the current cell, requested one cell ahead: the walk's next
        // cell depends on the ray only, so the range of cell i + 1 is in flight while
        // the spheres of cell i are tested
        int2 kr[4] = {};
        if(inside(cell))
        {
            const int cid = cell_id(cell);
#pragma unroll
            for(int s = 0; s < 4; s++)
                if(s < PP.nsrc)
                    kr[s] = PP.src[s].vrange[cid];
        }
        while(inside(cell) && !hit && tested <= rayLength)
        {
            if(COUNT)
                nCells++;
            // the walk's next cell (ties between axes go towards z)
            uint32_t next[3] = {cell[0], cell[1], cell[2]};
            float nextTested;
            const bool ax0 = t[0] < t[1] && t[0] < t[2];
            const bool ax1 = !ax0 && t[1] < t[0] && t[1] < t[2];
            if(ax0)
            {
                next[0] += uint32_t(ds[0]);
                nextTested = t[0];
            }
            else if(ax1)
            {
                next[1] += uint32_t(ds[1]);
                nextTested = t[1];
            }
            else
            {
                next[2] += uint32_t(ds[2]);
                nextTested = t[2];
            }
            int2 krn[4] = {};
            if(inside(next))
            {
                const int nid = cell_id(next);
#pragma unroll
                for(int s = 0; s < 4; s++)
                    if(s < PP.nsrc)
                        krn[s] = PP.src[s].vrange[nid];
            }
            const F3 cf = f3(float(cell[0]), float(cell[1]), float(cell[2]));
#pragma unroll
            for(int s = 0; s < 4; s++)
            {
                if(s >= PP.nsrc)
                    break;
                const ParticleSourceDev& S = PP.src[s];
                for(int k = kr[s].x; k < kr[s].y; k++)
                {
                    if(COUNT)
                        nTests++;
                    const float4 rec = S.recs[k];
                    const F3 ppos = mul(add(f3(rec.x, rec.y, rec.z), cf), ps);
                    const F3 L = sub(ppos, cur);
                    const float radius = (S.radius ? S.radius[k] : S.constRadius) * S.weight;
                    const float r2 = radius * radius;
                    const float tca = dot3(L, ray.dir);
                    const float d2 = dot3(L, L) - tca * tca;
                    if(d2 <= r2)
                    {
                        const float thc = sqrtf(r2 - d2);
                        const float t0 = tca - thc;
                        const float t1 = tca + thc;
                        if(t1 >= 0.0f && t0 < pdepth)
                        {
                            const float4 val = S.lut[__float_as_int(rec.w)];
                            if(val.w >= 0.5f)
                            {
                                pcol = val;
                                pdepth = t0;
                                hit = true;
                                pn = sub(add(cur, muls(ray.dir, t0)), ppos);
                                if(t0 < 0.0f && ray.isClipped)
                                    pn = f3(-ray.clipN.x, -ray.clipN.y, -ray.clipN.z);
                            }
                        }
                    }
                }
            }
            cell[0] = next[0];
            cell[1] = next[1];
            cell[2] = next[2];
            tested = nextTested;
            if(ax0)
                t[0] = t[0] + dt[0];
            else if(ax1)
                t[1] = t[1] + dt[1];
            else
                t[2] = t[2] + dt[2];
#pragma unroll
            for(int s = 0; s < 4; s++)
                kr[s] = krn[s];
        }
        if(hit)
        {
            normal = normalize3(pn);
            color = to_byte4(pcol.x, pcol.y, pcol.z, 1.0f);
            depth = pdepth + ray.startDepth;
        }
    }

    // workgroups of a march launch: one per tile, or the padded super-tile grid
    inline unsigned march_grid(const FrameParams& F)
    {
        const unsigned nb = unsigned(F.tilesX) * unsigned(F.tilesY);
        const unsigned S = unsigned(F.tileOrder);
        if(S == 0 || nb == 0)
            return nb;
        const unsigned ns = ((unsigned(F.tilesX) + S - 1u) / S) * ((unsigned(F.tilesY) + S - 1u) / S);
        return (ns + 7u) / 8u * 8u * S * S;
    }

    // ------------------------------------------------------------------ functor chain
    // pow stays out of line: inlined, its ~70 instructions per component and
    // functor slot made up most of the code of the marches that evaluate the
    // chain per sample (rarely used, and the call is only taken for it).
    static __device__ __noinline__ float chain_pow(float a, float b)
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

    // a source's chain is its natural one: no operations for a scalar source, one
    // `length` (then nothing) for a vector source
    inline bool natural_chain(const ChainDesc& c, int dim)
    {
        for(int k = 0; k < kMaxFunctors; k++)
        {
            const int want = (k == 0 && dim > 1) ? OP_LENGTH : OP_IDEM;
            if(c.op[k] != want)
                return false;
        }
        return true;
    }

    // ------------------------------------------------------------------ source signatures
    // Source signature: the component counts of the enabled sources in slot
    // order, as base-5 digits (slot 0 lowest), 0 = resolved at run time.  A
    // march compiled for one signature fetches the rows of all its sources
    // before interpolating any of them, so their latencies overlap.
    constexpr bool sig_natural(int sig)
    {
        return sig % kSigJoint >= kSigNatural;
    }

    constexpr bool sig_joint(int sig)
    {
        return sig >= kSigJoint;
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

    // tf_index(sqrtf(s), T) for s >= 0 (or NaN): v_sqrt_f32 is within one ulp of the square root, so the
    // value whose integer part is the index is within y * 2^-21 of the one that the correctly rounded
    // root gives, and the integer parts agree unless an integer lies that near; only then (about one
    // value in 1000 at T = 1024) the root is rounded correctly, which takes some 15 instructions
    __device__ inline int tf_index_sqrt(float s, int T)
    {
        const float y = __builtin_amdgcn_sqrtf(s) * float(T) + 0x1.fffffep-2f;
        // (a branch of the whole wave: per lane the compiler would compute both)
        if(__builtin_amdgcn_ballot_w64(!(fabsf(y - rintf(y)) > y * 0x1p-20f)) != 0) // (NaN and infinity too)
            return tf_index(sqrtf(s), T);
        return (int) __builtin_amdgcn_fmed3f(y, 0.0f, float(T - 1));
    }

    // the transfer index of a D-component sample's natural chain: of the value itself, or of the
    // length with apply_chain's association ((v0 v0 + v1 v1) + v2 v2)
    template<int D>
    __device__ inline int natural_index(const float (&v)[4], int T)
    {
        if constexpr(D == 1)
            return tf_index(v[0], T);
        else if constexpr(D == 2)
            return tf_index_sqrt(v[0] * v[0] + v[1] * v[1], T);
        else if constexpr(D == 3)
            return tf_index_sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2], T);
        else
            return tf_index_sqrt((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]), T);
    }
} // namespace isaac_hip
