// The brick form's march on gfx950 (post-classification over FP32 / FP16 / BF16 field
// bricks), of one frame and of a batch of frames in one persistent launch.
#include "render_device.hpp"

namespace isaac_hip
{
    static_assert(sizeof(FrameParams) + sizeof(PostParams) + sizeof(ParticleParams) <= 4096, "kernel argument block");

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
        uint32_t row; // pair row (x0, y0, z0) among all bricks' rows
        uint32_t dy, dz; // rows to (x0, y1, z0) and (x0, y0, z1): 8 and 72, or 0 at a clamped edge
        // trilinear weights of the corners (x, y, z) = 000 001 010 011 100 101 110 111,
        // shared by every component of every source at this position; where both x
        // taps are texel x0 (CLAMP at the x edge) the x1 corners weigh 0
        float w[8];
    };

    constexpr uint32_t kPairRowY = 8, kPairRowZ = 72; // pair rows from (y, z) to (y + 1, z) and (y, z + 1)

    __device__ inline void brick_weights(BrickTaps& t, float fx, float fy, float fz)
    {
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
    }

    template<bool LINEAR>
    __device__ inline BrickTaps brick_taps(const PostParams& Q, int X, int Y, int Z, float px, float py, float pz)
    {
        BrickTaps t;
        if(!LINEAR)
        {
            const uint32_t x = iclamp(int(px), 0, X - 1), y = iclamp(int(py), 0, Y - 1), z = iclamp(int(pz), 0, Z - 1);
            t.brick = ((z >> 3) * uint32_t(Q.nby) + (y >> 3)) * uint32_t(Q.nbx) + (x >> 3);
            t.row = t.brick * uint32_t(kBrickPairs) + ((z & 7) * 9 + (y & 7)) * 8 + (x & 7);
            t.dy = t.dz = 0u;
            return t;
        }
        const float cx = px - 0.5f, cy = py - 0.5f, cz = pz - 0.5f;
        const float flx = floorf(cx), fly = floorf(cy), flz = floorf(cz);
        const int bx = int(flx), by = int(fly), bz = int(flz);
        const uint32_t x0 = iclamp(bx, 0, X - 1), x1 = iclamp(bx + 1, 0, X - 1);
        const uint32_t y0 = iclamp(by, 0, Y - 1), y1 = iclamp(by + 1, 0, Y - 1);
        const uint32_t z0 = iclamp(bz, 0, Z - 1), z1 = iclamp(bz + 1, 0, Z - 1);
        t.brick = ((z0 >> 3) * uint32_t(Q.nby) + (y0 >> 3)) * uint32_t(Q.nbx) + (x0 >> 3);
        t.row = t.brick * uint32_t(kBrickPairs) + (x0 & 7u) + ((z0 & 7u) * 9u + (y0 & 7u)) * 8u;
        t.dy = (y1 - y0) * kPairRowY;
        t.dz = (z1 - z0) * kPairRowZ;
        brick_weights(t, x1 == x0 ? 0.0f : cx - flx, cy - fly, cz - flz);
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
        // one 64-bit product a source (one a row: march of three FP16 sources, 128^3 at 960x540,
        // 1157 us, 1072 us this way; strides known at compile time hold 30 more VGPRs: 1120 us)
        const uint32_t stride = uint32_t(S.stride);
        const uint32_t* rows = static_cast<const uint32_t*>(S.data) + size_t(t.row) * stride;
        const uint32_t at[4] = {0u, t.dy * stride, t.dz * stride, (t.dy + t.dz) * stride};
#pragma unroll
        for(int k = 0; k < (LINEAR ? 4 : 1); k++)
        {
            const Words<W> a = *reinterpret_cast<const Words<W>*>(rows + at[k]);
#pragma unroll
            for(int w = 0; w < W; w++)
                R.r[k][w] = a.w[w];
        }
        const Words<DIM> sc = *reinterpret_cast<const Words<DIM>*>(S.scale + size_t(t.brick) * uint32_t(S.scaleStride));
#pragma unroll
        for(int c = 0; c < DIM; c++)
            R.sc[c] = sc.w[c];
    }

    // the same of an interior sample (no clamps): one 32-bit byte offset from the source's
    // uniform base, the other rows at fixed distances.  (The addresses are marked as global
    // memory: of a batch, the compiler sees pointers read from memory.)
    typedef const __attribute__((address_space(1))) char* GlobalBytes;
    typedef const __attribute__((address_space(1))) uint32_t* GlobalWords;

    template<int DT, int DIM>
    __device__ inline void slot_fetch_interior(const BrickSource& S, uint32_t row, uint32_t brick, SlotRaw<DT>& R)
    {
        constexpr int W = row_words<DT, DIM>();
        constexpr uint32_t dist[4] = {0u, kPairRowY, kPairRowZ, kPairRowY + kPairRowZ};
        const uint32_t rowBytes = 4u * uint32_t(S.stride), at = row * rowBytes;
#pragma unroll
        for(int k = 0; k < 4; k++)
        {
            const GlobalBytes base = (GlobalBytes) S.data + dist[k] * rowBytes; // uniform
#pragma unroll
            for(int w = 0; w < W; w++)
                R.r[k][w] = ((GlobalWords) (base + at))[w];
        }
        const GlobalWords sc = (GlobalWords) ((GlobalBytes) S.scale + brick * (4u * uint32_t(S.scaleStride)));
#pragma unroll
        for(int c = 0; c < DIM; c++)
            R.sc[c] = sc[c];
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

    template<int DT, bool LINEAR, int SIG, int S>
    __device__ __attribute__((always_inline)) inline void sig_fetch(const PostParams& Q, const BrickTaps& t, SlotRaw<DT>* R)
    {
        if constexpr(S < sig_count(SIG))
        {
            slot_fetch_dim<DT, LINEAR, sig_dim(SIG, S)>(Q.src[S], t, R[S]);
            sig_fetch<DT, LINEAR, SIG, S + 1>(Q, t, R);
        }
    }

    template<int DT, int SIG, int S>
    __device__ __attribute__((always_inline)) inline void sig_fetch_interior(const PostParams& Q, uint32_t row, uint32_t brick, SlotRaw<DT>* R)
    {
        if constexpr(S < sig_count(SIG))
        {
            slot_fetch_interior<DT, sig_dim(SIG, S)>(Q.src[S], row, brick, R[S]);
            sig_fetch_interior<DT, SIG, S + 1>(Q, row, brick, R);
        }
    }

    // both sources of joint rows: 4 gathers and one of the scales
    template<int DT, int D0, int D1>
    __device__ __attribute__((always_inline)) inline void joint_fetch_interior(const PostParams& Q, uint32_t row, uint32_t brick, SlotRaw<DT>* R)
    {
        constexpr uint32_t dist[4] = {0u, kPairRowY, kPairRowZ, kPairRowY + kPairRowZ}, W = D0 + D1;
        const GlobalBytes base = (GlobalBytes) Q.src[0].data + row * (4u * W);
#pragma unroll
        for(int k = 0; k < 4; k++)
        {
            const GlobalWords w = (GlobalWords) (base + dist[k] * (4u * W));
#pragma unroll
            for(int c = 0; c < D0; c++)
                R[0].r[k][c] = w[c];
#pragma unroll
            for(int c = 0; c < D1; c++)
                R[1].r[k][c] = w[D0 + c];
        }
        const GlobalWords sc = (GlobalWords) ((GlobalBytes) Q.src[0].scale + brick * (4u * W));
#pragma unroll
        for(int c = 0; c < D0; c++)
            R[0].sc[c] = sc[c];
#pragma unroll
        for(int c = 0; c < D1; c++)
            R[1].sc[c] = sc[D0 + c];
    }

    // an interior sample's fetched rows and its fractions
    template<int DT, int SIG>
    struct InteriorSample
    {
        SlotRaw<DT> R[sig_count(SIG) ? sig_count(SIG) : 1];
        float fx, fy, fz;
    };

    template<int DT, int SIG>
    __device__ __attribute__((always_inline)) inline void fetch_interior(const PostParams& Q, float px, float py, float pz,
                                                                        InteriorSample<DT, SIG>& s)
    {
        const float cx = px - 0.5f, cy = py - 0.5f, cz = pz - 0.5f;
        // (c >= 0: truncation is the floor, and the fraction is exact)
        const uint32_t x = uint32_t(cx), y = uint32_t(cy), z = uint32_t(cz);
        s.fx = __builtin_amdgcn_fractf(cx);
        s.fy = __builtin_amdgcn_fractf(cy);
        s.fz = __builtin_amdgcn_fractf(cz);
        const uint32_t Bx = x >> 3, By = y >> 3, Bz = z >> 3;
        const uint32_t perY = uint32_t(kBrickPairs) * uint32_t(Q.nbx), perZ = perY * uint32_t(Q.nby);
        const uint32_t brick = (Bz * uint32_t(Q.nby) + By) * uint32_t(Q.nbx) + Bx;
        // 648 brick + (x & 7) + 8 (y & 7) + 72 (z & 7) with v & 7 = v - 8 (v >> 3)
        const uint32_t row = x + Bx * uint32_t(kBrickPairs - 8) + y * kPairRowY + By * (perY - 8u * kPairRowY) + z * kPairRowZ
            + Bz * (perZ - 8u * kPairRowZ);
        if constexpr(sig_joint(SIG))
            joint_fetch_interior<DT, sig_dim(SIG, 0), sig_dim(SIG, 1)>(Q, row, brick, s.R);
        else
            sig_fetch_interior<DT, SIG, 0>(Q, row, brick, s.R);
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
            const int li = sig_natural(SIG) ? natural_index<D>(v, Q.T) : tf_index(apply_chain(Q.src[S].chain, v[0], v[1], v[2], v[3], D), Q.T);
            post_accumulate(o, Q.src[S], lut[S * Q.T + li]);
            sig_classify<DT, LINEAR, SIG, S + 1>(Q, lut, t, R, o);
        }
    }

    template<int DT, int SIG>
    __device__ __attribute__((always_inline)) inline PostSample classify_interior(const PostParams& Q, const float4* lut,
                                                                                 const InteriorSample<DT, SIG>& s)
    {
        BrickTaps t;
        brick_weights(t, s.fx, s.fy, s.fz);
        PostSample o{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        sig_classify<DT, true, SIG, 0>(Q, lut, t, s.R, o);
        o.r = o.r * Q.invTotalWeight;
        o.g = o.g * Q.invTotalWeight;
        o.b = o.b * Q.invTotalWeight;
        o.a = o.a * Q.invTotalWeight;
        return o;
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

    // The steps i0..i1 of first..last whose samples lie inside [0, X-1) x [0, Y-1) x [0, Z-1) after
    // the texel centres' shift.  The estimate from the slabs is checked at both ends with the
    // march's own arithmetic, which is monotonic in i (every operation rounds monotonically),
    // so every step between them is inside too.  i1 < i0 where there are none.
    __device__ inline void brick_interior_steps(const FrameParams& F, const F3& start, const F3& v, int first, int last, int& i0, int& i1)
    {
        float lo = float(first), hi = float(last);
        auto slab = [&](float c, float d, int n)
        {
            const float a = (0.5f - c) / d, b = (float(n) - 0.5f - c) / d;
            lo = fmaxf(lo, fminf(a, b));
            hi = fminf(hi, fmaxf(a, b));
        };
        slab(start.x, v.x, F.X);
        slab(start.y, v.y, F.Y);
        slab(start.z, v.z, F.Z);
        i0 = 0;
        i1 = -1;
        if(!(lo <= hi)) // NaN bounds (an axis without movement) too
            return;
        const int j0 = int(ceilf(lo)), j1 = int(floorf(hi));
        auto inside = [&](int i)
        {
            const float fi = float(i);
            const float x = start.x + v.x * fi - 0.5f, y = start.y + v.y * fi - 0.5f, z = start.z + v.z * fi - 0.5f;
            return x >= 0.0f && x < float(F.X - 1) && y >= 0.0f && y < float(F.Y - 1) && z >= 0.0f && z < float(F.Z - 1);
        };
        // the slab bounds may be off by a rounding: one step in at each end is enough
        const int k0 = inside(j0) ? j0 : j0 + 1, k1 = inside(j1) ? j1 : j1 - 1;
        if(k0 <= k1 && inside(k0) && inside(k1))
        {
            i0 = k0;
            i1 = k1;
        }
    }

    template<int DT, bool LINEAR, bool COUNT, int SIG = 0>
    __device__ __attribute__((always_inline)) inline void brick_march_body(
        const FrameParams& F,
        const PostParams& Q,
        const ParticleParams& PP,
        const float4* lut,
        uint32_t tile,
        uint32_t wave)
    {
        int px, py;
        const bool valid = tile_pixel_at(F, tile, wave, px, py);
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
                    int i = startSteps;
                    // one step's classified sample: the iso test, the volume
                    auto take = [&](const PostSample& sm) __attribute__((always_inline))
                    {
                        if(COUNT)
                            nSteps++;
                        const float fi = float(i);
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
                        i++;
                    };
                    auto general = [&]() __attribute__((always_inline))
                    {
                        const float fi = float(i);
                        take(post_classify<DT, LINEAR, SIG>(Q, lut, F.X, F.Y, F.Z, startU.x + stepVec.x * fi, startU.y + stepVec.y * fi,
                                                            startU.z + stepVec.z * fi));
                    };
                    // The steps in front of the interior ones (whose corners need no clamp), those, and the
                    // steps after them: loops in turn, so that no lane runs the interior while its
                    // neighbours still wait to reach theirs.
                    if constexpr(SIG != 0 && !COUNT)
                    {
                        int in0 = 0, in1 = -1;
                        if(Q.off32 && endIso < (1 << 23))
                            brick_interior_steps(F, startU, stepVec, startSteps, endIso, in0, in1);
                        if(in0 <= in1)
                        {
                            while(i <= min(max(isoEnd, volEnd), in0 - 1))
                                general();
                            // the next step's rows are requested before this step's are classified,
                            // two buffers in turn
                            auto get = [&](int k, InteriorSample<DT, SIG>& smp) __attribute__((always_inline))
                            {
                                const float fk = float(min(k, in1));
                                fetch_interior<DT, SIG>(Q, startU.x + stepVec.x * fk, startU.y + stepVec.y * fk, startU.z + stepVec.z * fk, smp);
                            };
                            if(i <= min(max(isoEnd, volEnd), in1))
                            {
                                InteriorSample<DT, SIG> s0, s1;
                                get(i, s0);
                                for(;;)
                                {
                                    get(i + 1, s1);
                                    take(classify_interior<DT, SIG>(Q, lut, s0));
                                    if(i > min(max(isoEnd, volEnd), in1))
                                        break;
                                    get(i + 1, s0);
                                    take(classify_interior<DT, SIG>(Q, lut, s1));
                                    if(i > min(max(isoEnd, volEnd), in1))
                                        break;
                                }
                            }
                        }
                    }
                    while(i <= max(isoEnd, volEnd))
                        general();
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

    template<int DT, bool LINEAR, bool COUNT>
    __global__ __launch_bounds__(256) void brick_march_kernel(const FrameParams F, const PostParams Q, const ParticleParams PP)
    {
        extern __shared__ float4 lds_lut[];
        stage_luts(lds_lut, Q);
        __syncthreads();
        brick_march_body<DT, LINEAR, COUNT>(F, Q, PP, lds_lut, march_tile(F), threadIdx.x >> 6);
    }

    // trilinear march compiled for one source signature (see sig_count)
    template<int DT, int SIG>
    __global__ __launch_bounds__(256) void brick_march_sig_kernel(const FrameParams F, const PostParams Q, const ParticleParams PP)
    {
        extern __shared__ float4 lds_lut[];
        stage_luts(lds_lut, Q);
        __syncthreads();
        brick_march_body<DT, true, false, SIG>(F, Q, PP, lds_lut, march_tile(F), threadIdx.x >> 6);
    }

    // ------------------------------------------------------------------ persistent march
    // Work of a persistent march: the 8x8 quarters of the frames' 16x16 tiles, dealt in super-tiles
    // of 4x4 tiles to one queue per XCD (super-tile s of every frame to queue s % 8), so the rays
    // of a super-tile share an L2.  A wave pops from its own XCD's queue (workgroup b runs on XCD
    // b % 8) until that is empty and then helps with the others'.  Every wave takes its own work:
    // waves of one workgroup that shared a pop waited for the longest rays of all four.
    // Bound by the texture address unit, as the 8x8 rays of a wave touch 32 cache lines a gather
    // (27 cycles each): joint rows of two sources take 5 gathers a step in place of 10.  Measured on
    // MI355X, 12 sub-volumes of sides 32..256 x 4 views at 960x540 in FP16, for the batch: 13.3 ms
    // (one counter of 16x16 tiles for all workgroups, corners clamped at every step, parameter blocks
    // in vector registers), 9.8 ms with these queues and interior steps, 7.9 ms with joint rows.
    // Before joint rows: pops of 2, 4 and 8 quarters 10.1, 11.5 and 13.5 ms; one queue per CU 9.7 ms.
    struct MarchQueues
    {
        uint32_t sx, sy, perFrame, total; // super-tiles of a frame; units of a queue, per frame and in all
    };

    __device__ inline MarchQueues march_queues(uint32_t tilesX, uint32_t tilesY, uint32_t nframes)
    {
        MarchQueues m;
        m.sx = (tilesX + 3u) >> 2;
        m.sy = (tilesY + 3u) >> 2;
        m.perFrame = ((m.sx * m.sy + kMarchQueues - 1u) / kMarchQueues) * 64u;
        m.total = m.perFrame * nframes;
        return m;
    }

    // calls render(frame, tile, quarter) for every unit of the queues that this wave takes
    template<class F>
    __device__ inline void march_work(const MarchQueues& m, uint32_t tilesX, uint32_t tilesY, uint32_t chunk, uint32_t* counters, F render)
    {
        for(uint32_t k = 0; k < kMarchQueues; k++)
        {
            const uint32_t q = (blockIdx.x + k) % kMarchQueues;
            for(;;)
            {
                uint32_t work = 0u;
                if((threadIdx.x & 63u) == 0u)
                    work = atomicAdd(counters + q * kMarchQueueStride, 1u);
                // (in a scalar register: frame, tile and parameter blocks are uniform)
                const uint32_t u0 = uint32_t(__builtin_amdgcn_readfirstlane(int(work))) * chunk;
                if(u0 >= m.total)
                    break;
                const uint32_t u1 = min(u0 + chunk, m.total);
                for(uint32_t u = u0; u < u1; u++)
                {
                    const uint32_t f = u / m.perFrame, r = u - f * m.perFrame;
                    const uint32_t s = q + kMarchQueues * (r >> 6), w = (r >> 2) & 15u;
                    const uint32_t tx = (s % m.sx) * 4u + (w & 3u), ty = (s / m.sx) * 4u + (w >> 2);
                    if(tx < tilesX && ty < tilesY) // (also false where the frame has no super-tile s)
                        render(f, ty * tilesX + tx, r & 3u);
                }
            }
        }
    }

    // All frames of a batch in one persistent launch.  (The parameter blocks come as restrict
    // pointers of their own: their uniform loads then are scalar ones, which the stores of the
    // pixels would otherwise forbid.)
    template<int DT, bool LINEAR, int SIG = 0>
    __global__ __launch_bounds__(256) void batch_march_kernel(
        const FrameParams* __restrict__ frames,
        const PostParams* __restrict__ posts,
        const ParticleParams* __restrict__ parts,
        const uint32_t* __restrict__ order,
        const BatchParams B)
    {
        extern __shared__ float4 lds_lut[];
        stage_luts(lds_lut, posts[0]);
        __syncthreads();
        const MarchQueues m = march_queues(uint32_t(B.tilesX), uint32_t(B.tilesY), uint32_t(B.nframes));
        march_work(m, uint32_t(B.tilesX), uint32_t(B.tilesY), uint32_t(B.chunk), B.counters,
                   [&](uint32_t f, uint32_t tile, uint32_t quarter) __attribute__((always_inline))
                   {
                       const uint32_t item = uint32_t(__builtin_amdgcn_readfirstlane(int(order[f])));
                       brick_march_body<DT, LINEAR, false, SIG>(frames[item], posts[item], parts[item], lds_lut, tile, quarter);
                   });
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
            // joint rows: the pairs of sources that update_buffers joins
#define ISAAC_SIG_JOINT_CASE(dt, k, sg)                                                                                 \
    case dt * 8 + k:                                                                                                    \
        if(Q.joint && natural)                                                                                          \
            hipLaunchKernelGGL((brick_march_sig_kernel<dt, sg + kSigNatural + kSigJoint>), grid, block, lds, s, F, Q, PP); \
        else if(Q.joint)                                                                                                \
            hipLaunchKernelGGL((brick_march_sig_kernel<dt, sg + kSigJoint>), grid, block, lds, s, F, Q, PP);            \
        else if(natural)                                                                                                \
            hipLaunchKernelGGL((brick_march_sig_kernel<dt, sg + kSigNatural>), grid, block, lds, s, F, Q, PP);          \
        else                                                                                                            \
            hipLaunchKernelGGL((brick_march_sig_kernel<dt, sg>), grid, block, lds, s, F, Q, PP);                        \
        return hipGetLastError();
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
                ISAAC_SIG_JOINT_CASE(1, 2, 6)
                ISAAC_SIG_JOINT_CASE(1, 3, 8)
                ISAAC_SIG_JOINT_CASE(1, 4, 16)
                ISAAC_SIG_CASE(2, 0, 1)
                ISAAC_SIG_CASE(2, 1, 3)
                ISAAC_SIG_JOINT_CASE(2, 2, 6)
                ISAAC_SIG_JOINT_CASE(2, 3, 8)
                ISAAC_SIG_JOINT_CASE(2, 4, 16)
#undef ISAAC_SIG_JOINT_CASE
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
        const bool natural = sig_natural(sig), joint = sig_joint(sig);
        sig %= kSigNatural;
        // Compiled signatures: 1, 3 and 1 + 3 components, what batches hold.  Joint rows of 3 + 1 and
        // 1 + 1 components, which the single frame has compiled marches for, take the general one here:
        // 4 sub-volumes of sides 32..128 x 3 views at 480x270 in FP16 1005 us with joint rows and 975 us
        // with rows of their own (3 + 1), 880 us either way (1 + 1), 757 and 806 us for 1 + 3.
        if(linear && (sig == 1 || sig == 3 || sig == 16))
        {
            const int k = dtype * 3 + (sig == 1 ? 0 : sig == 3 ? 1 : 2);
            switch(k)
            {
#define ISAAC_BATCH_LAUNCH(dt, sg)                                                                                      \
    hipLaunchKernelGGL((batch_march_kernel<dt, true, sg>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B)
#define ISAAC_SIG_JOINT_CASE(dt, j, sg)                                                                                 \
    case dt * 3 + j:                                                                                                    \
        if(joint && natural)                                                                                            \
            ISAAC_BATCH_LAUNCH(dt, sg + kSigNatural + kSigJoint);                                                       \
        else if(joint)                                                                                                  \
            ISAAC_BATCH_LAUNCH(dt, sg + kSigJoint);                                                                     \
        else if(natural)                                                                                                \
            ISAAC_BATCH_LAUNCH(dt, sg + kSigNatural);                                                                   \
        else                                                                                                            \
            ISAAC_BATCH_LAUNCH(dt, sg);                                                                                 \
        return hipGetLastError();
#define ISAAC_SIG_CASE(dt, j, sg)                                                                                       \
    case dt * 3 + j:                                                                                                    \
        if(natural)                                                                                                     \
            ISAAC_BATCH_LAUNCH(dt, sg + kSigNatural);                                                                   \
        else                                                                                                            \
            ISAAC_BATCH_LAUNCH(dt, sg);                                                                                 \
        return hipGetLastError();
                ISAAC_SIG_CASE(0, 0, 1)
                ISAAC_SIG_CASE(0, 1, 3)
                ISAAC_SIG_CASE(0, 2, 16)
                ISAAC_SIG_CASE(1, 0, 1)
                ISAAC_SIG_CASE(1, 1, 3)
                ISAAC_SIG_JOINT_CASE(1, 2, 16)
                ISAAC_SIG_CASE(2, 0, 1)
                ISAAC_SIG_CASE(2, 1, 3)
                ISAAC_SIG_JOINT_CASE(2, 2, 16)
#undef ISAAC_SIG_JOINT_CASE
#undef ISAAC_BATCH_LAUNCH
#undef ISAAC_SIG_CASE
            default: break;
            }
        }
        const int v = dtype * 2 + (linear ? 1 : 0);
        switch(v)
        {
        case 0: hipLaunchKernelGGL((batch_march_kernel<0, false>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B); break;
        case 1: hipLaunchKernelGGL((batch_march_kernel<0, true>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B); break;
        case 2: hipLaunchKernelGGL((batch_march_kernel<1, false>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B); break;
        case 3: hipLaunchKernelGGL((batch_march_kernel<1, true>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B); break;
        case 4: hipLaunchKernelGGL((batch_march_kernel<2, false>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B); break;
        default: hipLaunchKernelGGL((batch_march_kernel<2, true>), dim3(grid), dim3(256), lds, s, B.frames, B.posts, B.parts, B.order, B); break;
        }
        return hipGetLastError();
    }
} // namespace isaac_hip
