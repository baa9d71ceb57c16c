// The brick form's data: volume sources re-laid into 8^3 bricks of x-pairs with a scale per
// brick and component (common.hpp, "precision form"), each on its own or two as joint rows.
#include "render_device.hpp"

namespace isaac_hip
{
    __device__ inline uint32_t to_bf16_rne(float f)
    {
        const uint32_t u = __float_as_uint(f);
        if((u & 0x7f800000u) == 0x7f800000u)
            return (u >> 16) | ((u & 0xffffu) ? 0x40u : 0u); // inf / nan
        return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
    }

    // v / s rounded to 16 bits; r = RN(1/s), 0 where s is outside [2^-60, 2^60] (there the
    // quotient takes the IEEE division).  x*r plus one fma residual step (div_by), with v's
    // sign (the residual step turns -0 into +0): the IEEE quotient for |v| <= s with s in
    // [2^-60, 2^60]; for BF16, whose range keeps tiny quotients, only where |v| >= 2^-60
    // (the residual stays normal).
    template<int DT>
    __device__ inline uint16_t brick_quotient(float v, float s, float r)
    {
        const bool fast = r != 0.0f && (DT == kDtF16 || fabsf(v) >= 0x1p-60f);
        const float q = fast ? copysignf(div_by(v, s, r), v) : v / s;
        return uint16_t(DT == kDtF16 ? uint32_t(__half_as_ushort(__float2half_rn(q))) : to_bf16_rne(q));
    }

    template<int N>
    struct Floats
    {
        float v[N];
    };

    // One workgroup per brick: every thread loads up to 3 voxels of the brick's 9^3 region (x,
    // y, z clamped to the local box) with all W = D0 + D1 components of the one or two sources,
    // the maxima of |v| become the scales (1 when the region is all zero or the form is FP32),
    // each voxel is divided and rounded once, in registers, and passes through LDS in its
    // stored form, from which the pairs (v[x], v[x+1]) are written row by row, all components
    // of a row in one store.  Output row brick*648 + pair, pair = (lz*9 + ly)*8 + lx.
    // Bound by memory: a 256^3 scalar and 3-component source in FP16 are 268 MB in and 340 MB
    // out, 119 us at the copy rate; 145 us (254 us with a launch per source, both ends of
    // every pair divided and rounded, 4-byte loads and stores; 192 us before the bricks of an
    // XCD were neighbours).
    template<int DT, int D0, int D1>
    __global__ __launch_bounds__(256) void brick_build_kernel(
        const BrickBuildSource a, const BrickBuildSource b, int X, int Y, int Z, int nbx, int nby, int nbricks, float* scale, void* out)
    {
        constexpr int W = D0 + D1, kVoxels = 729, N = (kVoxels + 255) / 256;
        using Stored = typename std::conditional<DT == kDtF32, float, uint16_t>::type;
        struct __align__(W == 3 ? sizeof(Stored) : W * sizeof(Stored)) Voxel
        {
            Stored v[W];
        };
        __shared__ Voxel reg[kVoxels];
        __shared__ float part[4][W], sc[W], rc[W];
        const int t = threadIdx.x;
        // workgroup b runs on XCD b % 8: each XCD takes a run of bricks, so the cache lines that
        // neighbouring bricks share (a line holds 4 bricks' rows of a scalar) meet in one L2
        const unsigned perXcd = (unsigned(nbricks) + 7u) / 8u, index = (blockIdx.x & 7u) * perXcd + (blockIdx.x >> 3);
        if(index >= unsigned(nbricks))
            return;
        const int64_t brick = index;
        const int Bx = int(index % unsigned(nbx)), By = int(index / unsigned(nbx) % unsigned(nby)), Bz = int(index / unsigned(nbx) / unsigned(nby));
        float v[N][W], m[W];
#pragma unroll
        for(int c = 0; c < W; c++)
            m[c] = 0.0f;
#pragma unroll
        for(int n = 0; n < N; n++)
        {
            const int i = min(t + n * 256, kVoxels - 1), row = i / 9, lx = i - row * 9, lz = row / 9, ly = row - lz * 9;
            const int64_t x = min(Bx * 8 + lx, X - 1), y = min(By * 8 + ly, Y - 1), z = min(Bz * 8 + lz, Z - 1);
            const Floats<D0> p = *reinterpret_cast<const Floats<D0>*>(a.src + (x * a.stride[0] + y * a.stride[1] + z * a.stride[2]) * D0);
#pragma unroll
            for(int c = 0; c < D0; c++)
                v[n][c] = p.v[c];
            if constexpr(D1 > 0)
            {
                const Floats<D1> q = *reinterpret_cast<const Floats<D1>*>(b.src + (x * b.stride[0] + y * b.stride[1] + z * b.stride[2]) * D1);
#pragma unroll
                for(int c = 0; c < D1; c++)
                    v[n][D0 + c] = q.v[c];
            }
        }
        if constexpr(DT != kDtF32)
        {
#pragma unroll
            for(int c = 0; c < W; c++)
            {
#pragma unroll
                for(int n = 0; n < N; n++)
                    m[c] = fmaxf(m[c], fabsf(v[n][c]));
#pragma unroll
                for(int off = 32; off > 0; off >>= 1)
                    m[c] = fmaxf(m[c], __shfl_xor(m[c], off));
                if((t & 63) == 0)
                    part[t >> 6][c] = m[c];
            }
            __syncthreads();
        }
        if(t < W)
        {
            float s = 1.0f;
            if constexpr(DT != kDtF32)
            {
                const float mx = fmaxf(fmaxf(part[0][t], part[1][t]), fmaxf(part[2][t], part[3][t]));
                s = mx > 0.0f ? mx : 1.0f;
            }
            sc[t] = s;
            rc[t] = (s >= 0x1p-60f && s <= 0x1p+60f) ? 1.0f / s : 0.0f;
            scale[brick * W + t] = s;
        }
        __syncthreads();
#pragma unroll
        for(int n = 0; n < N; n++)
        {
            Voxel o;
#pragma unroll
            for(int c = 0; c < W; c++)
            {
                if constexpr(DT == kDtF32)
                    o.v[c] = v[n][c];
                else
                    o.v[c] = brick_quotient<DT>(v[n][c], sc[c], rc[c]);
            }
            if(t + n * 256 < kVoxels)
                reg[t + n * 256] = o;
        }
        __syncthreads();
        constexpr int kWords = DT == kDtF32 ? 2 * W : W;
        struct __align__(kWords == 3 || kWords == 6 ? 4 : (kWords == 8 ? 16 : 4 * kWords)) Row
        {
            uint32_t w[kWords];
        };
        Row* rows = static_cast<Row*>(out) + brick * kBrickPairs;
        for(int e = t; e < kBrickPairs; e += 256)
        {
            const int vox = (e >> 3) * 9 + (e & 7);
            const Voxel lo = reg[vox], hi = reg[vox + 1];
            Row r;
#pragma unroll
            for(int c = 0; c < W; c++)
            {
                if constexpr(DT == kDtF32)
                {
                    r.w[2 * c] = __float_as_uint(lo.v[c]);
                    r.w[2 * c + 1] = __float_as_uint(hi.v[c]);
                }
                else
                    r.w[c] = uint32_t(lo.v[c]) | uint32_t(hi.v[c]) << 16;
            }
            rows[e] = r;
        }
    }

    template<int DT>
    hipError_t launch_brick_build(
        const BrickBuildSource* src, int nsources, int X, int Y, int Z, int nbx, int nby, int64_t nbricks, float* scale, void* out,
        hipStream_t s)
    {
        const dim3 grid = dim3(static_cast<unsigned>((nbricks + 7) / 8 * 8)), block = dim3(256);
        const BrickBuildSource a = src[0], b = nsources == 2 ? src[1] : BrickBuildSource{};
        switch(nsources * 100 + a.dim * 10 + b.dim)
        {
#define ISAAC_BRICK_CASE(k, d0, d1)                                                                                     \
    case k: hipLaunchKernelGGL((brick_build_kernel<DT, d0, d1>), grid, block, 0, s, a, b, X, Y, Z, nbx, nby, int(nbricks), scale, out); break;
            ISAAC_BRICK_CASE(110, 1, 0)
            ISAAC_BRICK_CASE(120, 2, 0)
            ISAAC_BRICK_CASE(130, 3, 0)
            ISAAC_BRICK_CASE(140, 4, 0)
            ISAAC_BRICK_CASE(211, 1, 1)
            ISAAC_BRICK_CASE(213, 1, 3)
            ISAAC_BRICK_CASE(231, 3, 1)
#undef ISAAC_BRICK_CASE
        default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    }

    hipError_t launch_bricks(
        const BrickBuildSource* sources, int nsources, int X, int Y, int Z, int dtype, float* scale, void* out, hipStream_t s)
    {
        const int nbx = (X + 7) / 8, nby = (Y + 7) / 8, nbz = (Z + 7) / 8;
        const int64_t nbricks = int64_t(nbx) * nby * nbz;
        if(nbricks == 0)
            return hipSuccess;
        if(nbricks > int64_t(0x7fffffff))
            return hipErrorInvalidValue;
        if(dtype == kDtF32)
            return nsources == 1 ? launch_brick_build<kDtF32>(sources, 1, X, Y, Z, nbx, nby, nbricks, scale, out, s) : hipErrorInvalidValue;
        if(dtype == kDtF16)
            return launch_brick_build<kDtF16>(sources, nsources, X, Y, Z, nbx, nby, nbricks, scale, out, s);
        return launch_brick_build<kDtBf16>(sources, nsources, X, Y, Z, nbx, nby, nbricks, scale, out, s);
    }

    // a source's own rows and scales out of joint ones (on request only)
    __global__ __launch_bounds__(256) void brick_split_kernel(
        const uint32_t* joint, const float* jointScale, int jointDim, int at, int dim, int64_t nrows, int64_t nbricks, uint32_t* out,
        float* scale)
    {
        for(int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; i < nrows; i += int64_t(gridDim.x) * 256)
            for(int c = 0; c < dim; c++)
            {
                out[i * dim + c] = joint[i * jointDim + at + c];
                if(i < nbricks)
                    scale[i * dim + c] = jointScale[i * jointDim + at + c];
            }
    }

    hipError_t launch_brick_split(
        const void* joint, const float* jointScale, int jointDim, int at, int dim, int64_t nbricks, void* out, float* scale, hipStream_t s)
    {
        const int64_t nrows = nbricks * kBrickPairs;
        if(nrows == 0)
            return hipSuccess;
        const unsigned grid = unsigned(std::min<int64_t>((nrows + 255) / 256, 8192));
        hipLaunchKernelGGL(brick_split_kernel, dim3(grid), dim3(256), 0, s, static_cast<const uint32_t*>(joint), jointScale, jointDim,
                           at, dim, nrows, nbricks, static_cast<uint32_t*>(out), scale);
        return hipGetLastError();
    }
} // namespace isaac_hip
