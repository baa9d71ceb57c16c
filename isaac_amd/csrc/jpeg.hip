// JPEG video frames on the GPU: the frame encoding of serverSendFrame
// (lib/isaac/isaac_communicator.hpp:221-287), which hands the RGBX frame to
// libjpeg-turbo (JCS_EXT_RGBX, jpeg_set_defaults, jpeg_set_quality(q, FALSE)) and
// sends {"payload": "data:image/jpeg;base64,..."}.  The same baseline JPEG,
// byte for byte, as libjpeg-turbo's published algorithm produces it:
//
//   code     one workgroup per 4 MCUs (24 blocks Y00 Y01 Y10 Y11 Cb Cr, 4:2:0): RGB ->
//            YCbCr in 16-bit fixed point, the 2x2 chroma box with alternating bias
//            1, 2, edges replicated (right edge to whole blocks, bottom edge to whole
//            MCU rows), the accurate integer DCT (13-bit constants, 2 extra bits in the
//            row pass), quantisation of DCT/8 by rounding division, zigzag order; blocks
//            past the image are dummies (zero AC, the DC of the last real block before
//            them in the MCU); then the group's Huffman codes as a bit string of its own
//   scan     exclusive prefix sum of the groups' lengths (bit offsets)
//   count    0xFF bytes among the bytes that begin in each group, and their prefix sum
//   file     markers, bytes with 0x00 after every 0xFF, EOI (1-bit padding to a byte)
//   text     for the frame message: prefix, base64 of the file, suffix
//
// The markers (SOI, JFIF APP0, DQT per table, SOF0 -- SOF1 when a table needs 16-bit
// entries --, DHT per table, SOS) come from the host.  Tables: T.81 Annex K.
//
// A 1920x1080 frame is 8 MB in and some 350 KB out, so nothing here is near the
// memory's rate: launches, the two waits of the host (the length has to be known before
// the bytes are fetched) and the fetch itself bound it.  Measured on a 1920x1080 frame
// of quality 90, call to text on the host: 480 us as thirteen launches with one thread
// per block and base64 on the host, 95 us now (kernels 207 -> 44 us).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <initializer_list>
#include <mutex>

#include "isaac_hip.h"

namespace isaac_hip
{
#define JPEG_TABLE(type, name, n) static constexpr type name[n]
#include "jpeg_tables.inc"
#undef JPEG_TABLE

    // Huffman codes, length << 16 | code, of every DC category and AC symbol, both tables
    struct JpegCodes
    {
        uint32_t dc[2][16];
        uint32_t ac[2][256];
    };

    constexpr JpegCodes jpeg_codes()
    {
        JpegCodes H{};
        const uint8_t* bits[4] = {kJpegBits_dc0, kJpegBits_dc1, kJpegBits_ac0, kJpegBits_ac1};
        const uint8_t* vals[4] = {kJpegVals_dc0, kJpegVals_dc1, kJpegVals_ac0, kJpegVals_ac1};
        for(int t = 0; t < 4; t++)
        {
            uint32_t code = 0;
            int k = 0;
            for(uint32_t len = 1; len <= 16; len++)
            {
                for(int i = 0; i < bits[t][len - 1]; i++, k++, code++)
                {
                    const int v = vals[t][k];
                    if(t < 2)
                        H.dc[t][v] = len << 16 | code;
                    else
                        H.ac[t - 2][v] = len << 16 | code;
                }
                code <<= 1;
            }
        }
        return H;
    }

    // Annex K tables in device memory: kernel arguments would be fetched from the host
    // by every workgroup
    static __device__ const JpegCodes jpegCodes = jpeg_codes();

    struct JpegQuant
    {
        uint8_t base[128]; // natural order, luma then chroma
        uint8_t position[64]; // zigzag position of natural index n
    };

    constexpr JpegQuant jpeg_quant()
    {
        JpegQuant Q{};
        for(int i = 0; i < 64; i++)
        {
            Q.base[i] = kJpegQuantLuma[i];
            Q.base[64 + i] = kJpegQuantChroma[i];
            Q.position[kJpegZigzag[i]] = uint8_t(i);
        }
        return Q;
    }

    static __device__ const JpegQuant jpegQuant = jpeg_quant();

    // jpeg_set_quality (jcparam.c): percentage for quality q, table entry from it
    __host__ __device__ inline int32_t jpeg_scale(int32_t quality)
    {
        const int32_t q = quality < 1 ? 1 : (quality > 100 ? 100 : quality);
        return q < 50 ? 5000 / q : 200 - 2 * q;
    }

    __host__ __device__ inline int32_t jpeg_quant_entry(int32_t base, int32_t scale)
    {
        const int32_t v = (base * scale + 50) / 100;
        return v < 1 ? 1 : (v > 32767 ? 32767 : v);
    }

    struct JpegGeom
    {
        int32_t W, H;
        int32_t mcux; // MCUs across
        int32_t ybw, ybh; // Y size in blocks
        int32_t Hg; // rows after completing the last 2-row conversion group
        int32_t scale; // jpeg_scale(quality)
        int64_t nmcu;
    };

    __device__ inline int32_t clampi(int32_t v, int32_t lo, int32_t hi)
    {
        return v < lo ? lo : (v > hi ? hi : v);
    }

    // pixels (x, y) (x + 1, y) (x, y + 1) (x + 1, y + 1), each clamped into the image
    // (edge replication)
    __device__ inline void jpeg_quad(const uint32_t* px, const JpegGeom& G, int x, int y, uint32_t p[4])
    {
        const uint32_t* r0 = px + int64_t(min(y, G.H - 1)) * G.W;
        const uint32_t* r1 = px + int64_t(min(y + 1, G.H - 1)) * G.W;
        if(x + 1 < G.W)
        {
            __builtin_memcpy(p, r0 + x, 8);
            __builtin_memcpy(p + 2, r1 + x, 8);
            return;
        }
        const int xc = G.W - 1;
        p[0] = p[1] = r0[xc];
        p[2] = p[3] = r1[xc];
    }

    // jccolor.c fixed point: FIX(x) = round(x * 2^16)
    constexpr int32_t jfix(double x)
    {
        return int32_t(x * 65536.0 + 0.5);
    }

    __device__ inline int32_t ycc_y(int r, int g, int b)
    {
        return (jfix(0.29900) * r + jfix(0.58700) * g + jfix(0.11400) * b + (1 << 15)) >> 16;
    }
    __device__ inline int32_t ycc_cb(int r, int g, int b)
    {
        return (-jfix(0.16874) * r - jfix(0.33126) * g + jfix(0.5) * b + (128 << 16) + (1 << 15) - 1) >> 16;
    }
    __device__ inline int32_t ycc_cr(int r, int g, int b)
    {
        return (jfix(0.5) * r - jfix(0.41869) * g - jfix(0.08131) * b + (128 << 16) + (1 << 15) - 1) >> 16;
    }

    __device__ inline void jpeg_rgb(uint32_t p, int& r, int& g, int& b)
    {
        r = int(p & 0xffu);
        g = int((p >> 8) & 0xffu);
        b = int((p >> 16) & 0xffu);
    }

    // the 8x8 quad positions of an MCU, one per lane: its 2x2 Y samples and the chroma
    // box.  Chroma rows past the last conversion group repeat its last row.
    struct JpegQuadOut
    {
        int32_t y[4], cb, cr; // already less 128
    };

    __device__ inline JpegQuadOut jpeg_convert(const uint32_t* px, const JpegGeom& G, int mx, int my, int qx, int qy)
    {
        uint32_t p[4];
        const int sy = my * 8 + qy, cy = min(sy, G.Hg / 2 - 1), x = mx * 16 + 2 * qx;
        jpeg_quad(px, G, x, 2 * sy, p);
        JpegQuadOut o;
        int r, g, b;
#pragma unroll
        for(int i = 0; i < 4; i++)
        {
            jpeg_rgb(p[i], r, g, b);
            o.y[i] = ycc_y(r, g, b) - 128;
        }
        if(cy != sy)
            jpeg_quad(px, G, x, 2 * cy, p);
        int32_t sb = 0, sr = 0;
#pragma unroll
        for(int i = 0; i < 4; i++)
        {
            jpeg_rgb(p[i], r, g, b);
            sb += ycc_cb(r, g, b);
            sr += ycc_cr(r, g, b);
        }
        // an MCU is 8 chroma columns wide: the parity of the column is that of qx
        o.cb = ((sb + 1 + (qx & 1)) >> 2) - 128;
        o.cr = ((sr + 1 + (qx & 1)) >> 2) - 128;
        return o;
    }

    // the marker bytes before the entropy-coded data, built in place (at most
    // 20 + 2 * 133 + 19 + 4 * 21 + 348 + 14 = 751 bytes)
    struct JpegHeaders
    {
        uint8_t b[768];
        int32_t n = 0;
        void put(std::initializer_list<uint8_t> v)
        {
            for(uint8_t x : v)
                b[n++] = x;
        }
        void put(const uint8_t* p, size_t k)
        {
            std::memcpy(b + n, p, k);
            n += int32_t(k);
        }
        void push_back(uint8_t x)
        {
            b[n++] = x;
        }
    };

    // jfdctint.c: LL&M integer DCT, constants round(x * 2^13)
    constexpr int32_t dfix(double x)
    {
        return int32_t(x * 8192.0 + 0.5);
    }

    template<bool FIRST>
    __device__ inline void fdct_pass(int32_t* d)
    {
        constexpr int CB = 13, P1 = 2, SH = FIRST ? CB - P1 : CB + P1;
        auto descale = [](int32_t x, int n) { return (x + (1 << (n - 1))) >> n; };
        const int32_t t0 = d[0] + d[7], t7 = d[0] - d[7];
        const int32_t t1 = d[1] + d[6], t6 = d[1] - d[6];
        const int32_t t2 = d[2] + d[5], t5 = d[2] - d[5];
        const int32_t t3 = d[3] + d[4], t4 = d[3] - d[4];
        const int32_t t10 = t0 + t3, t13 = t0 - t3, t11 = t1 + t2, t12 = t1 - t2;
        int32_t o[8];
        if(FIRST)
        {
            o[0] = (t10 + t11) * (1 << P1);
            o[4] = (t10 - t11) * (1 << P1);
        }
        else
        {
            o[0] = descale(t10 + t11, P1);
            o[4] = descale(t10 - t11, P1);
        }
        const int32_t z1 = (t12 + t13) * dfix(0.541196100);
        o[2] = descale(z1 + t13 * dfix(0.765366865), SH);
        o[6] = descale(z1 + t12 * (-dfix(1.847759065)), SH);
        int32_t y1 = t4 + t7, y2 = t5 + t6, y3 = t4 + t6, y4 = t5 + t7;
        const int32_t z5 = (y3 + y4) * dfix(1.175875602);
        const int32_t u4 = t4 * dfix(0.298631336), u5 = t5 * dfix(2.053119869), u6 = t6 * dfix(3.072711026), u7 = t7 * dfix(1.501321110);
        y1 = y1 * (-dfix(0.899976223));
        y2 = y2 * (-dfix(2.562915447));
        y3 = y3 * (-dfix(1.961570560)) + z5;
        y4 = y4 * (-dfix(0.390180644)) + z5;
        o[7] = descale(u4 + y1 + y3, SH);
        o[5] = descale(u5 + y2 + y4, SH);
        o[3] = descale(u6 + y2 + y3, SH);
        o[1] = descale(u7 + y1 + y4, SH);
#pragma unroll
        for(int k = 0; k < 8; k++)
            d[k] = o[k];
    }

    // position in the MCU of the block whose DC block `pos` of MCU (mx, my) has: its own,
    // or for a dummy (only Y blocks of the MCU's right column or bottom row) that of the
    // block before it in the MCU (jccoefct.c), i.e. of the last real one: for (1,1) in a
    // real row (1,0), else (0,1) when that column is real, else (0,0)
    __device__ inline int jpeg_real_pos(const JpegGeom& G, int mx, int my, int pos)
    {
        if(pos >= 4)
            return pos;
        const bool colReal = 2 * mx + 1 < G.ybw, rowReal = 2 * my + 1 < G.ybh;
        if((colReal || !(pos & 1)) && (rowReal || !(pos & 2)))
            return pos;
        if(pos == 3 && rowReal)
            return 2;
        return pos >= 2 && colReal ? 1 : 0;
    }

    __device__ inline int jpeg_nbits(int32_t v)
    {
        const uint32_t a = uint32_t(v < 0 ? -v : v);
        return a ? 32 - __clz(a) : 0;
    }

    // one quantised coefficient: |c| + q/2 over q by a multiplication.  m = floor((2^32 -
    // 1) / q) + 1 exceeds 2^32 / q by e / q, e <= q; the product is exact while (|c| +
    // q/2) * e < 2^32, true for q <= 65536 and |c| <= 8192; above that the quotient is 0
    // and (|c| + q/2) / q <= 0.63, which the excess cannot lift to 1.
    __device__ inline int32_t jpeg_quantise(int32_t c, uint32_t q, uint32_t m)
    {
        const uint32_t a = uint32_t(c < 0 ? -c : c);
        const int32_t r = int32_t(__umulhi(a + (q >> 1), m));
        return c < 0 ? -r : r;
    }

    // 4 MCUs (24 blocks) a workgroup; a block's samples and coefficients are 64 16-bit
    // values at a stride of 72, so that the 8 blocks of a wave start in different banks
    // and every row stays 16-byte aligned.  A block is at most 22 + 63 * 26 bits, its share
    // of the group's bit string (kJpegBlockBytes) has room for 63 * 32 + 27.
    constexpr int kJpegMcus = 4, kJpegStride = 72, kJpegBlockBytes = 256;
    constexpr int kJpegGroupWords = kJpegMcus * 6 * kJpegBlockBytes / 4;

    // Conversion: wave w takes MCU w, a lane the 2x2 pixels of one chroma sample.  Row and
    // column passes, quantisation and coding: 8 lanes a block (3 of the 4 waves), the
    // fourth wave meanwhile forms the DCs of the MCU before the group, which the first DC
    // differences need (the DC of the transform is the sum of the samples), so no group
    // waits for another.  A coefficient's run of zeros follows from the block's 64-bit mask
    // of nonzero coefficients, so the lanes of a block code their 8 coefficients each at
    // the same time, at the offset that a scan over the lanes gives: the order of threads
    // is the order of bits.  (One thread per block, as it was, made 765 waves of 1024 the
    // chip has room for 8 times over, and moved the coefficients through memory three
    // times: 71 + 19 + 47 us at 1920x1080; this kernel: 18 us.)
    __global__ __launch_bounds__(256) void jpeg_code_kernel(const uint32_t* px, const JpegGeom G, uint32_t* slots, uint32_t* groupBits)
    {
        __shared__ __align__(16) int16_t s[kJpegMcus * 6 * kJpegStride];
        __shared__ uint32_t words[kJpegGroupWords + 1];
        __shared__ uint32_t code[2][256], dcCode[2][16], q[128], qm[128], waveBits[4];
        __shared__ int32_t prevDc[3];
        __shared__ uint8_t position[64];
        const int t = threadIdx.x, w = t >> 6, lane = t & 63;
        const int64_t m0 = int64_t(blockIdx.x) * kJpegMcus;
        const int nm = int(min(int64_t(kJpegMcus), G.nmcu - m0));

        code[0][t] = jpegCodes.ac[0][t];
        code[1][t] = jpegCodes.ac[1][t];
        if(t < 32)
            dcCode[t >> 4][t & 15] = jpegCodes.dc[t >> 4][t & 15];
        if(t < 128)
        {
            q[t] = uint32_t(jpeg_quant_entry(jpegQuant.base[t], G.scale)) * 8u;
            qm[t] = 0xffffffffu / q[t] + 1u;
        }
        if(t < 64)
            position[t] = jpegQuant.position[t];
        for(int i = t; i < kJpegGroupWords + 1; i += 256)
            words[i] = 0u;

        if(w < nm)
        {
            const int mx = int((m0 + w) % G.mcux), my = int((m0 + w) / G.mcux), qx = lane & 7, qy = lane >> 3;
            const JpegQuadOut o = jpeg_convert(px, G, mx, my, qx, qy);
            int16_t* sb = s + w * 6 * kJpegStride;
            int16_t* yb = sb + ((qy >> 2) * 2 + (qx >> 2)) * kJpegStride + ((2 * qy) & 7) * 8 + ((2 * qx) & 7);
            *reinterpret_cast<uint32_t*>(yb) = uint32_t(uint16_t(o.y[0])) | uint32_t(o.y[1]) << 16;
            *reinterpret_cast<uint32_t*>(yb + 8) = uint32_t(uint16_t(o.y[2])) | uint32_t(o.y[3]) << 16;
            sb[4 * kJpegStride + lane] = int16_t(o.cb);
            sb[5 * kJpegStride + lane] = int16_t(o.cr);
        }
        __syncthreads();

        const int b = t >> 3, j = t & 7; // block of the group, lane of the block
        const bool coding = b < nm * 6;
        int16_t* blk = s + b * kJpegStride;
        if(coding)
        {
            int32_t d[8];
            int16_t v[8];
            __builtin_memcpy(v, blk + j * 8, 16);
#pragma unroll
            for(int i = 0; i < 8; i++)
                d[i] = v[i];
            fdct_pass<true>(d);
#pragma unroll
            for(int i = 0; i < 8; i++)
                v[i] = int16_t(d[i]);
            __builtin_memcpy(blk + j * 8, v, 16);
        }
        else if(w == 3)
        {
            int32_t sum[3] = {0, 0, 0};
            if(m0 > 0)
            {
                const int mx = int((m0 - 1) % G.mcux), my = int((m0 - 1) / G.mcux), qx = lane & 7, qy = lane >> 3;
                const JpegQuadOut o = jpeg_convert(px, G, mx, my, qx, qy);
                if((qy >> 2) * 2 + (qx >> 2) == jpeg_real_pos(G, mx, my, 3))
                    sum[0] = o.y[0] + o.y[1] + o.y[2] + o.y[3];
                sum[1] = o.cb;
                sum[2] = o.cr;
            }
#pragma unroll
            for(int i = 0; i < 3; i++)
            {
                for(int k = 32; k > 0; k >>= 1)
                    sum[i] += __shfl_xor(sum[i], k);
                const int n = i ? 64 : 0;
                if(lane == 0)
                    prevDc[i] = jpeg_quantise(sum[i], q[n], qm[n]);
            }
        }
        __syncthreads();

        int mcu = 0, pos = 0, real = 0;
        uint32_t lo = 0, hi = 0; // nonzero coefficients by zigzag position
        int32_t d[8];
        uint8_t zp[8];
        if(coding)
        {
            mcu = b / 6;
            pos = b - mcu * 6;
            real = jpeg_real_pos(G, int((m0 + mcu) % G.mcux), int((m0 + mcu) / G.mcux), pos);
#pragma unroll
            for(int i = 0; i < 8; i++)
                d[i] = blk[i * 8 + j];
            fdct_pass<false>(d);
#pragma unroll
            for(int i = 0; i < 8; i++)
            {
                const int n = i * 8 + j, qi = n + (pos < 4 ? 0 : 64);
                d[i] = jpeg_quantise(d[i], q[qi], qm[qi]);
                if(real != pos)
                    d[i] = 0;
                zp[i] = position[n];
                if(d[i] != 0)
                    (zp[i] < 32 ? lo : hi) |= 1u << (zp[i] & 31);
            }
        }
        __syncthreads();
        if(coding)
        {
#pragma unroll
            for(int i = 0; i < 8; i++)
                blk[zp[i]] = int16_t(d[i]);
#pragma unroll
            for(int k = 1; k < 8; k <<= 1)
            {
                lo |= __shfl_xor(lo, k);
                hi |= __shfl_xor(hi, k);
            }
        }
        __syncthreads();

        // codes of coefficients 8 j .. 8 j + 7: value and length of each, with the number
        // of runs of 16 zeros before it
        uint32_t cv[8] = {}, cl[8] = {}, zr[8] = {}, nbits = 0, eob = 0;
        const int tbl = pos < 4 ? 0 : 1;
        if(coding)
        {
            int16_t c[8];
            __builtin_memcpy(c, blk + j * 8, 16);
            const uint64_t mask = uint64_t(hi) << 32 | lo;
            const uint64_t below = (mask & ((1ull << (8 * j)) - 1ull)) | 1ull;
            int last = 63 - __clzll(below);
            const uint32_t zrl = code[tbl][0xF0];
#pragma unroll
            for(int i = 0; i < 8; i++)
            {
                const int k = 8 * j + i;
                uint32_t sym;
                int32_t v = c[i];
                if(k == 0)
                {
                    // the previous block of the component: before it in the MCU, or the
                    // last one of the MCU before
                    auto dcOf = [&](int mc, int p) {
                        const int64_t m = m0 + mc;
                        return int32_t(s[(mc * 6 + jpeg_real_pos(G, int(m % G.mcux), int(m / G.mcux), p)) * kJpegStride]);
                    };
                    const int32_t own = dcOf(mcu, pos);
                    const int32_t before = pos > 0 && pos < 4 ? dcOf(mcu, pos - 1)
                        : mcu > 0                             ? dcOf(mcu - 1, pos == 0 ? 3 : pos)
                                                              : prevDc[pos == 0 ? 0 : pos - 3];
                    v = own - before;
                    sym = dcCode[tbl][jpeg_nbits(v)];
                }
                else
                {
                    if(v == 0)
                        continue;
                    const int run = k - 1 - last;
                    last = k;
                    zr[i] = uint32_t(run) >> 4;
                    nbits += zr[i] * (zrl >> 16);
                    sym = code[tbl][((run & 15) << 4) | jpeg_nbits(v)];
                }
                const int n = jpeg_nbits(v);
                cv[i] = (sym & 0xffffu) << n | (uint32_t(v < 0 ? v - 1 : v) & ((1u << n) - 1u));
                cl[i] = (sym >> 16) + uint32_t(n);
                nbits += cl[i];
            }
            if(j == 7 && !(hi >> 31))
                eob = code[tbl][0];
            nbits += eob >> 16;
        }
        uint32_t incl = nbits;
#pragma unroll
        for(int k = 1; k < 64; k <<= 1)
        {
            const uint32_t o = __shfl_up(incl, k);
            if(lane >= k)
                incl += o;
        }
        if(lane == 63)
            waveBits[w] = incl;
        __syncthreads();
        uint32_t at = incl - nbits;
        for(int i = 0; i < w; i++)
            at += waveBits[i];
        const uint32_t total = waveBits[0] + waveBits[1] + waveBits[2];
        if(nbits)
        {
            auto put = [&](uint32_t v, uint32_t len) {
                const uint64_t x = uint64_t(v) << (64u - (at & 31u) - len);
                atomicOr(words + (at >> 5), uint32_t(x >> 32));
                if(uint32_t(x))
                    atomicOr(words + (at >> 5) + 1, uint32_t(x));
                at += len;
            };
#pragma unroll
            for(int i = 0; i < 8; i++)
            {
                for(uint32_t k = 0; k < zr[i]; k++)
                    put(code[tbl][0xF0] & 0xffffu, code[tbl][0xF0] >> 16);
                if(cl[i])
                    put(cv[i], cl[i]);
            }
            if(eob)
                put(eob & 0xffffu, eob >> 16);
        }
        __syncthreads();
        uint32_t* slot = slots + int64_t(blockIdx.x) * kJpegGroupWords;
        for(uint32_t i = uint32_t(t); i < (total + 31u) / 32u; i += 256u)
            slot[i] = words[i];
        if(t == 0)
            groupBits[blockIdx.x] = total;
    }

    // exclusive prefix sum of n 32-bit counts in one workgroup, a run of entries a thread:
    // one entry per 4 MCUs, 2 a thread at 1920x1080
    __global__ __launch_bounds__(1024) void jpeg_scan_kernel(const uint32_t* in, int64_t n, uint64_t* out, uint64_t* total)
    {
        __shared__ uint64_t waveSum[16];
        const int t = threadIdx.x, lane = t & 63, w = t >> 6;
        const int64_t per = (n + 1023) / 1024, i0 = min(n, per * t), i1 = min(n, i0 + per);
        uint64_t sum = 0;
        for(int64_t i = i0; i < i1; i++)
            sum += in[i];
        uint64_t incl = sum;
#pragma unroll
        for(int k = 1; k < 64; k <<= 1)
        {
            const uint64_t o = __shfl_up(incl, k);
            if(lane >= k)
                incl += o;
        }
        if(lane == 63)
            waveSum[w] = incl;
        __syncthreads();
        uint64_t at = incl - sum;
        for(int i = 0; i < w; i++)
            at += waveSum[i];
        for(int64_t i = i0; i < i1; i++)
        {
            out[i] = at;
            at += in[i];
        }
        if(t == 1023)
            *total = at;
    }

    // the bytes of the coded data that begin in group g: bit string of the group, then the
    // first bits of the next one (an MCU has at least 32 bits, so one is enough) or the
    // 1-bit padding of the last byte.  One wave; word k of the result is bytes first + 4 k
    // .. + 3, most significant byte first.
    struct JpegGroupBytes
    {
        int64_t first; // offset in the coded data
        uint32_t count, shift;
    };

    __device__ inline JpegGroupBytes jpeg_group_bytes(
        const uint32_t* slots, const uint32_t* groupBits, const uint64_t* groupAt, int64_t g, int64_t ngroups, uint32_t* words)
    {
        const uint32_t* slot = slots + g * kJpegGroupWords;
        const uint32_t len = groupBits[g], nw = (len + 31u) / 32u, r = len & 31u;
        const uint64_t at = groupAt[g];
        const uint32_t next = g + 1 < ngroups ? slot[kJpegGroupWords] : 0xffffffffu;
        for(uint32_t k = threadIdx.x; k < nw; k += 64u)
            words[k] = slot[k] | (r && k + 1 == nw ? next >> r : 0u);
        if(threadIdx.x == 0)
            words[nw] = r ? next << (32u - r) : next;
        __syncthreads();
        JpegGroupBytes B;
        B.first = int64_t((at + 7) >> 3);
        B.shift = uint32_t(uint64_t(B.first) * 8u - at);
        B.count = uint32_t(int64_t((at + len + 7) >> 3) - B.first);
        return B;
    }

    __device__ inline uint32_t jpeg_group_word(const uint32_t* words, const JpegGroupBytes& B, uint32_t k)
    {
        return uint32_t((uint64_t(words[k]) << 32 | words[k + 1]) >> (32u - B.shift));
    }

    // 0xFF bytes among the first n (1..4) bytes of a word
    __device__ inline uint32_t jpeg_ff(uint32_t v, uint32_t n)
    {
        uint32_t c = 0;
#pragma unroll
        for(uint32_t i = 0; i < 4; i++)
            c += i < n && ((v >> (24u - 8u * i)) & 0xffu) == 0xffu ? 1u : 0u;
        return c;
    }

    __global__ __launch_bounds__(64) void jpeg_ff_kernel(
        const uint32_t* slots, const uint32_t* groupBits, const uint64_t* groupAt, int64_t ngroups, uint32_t* ff)
    {
        __shared__ uint32_t words[kJpegGroupWords + 1];
        const int64_t g = blockIdx.x;
        const JpegGroupBytes B = jpeg_group_bytes(slots, groupBits, groupAt, g, ngroups, words);
        uint32_t c = 0;
        for(uint32_t k = threadIdx.x; 4u * k < B.count; k += 64u)
            c += jpeg_ff(jpeg_group_word(words, B, k), min(4u, B.count - 4u * k));
        for(int k = 32; k > 0; k >>= 1)
            c += __shfl_xor(c, k);
        if(threadIdx.x == 0)
            ff[g] = c;
    }

    // the file: markers, every byte at its offset plus the 0xFF bytes before it, EOI
    __global__ __launch_bounds__(64) void jpeg_file_kernel(
        const uint32_t* slots, const uint32_t* groupBits, const uint64_t* groupAt, const uint64_t* ffAt, const uint64_t* totals,
        int64_t ngroups, const JpegHeaders hdr, uint8_t* file, int64_t fileCap)
    {
        __shared__ uint32_t words[kJpegGroupWords + 1];
        const int64_t g = blockIdx.x;
        const int64_t end = hdr.n + int64_t((totals[0] + 7) / 8 + totals[1]);
        if(end + 2 > fileCap)
            return;
        const JpegGroupBytes B = jpeg_group_bytes(slots, groupBits, groupAt, g, ngroups, words);
        uint8_t* dst = file + hdr.n + B.first + int64_t(ffAt[g]);
        const int lane = threadIdx.x;
        for(uint32_t k0 = 0; 4u * k0 < B.count; k0 += 64u)
        {
            const uint32_t k = k0 + uint32_t(lane);
            const uint32_t n = 4u * k < B.count ? min(4u, B.count - 4u * k) : 0u;
            const uint32_t v = n ? jpeg_group_word(words, B, k) : 0u, c = jpeg_ff(v, n);
            uint32_t incl = c;
#pragma unroll
            for(int i = 1; i < 64; i <<= 1)
            {
                const uint32_t o = __shfl_up(incl, i);
                if(lane >= i)
                    incl += o;
            }
            uint8_t* p = dst + 4 * lane + (incl - c);
            for(uint32_t i = 0; i < n; i++)
            {
                const uint8_t x = uint8_t(v >> (24u - 8u * i));
                *p++ = x;
                if(x == 0xffu)
                    *p++ = 0u;
            }
            dst += 256u + __shfl(incl, 63);
        }
        if(g == 0)
            for(int i = lane; i < hdr.n; i += 64)
                file[i] = hdr.b[i];
        if(g + 1 == ngroups && lane < 2)
            file[end + lane] = lane ? 0xD9 : 0xFF;
    }

    constexpr char kJpegTextHead[] = "{\"payload\": \"data:image/jpeg;base64,";
    constexpr char kJpegTextTail[] = "\"}";
    constexpr int kJpegHeadLen = sizeof(kJpegTextHead) - 1, kJpegTailLen = sizeof(kJpegTextTail) - 1;
    struct JpegTextEnds
    {
        char head[kJpegHeadLen + 1], tail[kJpegTailLen + 1];
    };

    __device__ inline uint32_t jpeg_base64(uint32_t v)
    {
        return v < 26 ? 'A' + v : v < 52 ? 'a' + (v - 26) : v < 62 ? '0' + (v - 52) : v == 62 ? '+' : '/';
    }

    // the frame message around base64 as boost's iterators produce it: 6 bits at a time,
    // zero-filled tail, no '='.  A thread turns 12 bytes of the file into 16 characters;
    // chars is 16-byte aligned, the head lies before it.  Bytes past the file's end are
    // masked (the workspace goes on behind its space).
    __global__ __launch_bounds__(256) void jpeg_text_kernel(
        const uint8_t* file, int64_t fileCap, int64_t headerBytes, const uint64_t* totals, const JpegTextEnds ends, uint8_t* chars,
        int64_t charCap)
    {
        const int64_t n = headerBytes + int64_t((totals[0] + 7) / 8 + totals[1]) + 2, nc = (8 * n + 5) / 6;
        if(n > fileCap || nc + 16 > charCap)
            return;
        for(int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x; 16 * i < nc; i += int64_t(gridDim.x) * 256)
        {
            uint32_t d[3], o[4];
            __builtin_memcpy(d, file + 12 * i, 12);
            const int64_t left = n - 12 * i;
#pragma unroll
            for(int k = 0; k < 3; k++)
            {
                const int64_t l = left - 4 * k;
                d[k] = l >= 4 ? d[k] : l <= 0 ? 0u : d[k] & ((1u << (8 * l)) - 1u);
            }
            const uint32_t t[4] = {
                __builtin_bswap32(d[0]) >> 8,
                (d[0] >> 24) << 16 | (d[1] & 0xffu) << 8 | ((d[1] >> 8) & 0xffu),
                ((d[1] >> 16) & 0xffu) << 16 | (d[1] >> 24) << 8 | (d[2] & 0xffu),
                __builtin_bswap32(d[2]) & 0xffffffu};
#pragma unroll
            for(int k = 0; k < 4; k++)
                o[k] = jpeg_base64(t[k] >> 18) | jpeg_base64((t[k] >> 12) & 63u) << 8 | jpeg_base64((t[k] >> 6) & 63u) << 16
                    | jpeg_base64(t[k] & 63u) << 24;
            if(16 * i + 16 <= nc)
                __builtin_memcpy(chars + 16 * i, o, 16);
            else
                for(int k = 0; 16 * i + k < nc; k++)
                    chars[16 * i + k] = uint8_t(o[k >> 2] >> (8 * (k & 3)));
        }
        if(blockIdx.x == 0)
        {
            if(threadIdx.x < kJpegHeadLen)
                chars[int(threadIdx.x) - kJpegHeadLen] = uint8_t(ends.head[threadIdx.x]);
            if(threadIdx.x < kJpegTailLen)
                chars[nc + threadIdx.x] = uint8_t(ends.tail[threadIdx.x]);
        }
    }

    // jpeg_set_quality (jcparam.c): natural-order table entries for quality q
    void jpeg_quality_tables(int quality, int out[2][64])
    {
        const int32_t scale = jpeg_scale(quality);
        for(int i = 0; i < 64; i++)
        {
            out[0][i] = jpeg_quant_entry(kJpegQuantLuma[i], scale);
            out[1][i] = jpeg_quant_entry(kJpegQuantChroma[i], scale);
        }
    }

    // A workspace's pieces.  Every symbol (code and extra bits) is at most 26 bits and 22
    // for the DC, so a block is at most 1660 bits.  Every code has a 0 bit, and no sequence of
    // symbols makes more than 31 ones in a row (15 before the 0 of a code at its front, 6 at
    // its end and 10 extra bits), so at most 3 of 4 bytes in a row are 0xFF, and the file is
    // at most 1660 / 8 * 1.75 < 364 bytes a block, its base64 text 485.4, both without the
    // markers.  The text takes the place of the bit strings, which are dead by then.
    struct JpegLayout
    {
        int64_t nblocks, nmcu, ngroups, fileCap, charCap;
        size_t groupAt, ffAt, totals, groupBits, ff, file, slots, chars, end;
    };

    JpegLayout jpeg_layout(int32_t width, int32_t height)
    {
        JpegLayout L{};
        L.nmcu = int64_t((width + 15) / 16) * ((height + 15) / 16);
        L.nblocks = L.nmcu * 6;
        L.ngroups = (L.nmcu + kJpegMcus - 1) / kJpegMcus;
        auto a = [](size_t v) { return (v + 255) & ~size_t(255); };
        L.groupAt = 0;
        L.ffAt = L.groupAt + size_t(L.ngroups) * 8;
        L.totals = L.ffAt + size_t(L.ngroups) * 8;
        L.groupBits = L.totals + 16;
        L.ff = L.groupBits + size_t(L.ngroups) * 4;
        L.fileCap = (L.nblocks * 364 + 800 + 15) & ~int64_t(15);
        L.file = a(L.ff + size_t(L.ngroups) * 4);
        L.slots = (L.file + size_t(L.fileCap) + 63) & ~size_t(63);
        L.chars = L.slots + 64; // the message's head before it
        // what callers are told to bring (and the noalloc limit is stated in) for a frame
        const int64_t maxBytes = L.nblocks * 256 + 8, nscan = (L.nblocks + 1023) / 1024, nstuff = (maxBytes + 1023) / 1024;
        L.end = a(size_t(L.nblocks) * 128) + a(size_t(L.nblocks) * 4) + a(size_t(L.nblocks) * 8) + a(size_t(nscan) * 8 + 8) + a(8)
            + a(size_t(maxBytes + 8)) + a(size_t(nstuff) * 4) + a(size_t(nstuff) * 8 + 8) + a(size_t((nstuff + 1023) / 1024) * 8 + 8)
            + a(size_t(maxBytes) * 2 + 16);
        L.charCap = int64_t(L.end - L.chars);
        return L;
    }

    // the markers before the entropy-coded data (jcmarker.c order)
    void jpeg_headers(int32_t width, int32_t height, const int qt[2][64], JpegHeaders& h)
    {
        h.n = 0;
        h.put({0xFF, 0xD8, 0xFF, 0xE0, 0x00, 0x10, 'J', 'F', 'I', 'F', 0x00, 0x01, 0x01, 0x00, 0x00, 0x01, 0x00, 0x01, 0x00, 0x00});
        bool wide = false;
        for(int t = 0; t < 2; t++)
        {
            bool w16 = false;
            for(int i = 0; i < 64; i++)
                w16 = w16 || qt[t][i] > 255;
            wide = wide || w16;
            h.put({0xFF, 0xDB, 0x00, uint8_t(w16 ? 0x83 : 0x43), uint8_t((w16 ? 0x10 : 0x00) | t)});
            for(int k = 0; k < 64; k++)
            {
                const int v = qt[t][kJpegZigzag[k]];
                if(w16)
                    h.push_back(uint8_t(v >> 8));
                h.push_back(uint8_t(v & 0xff));
            }
        }
        h.put({0xFF, uint8_t(wide ? 0xC1 : 0xC0), 0x00, 0x11, 0x08, uint8_t(height >> 8), uint8_t(height & 0xff),
               uint8_t(width >> 8), uint8_t(width & 0xff), 0x03, 0x01, 0x22, 0x00, 0x02, 0x11, 0x01, 0x03, 0x11, 0x01});
        const uint8_t* bits[4] = {kJpegBits_dc0, kJpegBits_ac0, kJpegBits_dc1, kJpegBits_ac1};
        const uint8_t* vals[4] = {kJpegVals_dc0, kJpegVals_ac0, kJpegVals_dc1, kJpegVals_ac1};
        const uint8_t cls[4] = {0x00, 0x10, 0x01, 0x11};
        for(int t = 0; t < 4; t++)
        {
            int n = 0;
            for(int i = 0; i < 16; i++)
                n += bits[t][i];
            const int len = 3 + 16 + n;
            h.put({0xFF, 0xC4, uint8_t(len >> 8), uint8_t(len & 0xff), cls[t]});
            h.put(bits[t], 16);
            h.put(vals[t], size_t(n));
        }
        h.put({0xFF, 0xDA, 0x00, 0x0C, 0x03, 0x01, 0x00, 0x02, 0x11, 0x03, 0x11, 0x00, 0x3F, 0x00});
    }

    bool jpeg_size_ok(int32_t width, int32_t height)
    {
        return width >= 1 && height >= 1 && width <= 65535 && height <= 65535;
    }

    bool jpeg_workspace_ok(const void* rgbx, const void* workspace, int64_t bytes, const JpegLayout& L)
    {
        return bytes >= int64_t(L.end) && !(reinterpret_cast<uintptr_t>(rgbx) & 3u) && !(reinterpret_cast<uintptr_t>(workspace) & 255u);
    }

    // the kernels over a workspace laid out by jpeg_layout (L), arguments checked: the
    // file, and its message text if `text`; *fileLength: the file's length, waited for
    int jpeg_run(const uint8_t* rgbx, int32_t width, int32_t height, int32_t quality, uint8_t* ws, const JpegLayout& L, bool text,
                 int64_t* fileLength, hipStream_t s)
    {
        uint32_t* slots = reinterpret_cast<uint32_t*>(ws + L.slots);
        uint32_t* groupBits = reinterpret_cast<uint32_t*>(ws + L.groupBits);
        uint32_t* ff = reinterpret_cast<uint32_t*>(ws + L.ff);
        uint64_t* groupAt = reinterpret_cast<uint64_t*>(ws + L.groupAt);
        uint64_t* ffAt = reinterpret_cast<uint64_t*>(ws + L.ffAt);
        uint64_t* totals = reinterpret_cast<uint64_t*>(ws + L.totals);

        JpegGeom G{};
        G.W = width;
        G.H = height;
        G.mcux = (width + 15) / 16;
        G.ybw = (width + 7) / 8;
        G.ybh = (height + 7) / 8;
        G.Hg = height + (height & 1);
        G.scale = jpeg_scale(quality);
        G.nmcu = L.nmcu;
        int qt[2][64];
        jpeg_quality_tables(quality, qt);
        JpegHeaders hdr;
        jpeg_headers(width, height, qt, hdr);

        const dim3 groups{unsigned(L.ngroups)};
        hipLaunchKernelGGL(jpeg_code_kernel, groups, dim3(256), 0, s, reinterpret_cast<const uint32_t*>(rgbx), G, slots, groupBits);
        hipLaunchKernelGGL(jpeg_scan_kernel, dim3(1), dim3(1024), 0, s, groupBits, L.ngroups, groupAt, totals);
        hipLaunchKernelGGL(jpeg_ff_kernel, groups, dim3(64), 0, s, slots, groupBits, groupAt, L.ngroups, ff);
        hipLaunchKernelGGL(jpeg_scan_kernel, dim3(1), dim3(1024), 0, s, ff, L.ngroups, ffAt, totals + 1);
        hipLaunchKernelGGL(jpeg_file_kernel, groups, dim3(64), 0, s, slots, groupBits, groupAt, ffAt, totals, L.ngroups, hdr,
                           ws + L.file, L.fileCap);
        if(text)
        {
            JpegTextEnds ends;
            std::memcpy(ends.head, kJpegTextHead, sizeof(ends.head));
            std::memcpy(ends.tail, kJpegTextTail, sizeof(ends.tail));
            // about 8 bytes a block are coded at usual qualities: a thread for every 2 blocks
            const unsigned grid = unsigned(std::min<int64_t>((L.nblocks + 511) / 512, 4096));
            hipLaunchKernelGGL(jpeg_text_kernel, dim3(grid), dim3(256), 0, s, ws + L.file, L.fileCap, int64_t(hdr.n), totals, ends,
                               ws + L.chars, L.charCap);
        }
        if(hipGetLastError() != hipSuccess)
            return ISAAC_HIP_ERR_DEVICE;
        uint64_t t[2] = {0, 0}; // coded bits, 0xFF bytes
        if(hipMemcpyAsync(t, totals, 16, hipMemcpyDeviceToHost, s) != hipSuccess || hipStreamSynchronize(s) != hipSuccess)
            return ISAAC_HIP_ERR_DEVICE;
        *fileLength = hdr.n + int64_t((t[0] + 7) / 8 + t[1]) + 2;
        return *fileLength <= L.fileCap && (8 * *fileLength + 5) / 6 + 16 <= L.charCap ? 0 : ISAAC_HIP_ERR_DEVICE;
    }

    int jpeg_fetch(void* dst, const void* src, int64_t bytes, hipStream_t s)
    {
        return hipMemcpyAsync(dst, src, size_t(bytes), hipMemcpyDeviceToHost, s) == hipSuccess && hipStreamSynchronize(s) == hipSuccess
            ? 0
            : ISAAC_HIP_ERR_DEVICE;
    }

    int encode(const uint8_t* rgbx, int32_t width, int32_t height, int32_t quality, uint8_t* ws, const JpegLayout& L,
               uint8_t* jpeg, int64_t capacity, int64_t* length, hipStream_t s)
    {
        int64_t n = 0;
        const int rc = jpeg_run(rgbx, width, height, quality, ws, L, false, &n, s);
        if(rc)
            return rc;
        *length = n;
        if(capacity < n)
            return ISAAC_HIP_ERR_ARG;
        return jpeg_fetch(jpeg, ws + L.file, n, s);
    }

    // The workspace of isaac_hip_jpeg_encode_noalloc: a device array that every GPU
    // holds from the library's load to the end of the process.  Host code uses it only
    // through the address hipGetSymbolAddress returns for the current device (the
    // array's name in host code is a stand-in, not a device address).
    static_assert(ISAAC_HIP_JPEG_NOALLOC_SCRATCH_BYTES % 256 == 0, "scratch size");
    static __device__ __align__(256) uint8_t scratch[ISAAC_HIP_JPEG_NOALLOC_SCRATCH_BYTES];

    constexpr int kMaxScratchDevices = 64;
    std::mutex scratchLock;
    uint8_t* scratchAddr[kMaxScratchDevices] = {};

    // the scratch's address on the current device, looked up once per device
    int scratch_on_current_device(uint8_t** out)
    {
        int dev = -1;
        if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxScratchDevices)
            return ISAAC_HIP_ERR_DEVICE;
        std::lock_guard<std::mutex> guard(scratchLock);
        if(!scratchAddr[dev])
        {
            void* p = nullptr;
            if(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p)
                return ISAAC_HIP_ERR_DEVICE;
            scratchAddr[dev] = static_cast<uint8_t*>(p);
        }
        *out = scratchAddr[dev];
        return 0;
    }
} // namespace isaac_hip

using namespace isaac_hip;

extern "C"
{
    int64_t isaac_hip_jpeg_workspace_bytes(int32_t width, int32_t height)
    {
        if(!jpeg_size_ok(width, height))
            return -1;
        return int64_t(jpeg_layout(width, height).end);
    }

    int isaac_hip_jpeg_encode(
        const uint8_t* rgbx,
        int32_t width,
        int32_t height,
        int32_t quality,
        void* workspace,
        int64_t workspace_bytes,
        uint8_t* jpeg,
        int64_t capacity,
        int64_t* length,
        void* stream)
    {
        if(!rgbx || !workspace || !jpeg || !length || !jpeg_size_ok(width, height))
            return ISAAC_HIP_ERR_ARG;
        const JpegLayout L = jpeg_layout(width, height);
        if(!jpeg_workspace_ok(rgbx, workspace, workspace_bytes, L))
            return ISAAC_HIP_ERR_ARG;
        return encode(rgbx, width, height, quality, static_cast<uint8_t*>(workspace), L, jpeg, capacity, length,
                      (hipStream_t) stream);
    }

    int isaac_hip_jpeg_encode_noalloc(
        const uint8_t* rgbx,
        int32_t width,
        int32_t height,
        int32_t quality,
        uint8_t* jpeg,
        int64_t capacity,
        int64_t* length,
        void* stream)
    {
        if(!rgbx || !jpeg || !length || !jpeg_size_ok(width, height)
           || (reinterpret_cast<uintptr_t>(rgbx) & 3u))
            return ISAAC_HIP_ERR_ARG;
        const JpegLayout L = jpeg_layout(width, height);
        if(L.end > size_t(ISAAC_HIP_JPEG_NOALLOC_SCRATCH_BYTES))
            return ISAAC_HIP_ERR_ARG;
        const hipStream_t s = (hipStream_t) stream;
        int dev = -1, sdev = -1;
        if(hipGetDevice(&dev) != hipSuccess)
            return ISAAC_HIP_ERR_DEVICE;
        if(s && (hipStreamGetDevice(s, &sdev) != hipSuccess || sdev != dev))
            return ISAAC_HIP_ERR_ARG; // the scratch of another GPU than the stream's
        uint8_t* ws = nullptr;
        const int rc = scratch_on_current_device(&ws);
        if(rc)
            return rc;
        return encode(rgbx, width, height, quality, ws, L, jpeg, capacity, length, s);
    }

    int isaac_hip_jpeg_frame_message(
        const uint8_t* rgbx,
        int32_t width,
        int32_t height,
        int32_t quality,
        void* workspace,
        int64_t workspace_bytes,
        char* msg,
        int64_t capacity,
        int64_t* length,
        void* stream)
    {
        if(!msg || !length || width < 1 || height < 1)
            return ISAAC_HIP_ERR_ARG;
        if(!rgbx || !workspace || !jpeg_size_ok(width, height))
            return ISAAC_HIP_ERR_ARG;
        const JpegLayout L = jpeg_layout(width, height);
        if(!jpeg_workspace_ok(rgbx, workspace, workspace_bytes, L))
            return ISAAC_HIP_ERR_ARG;
        uint8_t* ws = static_cast<uint8_t*>(workspace);
        int64_t n = 0;
        const int rc = jpeg_run(rgbx, width, height, quality, ws, L, true, &n, (hipStream_t) stream);
        if(rc)
            return rc;
        *length = kJpegHeadLen + (8 * n + 5) / 6 + kJpegTailLen;
        if(capacity < *length + 1)
            return ISAAC_HIP_ERR_ARG;
        msg[*length] = '\0';
        return jpeg_fetch(msg, ws + L.chars - kJpegHeadLen, *length, (hipStream_t) stream);
    }
}
