// Shift convolutions and shift GEMMs on the matrix cores (int8 sparse MFMA, int32 accumulation), exact modulo 2^32.
//
// A term sgn * (x >> s) is not linear in x, but it is a short sum of products of 8-bit numbers.  With x written in
// 7-bit digits, x = d0 + 2^7 d1 + 2^14 d2 + 2^21 d3 + 2^28 d4 (d0, d1 in 0..127, the others balanced), and
// s = 7 q + r, 0 <= r < 7:
//     x >> s = (d_q >> r) + sum_{i > q} d_i * 2^(6-r) * 2^(7(i-q-1)+1)
//     64 * (d_q >> r) = sum_j (bit j of d_q, in place) * [r <= j] 2^(6-r)
// i.e. bit masks of a digit (one AND per four activations) times weight planes that hold 0 or a signed power of two
// up to 64 -- all of them int8 -- plus products of whole digits with the full weight plane of their q.  A weight has one
// q: of the digits d0 and d1 it meets one, of d1 and d2 (next power) one, and so on.  That is the matrix cores' 2:4
// sparsity: with digits (d0, d1) of each activation side by side, a weight is one of the two places, the index of
// v_smfmac_i32_32x32x64_i8 says which, and one instruction does for both q what took two.  A weight is stored as its
// index and one or two selector bytes (r <= 3 and r >= 4), from which one v_perm_b32 per four weights makes any plane;
// 12 selects the constant 0.  Shifts to 14 take 10 products per term (7 for the bits, one each for the two powers above
// them, one for s = 14; 2 more where a digit d3 is not zero), to 6 six, to 3 four: there the pair is one digit twice,
// masked differently for small and large r.  8-bit activations: x >> s selected from the pair (x, x >> 4), four products,
// or (x, x >> 2), two.
//
// Measured (us, dense products of one digit each -> this; 64 images, 3 x 3 layers, with their hand-off): shifts to 14, 64
// channels of 56 x 56: 107 -> 91, 512 of 7 x 7: 105 -> 78, with digit d3 164 -> 119 and 175 -> 107; 8-bit activations 63 ->
// 48 and 62 -> 39.  4096^3: 772 -> 551 us, 125 Tpair/s.  What bounds it is power: a loop of one product and seven vector
// instructions takes 28 ns (68 clocks of 2.4 GHz, of which the matrix core needs 32) on random bytes, 21 on bit planes and
// 26 on whole digits, whatever the number of waves; 4096^3 takes 27.  Sparse and dense products cost the same (22 ns alone
// on random bytes), so the number of products is what counts.
//
// Activations are laid out first (ds_mfma_prepare): [image][row][32-channel block][digits 0 and 1 in pairs, 2, 3, 4][column]
// [channels], so that the 32 pixels x 32 channels of one operand are a KiB in a row, two for the pairs; d3 and d4 are
// written, and read, only where one of them is not zero (|x| >= 16 in 16.16): flags tell it per row and share of its
// channels or, where the convolution before wrote the layout from its epilogue, per 32 of its pixels x 16 channels.
#include "ds_common.h"
#include "ds_epilogue.h"

namespace ds {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));

constexpr int kDigits = 5;          // 7-bit digits of an int32 activation
constexpr int kMfmaMaxK = 1 << 17;  // 64 * 127 * K stays within int32
constexpr int kMaxRows = 1 << 24;   // ds_mfma_prepare launches 256 threads per row, and a launch has less than 2^32
constexpr int kMaxParts = 1 << 15;  // of a row in ds_mfma_prepare; a launch has less than 2^16 workgroups along y
constexpr int kMaxPad = 1 << 28;

// Which products a launch forms (MfmaMode): the widest shift that occurs, and the activations' width.
enum { kI32S15 = 0, kI32S7 = 1, kI32S4 = 2, kI8S8 = 3, kI8S4 = 4 };
// Selector bytes per weight, and bytes of a 32-channel tile's share of one block: the selectors, then 4 bytes of indices
// per lane (which of two activation bytes each weight meets).
__host__ __device__ constexpr int mode_sels(int mode) { return mode == kI32S15 || mode == kI32S7 ? 2 : 1; }
__host__ __device__ constexpr int mode_block(int mode) { return mode_sels(mode) * 1024 + 256; }
__host__ __device__ constexpr bool mode_i8(int mode) { return mode >= kI8S8; }

// The reduction in blocks of 32 activation bytes that lie side by side: 32 channels of one tap, or, where a pixel has
// at most 16 channels, 32 / cp taps of one filter row (cp channels each).
struct MfmaGeom {
    int cp, cb, taps, fwg, kb, ntiles;
};
inline MfmaGeom mfma_geom(int N, int C, int FH, int FW)
{
    MfmaGeom g;
    g.cp = C <= 4 ? 4 : C <= 8 ? 8 : C <= 16 ? 16 : 32;
    if (FH * FW == 1) g.cp = 32;
    g.cb = ceil_div(C, g.cp);
    g.taps = 32 / g.cp;
    g.fwg = ceil_div(FW, g.taps);
    g.kb = g.cb * FH * g.fwg;
    g.ntiles = ceil_div(N, 64) * 2;
    return g;
}
inline size_t mfma_blob_corr(const MfmaGeom &g, int mode) { return (size_t)g.ntiles * g.kb * mode_block(mode); }

// One thread per (channel tile, block, lane): the selector bytes of its 16 weights, and which byte of a pair each meets.
// Weight i of lane l is reduction index 16 (i / 8) + 8 (l / 32) + i % 8 of the block: the half i / 8 of the wave holds the
// activations that it meets, 16 indices in a row.
__global__ __launch_bounds__(256) void mfma_tile_kernel(const int32_t *__restrict__ w_ref, int8_t *__restrict__ blob, int N,
                                                        int C, int FH, int FW, int bits, int mode, int cp, int cb,
                                                        int taps, int fwg, int kb, long total)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int lane = (int)(t & 63);
    const long tile_kb = t >> 6;
    const int b = (int)(tile_kb % kb), tile = (int)(tile_kb / kb);
    const int fg = b % fwg, fh = b / fwg % FH, c0 = b / fwg / FH * cp;
    const int n = tile * 32 + (lane & 31);
    const int K = C * FH * FW, num = codes_per_word(bits), comm = ceil_div(K, num);
    uint32_t sel[2][4], index = 0;
    for (int g = 0; g < 2; ++g)
        for (int w = 0; w < 4; ++w) sel[g][w] = 0x0c0c0c0cu;
    for (int i = 0; i < 16; ++i) {
        index |= (uint32_t)(2 * (i & 1)) << (2 * i);
        const int kk = (i >> 3) * 16 + (lane >> 5) * 8 + (i & 7);
        const int c = c0 + kk % cp, fw = fg * taps + kk / cp;
        if (n >= N || c >= C || fw >= FW) continue;
        const int k = (c * FH + fh) * FW + fw;
        const uint32_t code = (uint32_t)w_ref[(long)n * comm + k / num] >> ((k % num) * (bits + 1));
        uint32_t s = code & ((1u << bits) - 1u);
        const uint32_t neg = ((code >> bits) & 1u) ? 0u : 4u;
        if (s >= 32) continue;  // a zero weight
        uint32_t g = 0, l, second;   // selector, its value, the second byte of the pair
        if (mode == kI8S8) {
            s = s < 7 ? s : 7;
            l = s & 3;
            second = s >> 2;
        } else if (mode == kI8S4) {
            l = s & 1;
            second = s >> 1;
        } else if (mode == kI32S4) {
            l = s;
            second = s >> 1;
        } else {
            const uint32_t q = s / 7, r = s - 7 * q;
            g = q == 2 || r >= 4 ? 1 : 0;
            l = q == 2 ? 3 : r & 3;
            second = mode == kI32S7 ? g : q & 1;
        }
        if (l > 3 || second > 1) continue;  // the caller vouches that it does not occur
        index |= second << (2 * i);
        const int at = (i & 3) * 8;
        sel[g][i >> 2] = (sel[g][i >> 2] & ~(255u << at)) | ((l | neg) << at);
    }
    int8_t *o = blob + tile_kb * mode_block(mode);
    for (int g = 0; g < mode_sels(mode); ++g) {
        v4i v;
        for (int w = 0; w < 4; ++w) v[w] = (int)sel[g][w];
        *(v4i *)(o + g * 1024 + lane * 16) = v;
    }
    *(uint32_t *)(o + mode_sels(mode) * 1024 + lane * 4) = index;
}

// Per channel, what the offset of the second byte of 8-bit activations adds (offset 8 for x >> 4, 32 for x >> 2):
// sum_k sgn * (offset >> (s - 4 or 2)) over the shifts that take it.
__global__ __launch_bounds__(64) void mfma_corr_kernel(const int32_t *__restrict__ w_ref, int32_t *__restrict__ corr, int N,
                                                       int K, int bits, int mode)
{
    const int n = blockIdx.x, num = codes_per_word(bits), comm = ceil_div(K, num);
    const uint32_t from = mode == kI8S8 ? 4 : 2, offset = mode == kI8S8 ? 8 : 32;
    int sum = 0;
    if (n < N)
        for (int k = threadIdx.x; k < K; k += 64) {
            const uint32_t code = (uint32_t)w_ref[(long)n * comm + k / num] >> ((k % num) * (bits + 1));
            uint32_t s = code & ((1u << bits) - 1u);
            if (s < from || s >= 32) continue;
            s = s < 7 ? s : 7;
            const int v = (int)(offset >> (s - from));
            sum += ((code >> bits) & 1u) ? v : -v;
        }
    for (int o = 32; o; o >>= 1) sum += __shfl_xor(sum, o);
    if (threadIdx.x == 0) corr[n] = sum;
}

// ---------------------------------------------------------------------------------------------
// activations -> operand layout
// ---------------------------------------------------------------------------------------------

// Layout of the prepared activations, shared by the pass that writes them and the contraction.
struct MfmaX {
    int Hp, Wp, cp, cb, digits;
    int dstride, cbstride, rstride;  // bytes between digits, 32-channel blocks, rows
    int px01, half01, piece01;       // digits 0 and 1, side by side: bytes between pixels, halves of a wave, pieces of a block
    int fy, cbf;                     // flag bytes per row, channel blocks that each of them covers
    int tiles, th, tw, tph, tpw;     // written by a convolution: one flag per 32 of its th x tw pixels and 16 channels
    int c16;
    long rows;
    size_t planes;                   // bytes of the digits; the flags follow
};
inline MfmaX mfma_x(int Nb, int C, int Hp, int Wp, const MfmaGeom &g, bool i8)
{
    MfmaX x;
    x.Hp = Hp;
    x.Wp = Wp;
    x.cp = g.cp;
    x.cb = g.cb;
    x.digits = i8 ? 1 : kDigits;
    x.dstride = Wp * g.cp;
    x.cbstride = x.dstride * x.digits;
    x.rstride = x.cbstride * g.cb;
    x.px01 = g.cp == 32 ? 32 : 2 * g.cp;
    x.half01 = g.cp == 32 ? 16 : 32;
    x.piece01 = g.cp == 32 ? x.dstride : 16;
    x.rows = (long)Nb * Hp;
    // as many channel blocks of a row per workgroup as its threads take at a go (mfma_prepare_kernel)
    const int per_block = Wp * (g.cp == 32 ? 2 : 1);
    x.cbf = per_block >= 256 ? 1 : 256 / per_block < g.cb ? 256 / per_block : g.cb;
    if (x.cbf < ceil_div(g.cb, kMaxParts)) x.cbf = ceil_div(g.cb, kMaxParts);
    x.fy = ceil_div(g.cb, x.cbf);
    // a block of several taps may read up to 32 bytes past the last pixel
    x.planes = align_up((size_t)x.rows * x.rstride + 64, 256);
    x.tiles = 0;
    x.c16 = ceil_div(C, 16);
    return x;
}

enum { kSrcF32 = 0, kSrcI32 = 1, kSrcI8 = 2 };

struct PrepArgs {
    const void *x;
    int8_t *dst;
    uint8_t *flags;
    MfmaX lay;
    int C, H, W, ph, pw;
    int M, K;        // rows of a matrix: image n holds rows 64 n .. 64 n + 63, C = K
    int vec;         // a matrix of 32-bit values whose rows can be read four at a time
    int per, rpw;    // items of a row's part, rows per workgroup
    FastDiv by_per, by_wp, by_hp;
    QuantSpec spec;
};

template <int CH>
__device__ __forceinline__ void quantize_many(const int32_t (&raw)[CH], int32_t (&v)[CH], const QuantSpec &spec)
{
    // one look at the mode, not one per value
    QuantSpec s = spec;
    if (spec.mode == DS_Q_CAST) {
        s.mode = DS_Q_CAST;
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = quantize_one(__int_as_float(raw[i]), s);
    } else if (spec.I == 1) {
        s.mode = DS_Q_ROUND_TO_FIXED;
        s.I = 1;
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = quantize_one(__int_as_float(raw[i]), s);
    } else {
        s.mode = DS_Q_ROUND_TO_FIXED;
        s.I = 2;   // the bounds are in lo and hi
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = quantize_one(__int_as_float(raw[i]), s);
    }
}

__device__ __forceinline__ void digits_of(int32_t v, int32_t d[kDigits])
{
    const int32_t b = v >> 14;
    d[0] = v & 127;
    d[1] = (v >> 7) & 127;
    d[2] = (int32_t)((uint32_t)b << 25) >> 25;
    const int32_t c = (b - d[2]) >> 7;
    d[3] = (int32_t)((uint32_t)c << 25) >> 25;
    d[4] = (c - d[3]) >> 7;
}

// Digits 0 and 1 of a value in two bytes.
__device__ __forceinline__ uint32_t pair01(int32_t v) { return ((uint32_t)v & 127u) | (((uint32_t)v << 1) & 0x7f00u); }

// CH channels of one pixel: what a thread of mfma_prepare_kernel converts.  All values are asked for before the first is
// converted; outside the image some value that is there, so that no load waits behind a branch.
template <int SRC, bool MATRIX, int CH>
__device__ __forceinline__ void prep_values(const PrepArgs &a, int n, int h, int wp, int c0, int32_t (&v)[CH])
{
    int32_t raw[CH];
    bool in;
    if (MATRIX) {
        const int m = n * 64 + wp;
        in = m < a.M;
        const size_t base = (size_t)(in ? m : 0) * a.K;
        if (SRC == kSrcI8) {
#pragma unroll
            for (int i = 0; i < CH; ++i) raw[i] = ((const int8_t *)a.x)[base + (c0 + i < a.K ? c0 + i : 0)];
        } else if (a.vec) {
            // rows and base aligned: four values per load
#pragma unroll
            for (int q = 0; q < CH / 4; ++q) {
                const int c = c0 + 4 * q;
                const v4i r = *(const v4i *)((const int32_t *)a.x + base + (c < a.K ? c : 0));
#pragma unroll
                for (int i = 0; i < 4; ++i) raw[4 * q + i] = r[i];
            }
        } else {
#pragma unroll
            for (int i = 0; i < CH; ++i)
                raw[i] = ((const int32_t *)a.x)[base + (c0 + i < a.K ? c0 + i : 0)];
        }
    } else {
        const int w = wp - a.pw;
        in = (unsigned)h < (unsigned)a.H && (unsigned)w < (unsigned)a.W;
        const size_t plane = (size_t)a.H * a.W;
        const size_t base = (size_t)n * a.C * plane + (in ? (size_t)h * a.W + w : 0);
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const size_t at = base + (c0 + i < a.C ? c0 + i : a.C - 1) * plane;
            raw[i] = SRC == kSrcI8 ? ((const int8_t *)a.x)[at] : ((const int32_t *)a.x)[at];
        }
    }
    if (SRC == kSrcF32)
        quantize_many<CH>(raw, v, a.spec);
    else
#pragma unroll
        for (int i = 0; i < CH; ++i) v[i] = raw[i];
#pragma unroll
    for (int i = 0; i < CH; ++i)
        if (!in || c0 + i >= a.C) v[i] = 0;
}

// Words to an address of any four bytes, in one store.
template <int N>
__device__ __forceinline__ void store_words(int8_t *o, const uint32_t (&w)[N])
{
    typedef uint32_t words __attribute__((ext_vector_type(N), aligned(4)));
    words v;
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = w[i];
    *(words *)o = v;
}

// A thread converts CH channels of one pixel, two threads side by side for the halves of a 32-channel block, so that loads
// run along the row and stores are contiguous; a workgroup takes the blocks of one part of a row, or of several rows where
// they are short.  Bound by memory: 4 bytes read and 3 written per element (5 where a digit d3 or d4 of the row's part is not
// zero: they wait in registers until the workgroup knows; rows of more than 256 items are read a second time for them).
// Before, every value was loaded behind its own bounds check and waited for, and a workgroup had one row: us then and now,
// with the ordinary range and, second, with d3 in every row: 64 images of 64 x 56 x 56, 3 x 3: 33 and 21 (4.4 TB/s), 55 and
// 23; 256 of 16 x 32 x 32: 42 and 9, 61 and 10; 128 of 256 x 56 x 56, unpadded: 295 and 152 (4.7 TB/s).
template <int SRC, bool I8, bool MATRIX, int CH>
__global__ __launch_bounds__(256) void mfma_prepare_kernel(PrepArgs a)
{
    __shared__ int seen[256];   // of a row: 1, d3 or d4; 2, d4
    const MfmaX &L = a.lay;
    const int part = blockIdx.y;
    const int halves = CH == 16 && L.cp == 32 ? 2 : 1;
    const int cb0 = part * L.cbf, cb1 = cb0 + L.cbf < L.cb ? cb0 + L.cbf : L.cb;
    const int items = (cb1 - cb0) * L.Wp * halves;   // of a row
    const int r = a.rpw == 1 ? 0 : (int)div_by(threadIdx.x, a.by_per);
    const int first = (int)threadIdx.x - r * a.per;
    const long at = (long)blockIdx.x * a.rpw + r;
    const bool on = r < a.rpw && at < L.rows && first < items;
    const uint32_t row = (uint32_t)(on ? at : 0);
    const int n = (int)div_by(row, a.by_hp), h = (int)row - n * L.Hp - a.ph;
    int8_t *dst = a.dst + (size_t)row * L.rstride;
    constexpr int Q = CH / 4;

    // Item t: its digits 0 to 2 (or its 8-bit values) stored if `low`; the others left in w3, w4, to be stored at `o`.
    const auto convert = [&](int t, bool low, int8_t *&o, uint32_t (&w3)[Q], uint32_t (&w4)[Q]) {
        const int half = halves == 2 ? t & 1 : 0;
        const uint32_t tw = halves == 2 ? t >> 1 : t;
        const int cbi = (int)div_by(tw, a.by_wp), wp = (int)tw - cbi * L.Wp, cb = cb0 + cbi;
        int32_t v[CH];
        prep_values<SRC, MATRIX, CH>(a, n, h, wp, cb * L.cp + half * CH, v);
        o = dst + (size_t)cb * L.cbstride + wp * L.cp + half * CH;
        uint32_t w2[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            w2[q] = w3[q] = w4[q] = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (I8) {
                    w2[q] |= ((uint32_t)v[q * 4 + i] & 255u) << (8 * i);
                    continue;
                }
                int32_t dg[kDigits];
                digits_of(v[q * 4 + i], dg);
                w2[q] |= ((uint32_t)dg[2] & 255u) << (8 * i);
                w3[q] |= ((uint32_t)dg[3] & 255u) << (8 * i);
                w4[q] |= ((uint32_t)dg[4] & 255u) << (8 * i);
            }
        }
        if (low) {
            store_words<Q>(o + (I8 ? 0 : 2) * L.dstride, w2);
            if (!I8) {
                // digits 0 and 1 in pairs, eight channels a piece
                int8_t *o01 = dst + (size_t)cb * L.cbstride + wp * L.px01 + half * L.half01;
                constexpr int P = CH < 8 ? CH / 2 : 4;
#pragma unroll
                for (int p = 0; p < CH / 2 / P; ++p) {
                    uint32_t pairs[P];
#pragma unroll
                    for (int i = 0; i < P; ++i) pairs[i] = pair01(v[(p * P + i) * 2]) | pair01(v[(p * P + i) * 2 + 1]) << 16;
                    store_words<P>(o01 + p * L.piece01, pairs);
                }
            }
        }
        int high = 0;
#pragma unroll
        for (int q = 0; q < Q; ++q) high |= w4[q] ? 3 : w3[q] ? 1 : 0;
        return high;
    };
    const auto store_high = [&](int8_t *o, const uint32_t (&w3)[Q], const uint32_t (&w4)[Q]) {
        store_words<Q>(o + 3 * L.dstride, w3);
        store_words<Q>(o + 4 * L.dstride, w4);
    };

    if (!I8) {
        if ((int)threadIdx.x < a.rpw) seen[threadIdx.x] = 0;
        __syncthreads();
    }
    int8_t *o = nullptr;
    uint32_t w3[Q], w4[Q];
    int high = 0;
    if (a.per <= 256) {
        if (on) high = convert(first, true, o, w3, w4);
    } else {
        for (int t = first; t < items; t += 256) high |= convert(t, true, o, w3, w4);
    }
    if (I8) return;
    if (high) atomicOr(&seen[r], high);
    __syncthreads();
    if (!on) return;
    const int any = seen[r];
    if (first == 0) a.flags[(size_t)row * L.fy + part] = (uint8_t)any;
    if (!any) return;
    if (a.per <= 256) {
        store_high(o, w3, w4);
    } else {
        for (int t = first; t < items; t += 256) {
            convert(t, false, o, w3, w4);
            store_high(o, w3, w4);
        }
    }
}

// ---------------------------------------------------------------------------------------------
// the contraction
// ---------------------------------------------------------------------------------------------

struct MfmaArgs {
    const int8_t *x;
    const uint8_t *flags;
    const int8_t *blob;
    const int32_t *corr, *bias;
    int32_t *y;                 // int32 sums, or
    float *out;                 // the float result and / or
    void *q;                    // the next layer's input
    const float *scale, *shift, *residual;
    MfmaX lay;
    int N, KB, FH, fwg, tapstep, tapstep01;
    int OH, OW, sh, sw, crop_h, crop_w;
    uint32_t pixels;
    int ks, tc, ctiles;         // K parts, channel tiles per workgroup, workgroups along channels
    uint32_t whole, tail_tile;  // workgroups that this holds for; the others share tiles of pixels from tail_tile on four ways
    long ostride_n;
    int ostride_c;
    int matrix;                 // pixels are matrix rows
    MfmaX qlay;                 // q in the operand layout of the next layer (qlay.planes != 0)
    uint8_t *qflags;
    int relu, q_bytes, qHp, qWp, qph, qpw;
    float inv;
    // the shorter epilogue: 2^F of the sums, 2^F of q if nothing else is written (q_only)
    float unfold, qfold;
    int q_only;
    QuantSpec qspec;
    // at odd multiples of 4 bytes the layers of 8-bit networks took 0.7 % more, those of ResNet-20 0.6 %
    alignas(8) FastDiv by_image, by_row, by_ctiles;
};

__device__ __forceinline__ v4i perm4(uint32_t neg, uint32_t pos, v4i sel)
{
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (int)__builtin_amdgcn_perm(neg, pos, (uint32_t)sel[i]);
    return r;
}
__device__ __forceinline__ v4i and4(v4i v, uint32_t m)
{
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = v[i] & (int)m;
    return r;
}
__device__ __forceinline__ v4i or4(v4i a, v4i b)
{
    v4i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = a[i] | b[i];
    return r;
}

// Look-up words of the weight planes: byte l = the value of the group's l-th shift, for positive and negative weights.
constexpr uint32_t kPosLo = 0x08102040u, kNegLo = 0xf8f0e0c0u;   // r = 0..3: 64, 32, 16, 8
constexpr uint32_t kPosHi = 0x00010204u, kNegHi = 0x00fffefcu;   // r = 4..6: 4, 2, 1
constexpr uint32_t kPos14 = 0x40000000u, kNeg14 = 0xc0000000u;   // s = 14, the last of its group: 64
__host__ __device__ constexpr uint32_t low_bytes(uint32_t v, int n) { return n >= 4 ? v : v & ((1u << (8 * n)) - 1u); }

typedef int v8i __attribute__((ext_vector_type(8)));

// What a wave holds of one block: CT x 32 channels, NT x 32 pixels.  lo: digits 0 and 1 in pairs, or the 8-bit values.
template <int MODE, int CT, int NT, bool HIGH>
struct Operands {
    static constexpr int S = mode_sels(MODE), L = mode_i8(MODE) ? 1 : 2;
    v4i sel[CT][S];
    int index[CT];
    v4i lo[NT][L];
    v4i d2[mode_i8(MODE) ? 1 : NT], d3[HIGH ? NT : 1];
    uint32_t on[HIGH ? NT : 1];   // the flag of d3, and whether its place is inside the image
    bool in[HIGH ? NT : 1];
};

template <int CT, int NT>
__device__ __forceinline__ void product(v16i (&acc)[CT][NT], const v4i (&w)[CT], const v8i (&b)[NT], const int (&index)[CT])
{
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int p = 0; p < NT; ++p)
            acc[c][p] = __builtin_amdgcn_smfmac_i32_32x32x64_i8(w[c], b[p], acc[c][p], index[c], 0, 0);
}
template <int CT>
__device__ __forceinline__ void weights(v4i (&w)[CT], uint32_t neg, uint32_t pos, const v4i (&sel)[CT])
{
#pragma unroll
    for (int c = 0; c < CT; ++c) w[c] = perm4(neg, pos, sel[c]);
}
template <int CT>
__device__ __forceinline__ void both(v4i (&w)[CT], const v4i (&a)[CT], const v4i (&b)[CT])
{
#pragma unroll
    for (int c = 0; c < CT; ++c) w[c] = or4(a[c], b[c]);
}
__device__ __forceinline__ v8i and8(const v8i &v, uint32_t m)
{
    v8i r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = v[i] & (int)m;
    return r;
}
__device__ __forceinline__ v8i join8(const v4i &a, const v4i &b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }
// Pairs of bytes: byte i of a beside byte i of b (16 activations).
__device__ __forceinline__ v8i pairs_of(const v4i &a, const v4i &b)
{
    v8i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[2 * i] = (int)__builtin_amdgcn_perm((uint32_t)b[i], (uint32_t)a[i], 0x05010400u);
        r[2 * i + 1] = (int)__builtin_amdgcn_perm((uint32_t)b[i], (uint32_t)a[i], 0x07030602u);
    }
    return r;
}
__device__ __forceinline__ v8i pairs_with_zero(const v4i &a)
{
    v8i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[2 * i] = (int)__builtin_amdgcn_perm(0u, (uint32_t)a[i], 0x0c010c00u);
        r[2 * i + 1] = (int)__builtin_amdgcn_perm(0u, (uint32_t)a[i], 0x0c030c02u);
    }
    return r;
}
// Digit 1 of pairs (0, 1) beside digit 2.
__device__ __forceinline__ v8i pairs12(const v8i &p01, const v4i &d2)
{
    v8i r;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        r[2 * i] = (int)__builtin_amdgcn_perm((uint32_t)d2[i], (uint32_t)p01[2 * i], 0x05030401u);
        r[2 * i + 1] = (int)__builtin_amdgcn_perm((uint32_t)d2[i], (uint32_t)p01[2 * i + 1], 0x07030601u);
    }
    return r;
}

// The sums of a tile: bits (times 64), and whole digits by power of two, 2^(7 i + 1).
template <int CT, int NT, bool HIGH>
struct Sums {
    v16i bits[CT][NT], d[HIGH ? 3 : 2][CT][NT];
};

// Shifts to 14.  s = 7 q + r: the first byte of each pair is q's digit 0, the second digit 1, and so on up; q = 2 meets
// first bytes only, in products of its own.
template <int CT, int NT, bool HIGH, typename Reload>
__device__ __forceinline__ void block_s15(const Operands<kI32S15, CT, NT, HIGH> &o, Sums<CT, NT, HIGH> &t, Reload reload)
{
    v8i x01[NT], b[NT];
    v4i w[CT], wlo[CT], slo[CT], shi[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        slo[c] = o.sel[c][0];
        shi[c] = o.sel[c][1];
    }
#pragma unroll
    for (int p = 0; p < NT; ++p) x01[p] = join8(o.lo[p][0], o.lo[p][1]);
#pragma unroll
    for (int j = 0; j < 7; ++j) {
        // r <= 3: bits 3 to 6 meet the same weights; r >= 4: bits 4, 5, 6 one by one
        if (j <= 3)
            weights<CT>(w, low_bytes(kNegLo, j + 1), low_bytes(kPosLo, j + 1), slo);
        else
            weights<CT>(w, low_bytes(kNegHi, j - 3), low_bytes(kPosHi, j - 3), shi);
#pragma unroll
        for (int p = 0; p < NT; ++p) b[p] = and8(x01[p], j == 3 ? 0x78787878u : 0x01010101u << j);
        product<CT, NT>(t.bits, w, b, o.index);
        if (j == 3) {
#pragma unroll
            for (int c = 0; c < CT; ++c) wlo[c] = w[c];
        }
    }
    both<CT>(wlo, wlo, w);
    int index[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) index[c] = o.index[c];
#pragma unroll
    for (int p = 0; p < NT; ++p) b[p] = pairs12(x01[p], o.d2[p]);
    product<CT, NT>(t.d[0], wlo, b, o.index);
    weights<CT>(w, kNeg14, kPos14, shi);
    if constexpr (HIGH) {
        v8i b3[NT];
#pragma unroll
        for (int p = 0; p < NT; ++p) {
            const v4i d3 = and4(o.d3[p], o.in[p] && o.on[p] ? 0xffffffffu : 0u);
            b[p] = pairs_of(o.d2[p], d3);
            b3[p] = pairs_with_zero(d3);
        }
        reload();
        product<CT, NT>(t.d[1], wlo, b, index);
        product<CT, NT>(t.bits, w, b, index);
        product<CT, NT>(t.d[2], wlo, b3, index);
        product<CT, NT>(t.d[0], w, b3, index);
    } else {
#pragma unroll
        for (int p = 0; p < NT; ++p) b[p] = pairs_with_zero(o.d2[p]);
        reload();
        product<CT, NT>(t.d[1], wlo, b, index);
        product<CT, NT>(t.bits, w, b, index);
    }
}

// Shifts to 6 or to 3: every weight meets digit 0; the pair is that digit twice, masked differently for small and large
// shifts.
template <int MODE, int CT, int NT, bool HIGH, typename Reload>
__device__ __forceinline__ void block_s7(const Operands<MODE, CT, NT, HIGH> &o, Sums<CT, NT, HIGH> &t, Reload reload)
{
    v8i x01[NT], x0[NT], b[NT];
    v4i w[CT], full[CT], slo[CT], shi[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        slo[c] = o.sel[c][0];
        shi[c] = o.sel[c][mode_sels(MODE) - 1];
    }
#pragma unroll
    for (int p = 0; p < NT; ++p) {
        x01[p] = join8(o.lo[p][0], o.lo[p][1]);
#pragma unroll
        for (int i = 0; i < 8; ++i) x0[p][i] = (int)__builtin_amdgcn_perm(0u, (uint32_t)x01[p][i], 0x02020000u);
    }
    if constexpr (MODE == kI32S4) {
        // shifts 0, 1 beside 2, 3: bit 0 for a shift of 0 beside bit 2 for one of 2, then the rest of both
#pragma unroll
        for (int p = 0; p < NT; ++p) b[p] = and8(x0[p], 0x04010401u);
        weights<CT>(w, kNegLo & 0x00ff00ffu, kPosLo & 0x00ff00ffu, slo);
        product<CT, NT>(t.bits, w, b, o.index);
#pragma unroll
        for (int p = 0; p < NT; ++p) b[p] = and8(x0[p], 0x787e787eu);
        weights<CT>(full, kNegLo, kPosLo, slo);
        product<CT, NT>(t.bits, full, b, o.index);
    } else {
        // shifts 0 to 3 beside 4 to 6: bits j beside bits 4 + j, then bits 3 to 6 of the former
        v4i hi[CT];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            weights<CT>(w, low_bytes(kNegLo, j + 1), low_bytes(kPosLo, j + 1), slo);
            if (j < 3) {
                weights<CT>(hi, low_bytes(kNegHi, j + 1), low_bytes(kPosHi, j + 1), shi);
                v4i sum[CT];
                both<CT>(sum, w, hi);
#pragma unroll
                for (int p = 0; p < NT; ++p) b[p] = and8(x0[p], 0x10011001u << j);
                product<CT, NT>(t.bits, sum, b, o.index);
            } else {
#pragma unroll
                for (int p = 0; p < NT; ++p) b[p] = and8(x0[p], 0x00780078u);
                product<CT, NT>(t.bits, w, b, o.index);
            }
        }
        both<CT>(full, w, hi);
    }
    // whole digits: first or second bytes of pairs (1, 2), (3, 0) for all weights
    int first[CT], second[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        first[c] = (int)0x88888888u;
        second[c] = (int)0xddddddddu;
    }
#pragma unroll
    for (int p = 0; p < NT; ++p) b[p] = pairs12(x01[p], o.d2[p]);
    if constexpr (HIGH) {
        v8i b3[NT];
#pragma unroll
        for (int p = 0; p < NT; ++p) b3[p] = pairs_with_zero(and4(o.d3[p], o.in[p] && o.on[p] ? 0xffffffffu : 0u));
        reload();
        product<CT, NT>(t.d[2], full, b3, first);
    } else {
        reload();
    }
    product<CT, NT>(t.d[0], full, b, first);
    product<CT, NT>(t.d[1], full, b, second);
}

// 8-bit activations: x >> s = (y >> l), y the value itself for small shifts, x >> 4 (or >> 2) with an offset that makes it
// positive for large ones: a pair of bytes, of which every shift l takes the upper 8 - l bits.
template <int MODE, int CT, int NT>
__device__ __forceinline__ void block_i8(const Operands<MODE, CT, NT, false> &o, v16i (&acc)[CT][NT])
{
    constexpr int S = MODE == kI8S8 ? 4 : 2;
    v8i x[NT], b[NT];
    v4i w[CT], sel[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) sel[c] = o.sel[c][0];
#pragma unroll
    for (int p = 0; p < NT; ++p) {
        v4i y;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            y[i] = MODE == kI8S8 ? (int)((((uint32_t)o.lo[p][0][i] >> 4) & 0x0f0f0f0fu) ^ 0x08080808u)
                                 : (int)((((uint32_t)o.lo[p][0][i] >> 2) & 0x3f3f3f3fu) ^ 0x20202020u);
        x[p] = pairs_of(o.lo[p][0], y);
    }
#pragma unroll
    for (int l = 0; l < S; ++l) {
        constexpr uint32_t pos = MODE == kI8S8 ? 0x01020408u : 0x0102u, neg = MODE == kI8S8 ? 0xfffefcf8u : 0xfffeu;
        weights<CT>(w, neg & (0xffu << (8 * l)), pos & (0xffu << (8 * l)), sel);
#pragma unroll
        for (int p = 0; p < NT; ++p) b[p] = l == 0 ? x[p] : and8(x[p], ((0xffu << l) & 0xffu) * 0x01010101u);
        product<CT, NT>(acc, w, b, o.index);
    }
}

// Position in the reduction: blocks run over (32-channel block, filter row, group of taps), the last fastest.
struct KPos {
    int cb, fh, fg, off, off01;
};

__device__ __forceinline__ void k_start(const MfmaArgs &a, KPos &k, int kb)
{
    const int per = a.FH * a.fwg;
    k.cb = kb / per;
    const int rest = kb - k.cb * per;
    k.fh = rest / a.fwg;
    k.fg = rest - k.fh * a.fwg;
    const int row = k.cb * a.lay.cbstride + k.fh * a.lay.rstride;
    k.off = row + k.fg * a.tapstep;
    k.off01 = row + k.fg * a.tapstep01;
}
__device__ __forceinline__ void k_next(const MfmaArgs &a, KPos &k)
{
    k.off += a.tapstep;
    k.off01 += a.tapstep01;
    if (++k.fg == a.fwg) {
        k.fg = 0;
        int step = a.lay.rstride;
        if (++k.fh == a.FH) {
            k.fh = 0;
            ++k.cb;
            step += a.lay.cbstride - a.FH * a.lay.rstride;
        }
        k.off += step - a.fwg * a.tapstep;
        k.off01 += step - a.fwg * a.tapstep01;
    }
}

struct PixelAt {
    uint32_t n, oh, ow;
};
__device__ __forceinline__ PixelAt pixel_at(const MfmaArgs &a, uint32_t p)
{
    PixelAt r;
    r.n = div_by(p, a.by_image);
    const uint32_t rem = p - r.n * a.by_image.d;
    r.oh = div_by(rem, a.by_row);
    r.ow = rem - r.oh * a.by_row.d;
    return r;
}

// The flag of digits d3 and d4 for the 16 bytes that a lane reads at a block: where it lies, and whether they are inside
// the image (some flag that is there if they are not, so that no load waits behind a branch).
__device__ __forceinline__ const uint8_t *high_flag(const MfmaArgs &a, const PixelAt &at, int half, const KPos &k, bool &in)
{
    const int ih = at.oh * a.sh + a.crop_h + k.fh;
    in = true;
    if (!a.lay.tiles) return a.flags + ((size_t)at.n * a.lay.Hp + ih) * a.lay.fy + k.cb / a.lay.cbf;
    const int iw = at.ow * a.sw + a.crop_w + (a.lay.cp == 16 ? k.fg * 2 + half : k.fg) - a.lay.tpw;
    const int h = ih - a.lay.tph;
    const int ch16 = a.lay.cp == 16 ? k.cb : k.cb * 2 + half;
    in = (unsigned)h < (unsigned)a.lay.th && (unsigned)iw < (unsigned)a.lay.tw && ch16 < a.lay.c16;
    const uint32_t p = (at.n * a.lay.th + h) * a.lay.tw + iw;
    return a.flags + (in ? (size_t)(p >> 5) * a.lay.c16 + ch16 : 0);
}

template <int MODE, int CT, int NT, bool HIGH>
__device__ __forceinline__ void load_block(const MfmaArgs &a, Operands<MODE, CT, NT, HIGH> &o, const int8_t *w, int kb,
                                           const KPos &k, const uint32_t (&px)[NT], const uint32_t (&px01)[NT],
                                           const PixelAt (&at)[NT], int lane)
{
    const int wtile = a.KB * mode_block(MODE);
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        const int8_t *wb = w + c * wtile + kb * mode_block(MODE);
#pragma unroll
        for (int g = 0; g < mode_sels(MODE); ++g) o.sel[c][g] = *(const v4i *)(wb + g * 1024 + lane * 16);
        o.index[c] = *(const int *)(wb + mode_sels(MODE) * 1024 + lane * 4);
    }
#pragma unroll
    for (int p = 0; p < NT; ++p) {
        if constexpr (mode_i8(MODE)) {
            o.lo[p][0] = *(const v4i *)(a.x + k.off + px[p]);
        } else {
            o.lo[p][0] = *(const v4i *)(a.x + k.off01 + px01[p]);
            o.lo[p][1] = *(const v4i *)(a.x + (k.off01 + a.lay.piece01) + px01[p]);
            o.d2[p] = *(const v4i *)(a.x + (k.off + 2 * a.lay.dstride) + px[p]);
        }
        if constexpr (HIGH) {
            o.d3[p] = *(const v4i *)(a.x + (k.off + 3 * a.lay.dstride) + px[p]);
            o.on[p] = *high_flag(a, at[p], lane >> 5, k, o.in[p]);
        }
    }
}

// Whether any input row of a tile has them (1), and digit d4 at that (2): p0 and p1 are its first and last pixel.
__device__ __forceinline__ int any_high(const MfmaArgs &a, uint32_t p0, uint32_t p1, int lane)
{
    const PixelAt u = pixel_at(a, p0), v = pixel_at(a, p1);
    int h0 = u.oh * a.sh + a.crop_h, h1 = v.oh * a.sh + a.crop_h + a.FH - 1;
    size_t from, to;
    if (!a.lay.tiles) {
        from = ((size_t)u.n * a.lay.Hp + h0) * a.lay.fy;
        to = ((size_t)v.n * a.lay.Hp + h1 + 1) * a.lay.fy;
    } else {
        h0 = h0 > a.lay.tph ? h0 - a.lay.tph : 0;
        h1 = h1 - a.lay.tph;
        if (h0 > a.lay.th - 1) h0 = a.lay.th - 1;
        if (h1 > a.lay.th - 1) h1 = a.lay.th - 1;
        if (h1 < 0) h1 = 0;
        from = (((size_t)u.n * a.lay.th + h0) * a.lay.tw >> 5) * a.lay.c16;
        to = (((((size_t)v.n * a.lay.th + h1 + 1) * a.lay.tw - 1) >> 5) + 1) * a.lay.c16;
    }
    int any = 0;
    for (size_t i = from + lane; i < to; i += 64) any |= a.flags[i];
    return (__any(any) ? 1 : 0) | (__any(any & 2) ? 2 : 0);
}

// Digit d4 of the rows that have any (|x| past 2^27, saturated values as a rule): what it adds to the sums, modulo 2^32.  A
// walk of its own over the reduction; a digit that was not written is masked after its load, not branched around.
template <int MODE, int CT, int NT>
__device__ __forceinline__ void digit4(const MfmaArgs &a, int32_t (*slot)[64], int lane, const int8_t *w, int kb0, int kb1,
                                       const uint32_t (&px)[NT], const PixelAt (&at)[NT])
{
    constexpr bool S15 = MODE == kI32S15;
    v16i acc[3][CT][NT] = {};   // 2^22, 2^15, 2^8
    int first[CT], second[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) {
        first[c] = (int)0x88888888u;
        second[c] = (int)0xddddddddu;
    }
    KPos k;
    k_start(a, k, kb0);
#pragma unroll 1
    for (int kb = kb0; kb < kb1; ++kb, k_next(a, k)) {
        v8i b[NT];
        v4i full[CT], lo[CT], hi[CT];
        int index[CT];
        const int wtile = a.KB * mode_block(MODE);
#pragma unroll
        for (int c = 0; c < CT; ++c) {
            const int8_t *wb = w + c * wtile + kb * mode_block(MODE);
            lo[c] = *(const v4i *)(wb + lane * 16);
            hi[c] = *(const v4i *)(wb + (mode_sels(MODE) - 1) * 1024 + lane * 16);
            index[c] = *(const int *)(wb + mode_sels(MODE) * 1024 + lane * 4);
        }
        v4i d4[NT];
#pragma unroll
        for (int p = 0; p < NT; ++p) {
            bool in;
            const uint8_t *flag = high_flag(a, at[p], lane >> 5, k, in);
            d4[p] = *(const v4i *)(a.x + (k.off + 4 * a.lay.dstride) + px[p]);
            d4[p] = and4(d4[p], *flag && in ? 0xffffffffu : 0u);
            b[p] = pairs_with_zero(d4[p]);
        }
        weights<CT>(full, kNegLo, kPosLo, lo);
        if constexpr (mode_sels(MODE) == 2) {
            v4i top[CT];
            weights<CT>(top, kNegHi, kPosHi, hi);
            both<CT>(full, full, top);
        }
        if constexpr (S15) {
            // q = 0 meets d4 at 2^22, q = 1 (second bytes) at 2^15, q = 2 at 2^8
            product<CT, NT>(acc[0], full, b, index);
            weights<CT>(lo, kNeg14, kPos14, hi);
            product<CT, NT>(acc[2], lo, b, first);
#pragma unroll
            for (int p = 0; p < NT; ++p)
#pragma unroll
                for (int i = 0; i < 8; ++i) b[p][i] = (int)((uint32_t)b[p][i] << 8);
            product<CT, NT>(acc[1], full, b, index);
        } else {
            product<CT, NT>(acc[0], full, b, first);
        }
    }
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int p = 0; p < NT; ++p)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                uint32_t v = (uint32_t)acc[0][c][p][i] << 22;
                if (S15) v += ((uint32_t)acc[1][c][p][i] << 15) + ((uint32_t)acc[2][c][p][i] << 8);
                slot[(c * NT + p) * 16 + i][lane] = (int32_t)v;
            }
}

// The sums of one wave's tile over blocks kb0 .. kb1 - 1.  Two sets of operands, the loads of a block in flight during the
// products of the one before; with digit d3, whose sums leave no room for them (14 VGPRs went to scratch and back in every
// block), and for 64 pixels (17 VGPRs; 32 channels of 16 x 16, 256 images: 15.8 us, so 14.7), one set, loaded again once the
// last operands of a block are formed and behind its last products.  Launches of 32 channels x 64 pixels still keep VGPRs in
// scratch, but across a loop, not in one: 6, 16 and 2 (shifts to 14, 6 and 3) are stored before the loop with digit d3 and loaded
// behind it, 3 (8-bit activations) before the epilogue's separate pieces.
template <int MODE, int CT, int NT, bool HIGH, bool ONE_SET = HIGH || (NT == 2 && !mode_i8(MODE)), typename Asked>
__device__ __forceinline__ void contract(const MfmaArgs &a, v16i (&total)[CT][NT], const int8_t *w, int kb0, int kb1,
                                         const uint32_t (&px)[NT], const uint32_t (&px01)[NT], const PixelAt (&at)[NT], int lane,
                                         Asked first_asked)
{
    typedef Operands<MODE, CT, NT, HIGH> Ops;
    Sums<CT, NT, HIGH> t = {};
    Ops o0;
    KPos k;
    k_start(a, k, kb0);
    int kb = kb0;
    const auto load = [&](Ops &o) { load_block<MODE, CT, NT, HIGH>(a, o, w, kb, k, px, px01, at, lane); };
    const auto multiply = [&](const Ops &o, const auto &reload) {
        if constexpr (mode_i8(MODE))
            block_i8<MODE, CT, NT>(o, t.bits);
        else if constexpr (MODE == kI32S15)
            block_s15<CT, NT, HIGH>(o, t, reload);
        else
            block_s7<MODE, CT, NT, HIGH>(o, t, reload);
    };
    load(o0);
    first_asked();
    if constexpr (ONE_SET) {
        bool more;
#pragma unroll 1
        do {
            multiply(o0, [&] {
                more = kb + 1 < kb1;
                if (more) {
                    ++kb;
                    k_next(a, k);
                }
                load(o0);   // the last block once more at the end: nobody waits for it
                __builtin_amdgcn_sched_barrier(0);
            });
        } while (more);
    } else {
        Ops o1;
        const auto none = [] {};
#pragma unroll 1
        while (kb + 2 < kb1) {
            ++kb;
            k_next(a, k);
            load(o1);
            multiply(o0, none);
            ++kb;
            k_next(a, k);
            load(o0);
            multiply(o1, none);
        }
        if (kb + 1 < kb1) {
            ++kb;
            k_next(a, k);
            load(o1);
            multiply(o0, none);
            multiply(o1, none);
        } else {
            multiply(o0, none);
        }
    }
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int p = 0; p < NT; ++p)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if constexpr (mode_i8(MODE)) {
                    total[c][p][i] = t.bits[c][p][i] >> (MODE == kI8S8 ? 3 : 1);
                } else {
                    uint32_t v = (uint32_t)(t.bits[c][p][i] >> 6) + ((uint32_t)t.d[0][c][p][i] << 1) + ((uint32_t)t.d[1][c][p][i] << 8);
                    if constexpr (HIGH) v += (uint32_t)t.d[2][c][p][i] << 15;
                    total[c][p][i] = (int)v;
                }
            }
}

// What follows the sums of eight channels (two groups of four, 8 apart) at one pixel.  The per-channel constants of a
// workgroup's channels lie in LDS: read from memory by every wave they were 96 loads of one word per 64 channels, which
// bounded short reductions (8-bit activations, 64 -> 256 channels, 1 x 1, 128 images of 56 x 56: 146 -> 97 us, with
// residual and float result 245 -> 195, the rate of a copy; 256 -> 64: 58 -> 45).
constexpr int kUnit = 8;
template <int CHANNELS>
struct ChannelTails {
    int32_t add[CHANNELS];
    float scale[CHANNELS], shift[CHANNELS];
    float scale1[CHANNELS], shift1[CHANNELS];   // the same for the shorter epilogue
    int odd[4];                                 // per wave: whether one of its channels has no exact shorter form
};
// A thread's channel of these, asked for first and stored once the first operands have been asked for too: one latency, not
// two, before the first product, which short reductions are made of (8-bit, 64 -> 256 channels,
// 1 x 1, 128 images of 56 x 56: 97 -> 89 us; 256 -> 64: 39.4 -> 37.4; one image of 512 x 7 x 7, 3 x 3, int32: 18.9 -> 17.1).
struct TailOfThread {
    int32_t add;
    float scale, shift;
};
__device__ __forceinline__ TailOfThread ask_tail(const MfmaArgs &a, int first, int count)
{
    TailOfThread r{0, 1.0f, 0.0f};
    const int i = threadIdx.x, c = first + i < a.N ? first + i : a.N - 1;
    if (i >= count) return r;
    r.add = (a.bias ? a.bias[c] : 0) - (a.corr ? a.corr[c] : 0);
    r.scale = a.scale ? a.scale[c] : 1.0f;
    r.shift = a.shift ? a.shift[c] : 0.0f;
    return r;
}
// The shorter epilogue: powers of two -- 2^-F of the sums, and 2^F of the next layer's grid where only its input is written --
// are multiplied into scale and shift, which changes no rounding while nothing leaves the range of normal numbers.  That is
// looked at here, per channel: a factor that loses bits, a scale or shift past any use take the other way.  For int32
// activations: 8-bit launches, whose registers are a third fewer, spill over it (block ends 195 -> 208 us) and gain nothing.
// 64 channels of 56 x 56, 3 x 3, 64 images: 87.6 -> 84.3 us; 16 of 32 x 32, 256 images: 30.0 -> 29.2; 64 -> 256, 1 x 1: 278 -> 258.
template <int CHANNELS>
__device__ __forceinline__ void stage_tails(const MfmaArgs &a, ChannelTails<CHANNELS> &t, const TailOfThread &r, int count)
{
    const int i = threadIdx.x;
    const float folded = r.scale * a.inv;
    const bool plain = folded * a.unfold == r.scale && fabsf(r.scale) < 0x1p60f && fabsf(r.shift) < 0x1p60f;
    if (i < count) {
        t.add[i] = r.add;
        t.scale[i] = r.scale;
        t.shift[i] = r.shift;
        t.scale1[i] = folded * a.qfold;
        t.shift1[i] = r.shift * a.qfold;
    }
    const int odd = __any(i < count && !plain) ? 1 : 0;
    if ((i & 63) == 0 && i < 256) t.odd[i >> 6] = odd;
}
struct ChannelTail {
    int32_t add[kUnit];
    float scale[kUnit], shift[kUnit];
};
template <int CHANNELS>
__device__ __forceinline__ void load_tail(const ChannelTails<CHANNELS> &t, ChannelTail &tl, int at)
{
#pragma unroll
    for (int i = 0; i < kUnit; ++i) {
        const int c = at + 8 * (i >> 2) + (i & 3);
        tl.add[i] = t.add[c];
        tl.scale[i] = t.scale[c];
        tl.shift[i] = t.shift[c];
    }
}
struct OutAt {
    size_t i;         // of channel 0 in y / out / residual
    size_t j, j01;    // of channel 0 in q; of its digits 0 and 1
    uint32_t p;
    bool in;
};
__device__ __forceinline__ OutAt out_at(const MfmaArgs &a, const PixelAt &at, uint32_t p)
{
    OutAt o;
    o.in = p < a.pixels;
    o.i = a.matrix ? (size_t)p * a.N : (size_t)at.n * a.ostride_n + (at.oh * a.OW + at.ow);
    o.p = p;
    o.j = a.qflags ? (size_t)(at.n * a.qHp + at.oh + a.qph) * a.qlay.rstride + (at.ow + a.qpw) * a.qlay.cp
                   : ((size_t)at.n * a.N * a.qHp + at.oh + a.qph) * a.qWp + at.ow + a.qpw;
    o.j01 = (size_t)(at.n * a.qHp + at.oh + a.qph) * a.qlay.rstride + (at.ow + a.qpw) * a.qlay.px01;
    return o;
}
// Eight values per lane (channels ch0 + 8 g + 0..3, ch0 = 16 u + 4 (lane >> 5)) into the next layer's operand layout: the
// halves of a wave swap words, so that a lane holds eight channels side by side and the 32 pixels of a digit are stored
// in a row.  Digits d3 and d4 only, with a flag, where the 32 pixels x 16 channels have any.  SCATTERED: a unit's pixels are not
// 32 in a row of the output, so its flags are shared with other units.
template <bool SCATTERED>
__device__ __forceinline__ void store_operands(const MfmaArgs &a, const int32_t (&qv)[kUnit], int ch0, const OutAt &o)
{
    const int half = (ch0 >> 2) & 1, u16 = ch0 >> 4;   // half = lane >> 5: ch0 is a multiple of 16 plus 0 or 4
    const MfmaX &L = a.qlay;
    const int c = u16 * 16 + half * 8, cb = L.cp == 16 ? c >> 4 : c >> 5;   // the lane's channels after the swap
    int8_t *q = (int8_t *)a.q + o.j + (size_t)cb * L.cbstride + (c & (L.cp - 1));
    if (L.digits == 1) {
        uint32_t b[2];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const uint32_t lo = __builtin_amdgcn_perm((uint32_t)qv[g * 4 + 1], (uint32_t)qv[g * 4], 0x0c0c0400u);
            const uint32_t hi = __builtin_amdgcn_perm((uint32_t)qv[g * 4 + 3], (uint32_t)qv[g * 4 + 2], 0x04000c0cu);
            b[g] = lo | hi;
        }
        const auto x = __builtin_amdgcn_permlane32_swap(b[0], b[1], false, false);
        if (o.in && cb < L.cb) *(uint2 *)q = uint2{x[0], x[1]};
        return;
    }
    uint32_t w[kDigits][2] = {}, e[2][2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int32_t dg[kDigits];
            digits_of(qv[g * 4 + i], dg);
#pragma unroll
            for (int d = 2; d < kDigits; ++d) w[d][g] |= ((uint32_t)dg[d] & 255u) << (8 * i);
        }
        e[g][0] = pair01(qv[g * 4]) | pair01(qv[g * 4 + 1]) << 16;
        e[g][1] = pair01(qv[g * 4 + 2]) | pair01(qv[g * 4 + 3]) << 16;
    }
    const uint32_t high4 = w[4][0] | w[4][1], high = w[3][0] | w[3][1] | high4;
    bool any = true;
    if constexpr (SCATTERED) {
        // d3 and d4 are always there; flags, zero before the launch, gather what their 32 pixels have.  One atomic for each flag
        // that the wave meets, some four or eight of them: one for each lane queued at the same words wherever most results are
        // past 16 (16.16; 3 x 3, us then and now, 64 images of 64 -> 128 channels of 112 x 112, 2 x 2 windows: 1060 and 625, as
        // sums and a pass 810; 64 of 512 of 28 x 28: 1590 and 1112; 32 of 64 of 32 x 32, 3 x 3 stride 1: 117 and 44, 49)
        const uint32_t flag = o.p >> 5;
        const bool set = u16 < L.c16 && o.in && high;
        for (uint64_t left = __ballot(set); left;) {
            const int first = __ffsll((unsigned long long)left) - 1;
            const uint32_t f = (uint32_t)__builtin_amdgcn_readlane((int)flag, first);
            const bool same = set && flag == f;
            const bool four = __any(same && high4);
            left &= ~__ballot(same);
            if ((int)(threadIdx.x & 63) == first) {
                const size_t at = (size_t)f * L.c16 + u16;
                atomicOr((uint32_t *)a.qflags + (at >> 2), (four ? 3u : 1u) << (8 * (at & 3)));
            }
        }
    } else {
        any = __any(o.in && high != 0);
        const bool any4 = __any(o.in && high4 != 0);
        if (u16 < L.c16 && (threadIdx.x & 63) == 0 && o.in)
            a.qflags[(size_t)(o.p >> 5) * L.c16 + u16] = any4 ? 3 : any ? 1 : 0;
    }
    const bool mine = o.in && cb < L.cb;
    {
        // eight channels of pairs: a 32-channel block keeps them by their place in its halves, others in a row
        const auto x = __builtin_amdgcn_permlane32_swap(e[0][0], e[1][0], false, false);
        const auto y = __builtin_amdgcn_permlane32_swap(e[0][1], e[1][1], false, false);
        int8_t *q01 = (int8_t *)a.q + o.j01 + (size_t)cb * L.cbstride + (L.cp == 32 ? (u16 & 1) * 16 : 0) + half * L.piece01;
        if (mine) *(v4i *)q01 = v4i{(int)x[0], (int)y[0], (int)x[1], (int)y[1]};
    }
#pragma unroll
    for (int d = 2; d < kDigits; ++d) {
        if (d >= 3 && !any) break;
        const auto x = __builtin_amdgcn_permlane32_swap(w[d][0], w[d][1], false, false);
        if (mine) *(uint2 *)(q + d * L.dstride) = uint2{x[0], x[1]};
    }
}

__device__ __forceinline__ void load_residual(const MfmaArgs &a, float (&res)[kUnit], int ch0, const OutAt &o)
{
#pragma unroll
    for (int i = 0; i < kUnit; ++i) {
        // past the end: some value that is there (it is not used), so that no load waits behind a branch
        const int ch = ch0 + 8 * (i >> 2) + (i & 3), c = ch < a.N ? ch : a.N - 1;
        res[i] = a.residual[(o.in ? o.i : 0) + (size_t)c * a.ostride_c];
    }
}

// Stores of eight values; the uniform test spares full tiles the per-channel ones.
template <typename T>
__device__ __forceinline__ void store_channels(T *dst, const T (&v)[kUnit], int ch0, int stride, int N, bool in)
{
    if ((ch0 & ~15) + 2 * kUnit <= N) {
        if (in)
#pragma unroll
            for (int i = 0; i < kUnit; ++i) dst[(size_t)(ch0 + 8 * (i >> 2) + (i & 3)) * stride] = v[i];
    } else {
#pragma unroll
        for (int i = 0; i < kUnit; ++i) {
            const int ch = ch0 + 8 * (i >> 2) + (i & 3);
            if (in && ch < N) dst[(size_t)ch * stride] = v[i];
        }
    }
}
__device__ __forceinline__ void quantize_all(const float (&f)[kUnit], int32_t (&q)[kUnit], const QuantSpec &spec)
{
    QuantSpec s = spec;
    s.mode = DS_Q_ROUND_TO_FIXED;
    if (spec.I == 1) {
        s.I = 1;
#pragma unroll
        for (int i = 0; i < kUnit; ++i) q[i] = quantize_one(f[i], s);
    } else {
        s.I = 2;   // the bounds are in lo and hi
#pragma unroll
        for (int i = 0; i < kUnit; ++i) q[i] = quantize_one(f[i], s);
    }
}
// The next layer's input of a unit, quantised.
template <bool SCATTERED>
__device__ __forceinline__ void store_q(const MfmaArgs &a, int32_t (&qv)[kUnit], int ch0, const OutAt &o)
{
    if (a.qflags) {
        if ((ch0 & ~15) + 2 * kUnit > a.N)
#pragma unroll
            for (int i = 0; i < kUnit; ++i)
                if (ch0 + 8 * (i >> 2) + (i & 3) >= a.N) qv[i] = 0;
        store_operands<SCATTERED>(a, qv, ch0, o);
    } else if (a.q_bytes == 1) {
        int8_t b[kUnit];
#pragma unroll
        for (int i = 0; i < kUnit; ++i) b[i] = (int8_t)qv[i];
        store_channels((int8_t *)a.q + o.j, b, ch0, a.qHp * a.qWp, a.N, o.in);
    } else {
        store_channels((int32_t *)a.q + o.j, qv, ch0, a.qHp * a.qWp, a.N, o.in);
    }
}
// What follows the affine step.
template <bool SCATTERED>
__device__ __forceinline__ void store_values(const MfmaArgs &a, float (&f)[kUnit], const float (&res)[kUnit], int ch0, const OutAt &o)
{
    if (a.residual)
#pragma unroll
        for (int i = 0; i < kUnit; ++i) f[i] += res[i];
    if (a.relu)
#pragma unroll
        for (int i = 0; i < kUnit; ++i) f[i] = fmaxf(f[i], 0.0f);
    if (a.out) store_channels(a.out + o.i, f, ch0, a.ostride_c, a.N, o.in);
    if (!a.q) return;
    int32_t qv[kUnit];
    if (a.relu && a.qspec.I != 1) {
        // neither negative nor NaN: the conversion's truncation is the floor, the lower bound is met
#pragma unroll
        for (int i = 0; i < kUnit; ++i) qv[i] = f2i_sat(fminf(f[i] * a.qspec.scale, a.qspec.hi));
    } else {
        quantize_all(f, qv, a.qspec);
    }
    store_q<SCATTERED>(a, qv, ch0, o);
}
template <bool SCATTERED>
__device__ __forceinline__ void store_tail(const MfmaArgs &a, const ChannelTail &t, const int32_t (&sum)[kUnit],
                                           const float (&res)[kUnit], int ch0, const OutAt &o)
{
    int32_t v[kUnit];
#pragma unroll
    for (int i = 0; i < kUnit; ++i) v[i] = sum[i] + t.add[i];
    if (a.y) {
        store_channels(a.y + o.i, v, ch0, a.ostride_c, a.N, o.in);
        return;
    }
    float f[kUnit];
#pragma unroll
    for (int i = 0; i < kUnit; ++i) f[i] = affine_one(v[i], a.inv, t.scale[i], t.shift[i], nullptr, 0);
    store_values<SCATTERED>(a, f, res, ch0, o);
}
// The shorter epilogue (stage_tails): sum is complete, scale and shift of t are the folded ones.
__device__ __forceinline__ void store_tail_folded(const MfmaArgs &a, const ChannelTail &t, const int32_t (&sum)[kUnit],
                                                  const float (&res)[kUnit], int ch0, const OutAt &o)
{
    float f[kUnit];
#pragma unroll
    for (int i = 0; i < kUnit; ++i) f[i] = affine_one(sum[i], 1.0f, t.scale[i], t.shift[i], nullptr, 0);
    if (!a.q_only) {
        store_values<false>(a, f, res, ch0, o);
        return;
    }
    // ReLU, the upper bound and the floor in two instructions a value
    int32_t qv[kUnit];
#pragma unroll
    for (int i = 0; i < kUnit; ++i) qv[i] = f2i_sat(__builtin_amdgcn_fmed3f(f[i], 0.0f, a.qspec.hi));
    store_q<false>(a, qv, ch0, o);
}

// Four or eight waves per workgroup; a wave owns CT * 32 channels x NT * 32 pixels and one of ks parts of the reduction (the
// parts of a tile lie in one workgroup and meet in LDS).  No operand passes through LDS: activations and selectors are
// fragments in memory already, each a contiguous KiB.
template <int MODE, int CT, int NT, int WAVES>
__global__ __launch_bounds__(WAVES * 64, mode_i8(MODE) && WAVES == 4 ? 3 : 2) void mfma_kernel(MfmaArgs a)
{
    __shared__ int32_t part[WAVES][CT * NT * 16][64];
    __shared__ ChannelTails<CT * 64> tails;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // the compiler moves no load of an argument past this: ks and the like are asked for with the others, not one by one in the
    // branch that needs them, 5 waits in front of the first operand in place of 7 (64 -> 64 channels, 3 x 3, 32 images of 56 x 56,
    // with layout pass: 51.2 -> 50.6 us; 1000 x 1537 x 777: 28.1 -> 27.8; 8-bit launches, which have 4, gain nothing)
    if constexpr (!mode_i8(MODE)) asm volatile("");
    // workgroups are dealt to the eight XCDs in turn: give each XCD neighbouring tiles
    uint32_t wg = blockIdx.x, tile0 = 0;
    const uint32_t per = a.whole >> 3;
    int ks = a.ks;
    if (wg >= a.whole) {
        wg -= a.whole;
        tile0 = a.tail_tile;
        ks = 4;
    } else if (wg < per * 8) {
        wg = (wg & 7) * per + (wg >> 3);
    }
    const uint32_t pt = div_by_uniform(wg, a.by_ctiles);
    const int ct = (int)(wg - pt * a.ctiles);
    const int kpart = wave % ks, t = wave / ks;
    const int pw = WAVES / ks / a.tc;   // pixel tiles per workgroup
    const int c0 = (ct * a.tc + t % a.tc) * (CT * 32);
    const uint32_t p0 = (tile0 + pt * pw + t / a.tc) * (NT * 32);
    const int kb0 = (int)((long)a.KB * kpart / ks), kb1 = (int)((long)a.KB * (kpart + 1) / ks);

    const bool live = c0 < a.N && p0 < a.pixels;
    uint32_t pix[NT], px[NT], px01[NT];
    PixelAt at[NT];
#pragma unroll
    for (int p = 0; p < NT; ++p) {
        pix[p] = p0 + p * 32 + (lane & 31);
        at[p] = pixel_at(a, pix[p] < a.pixels ? pix[p] : a.pixels - 1);
        const uint32_t row = (at[p].n * a.lay.Hp + at[p].oh * a.sh + a.crop_h) * a.lay.rstride, col = at[p].ow * a.sw + a.crop_w;
        px[p] = row + col * a.lay.cp + (lane >> 5) * 16;
        px01[p] = row + col * a.lay.px01 + (lane >> 5) * a.lay.half01;
    }
    const int tail0 = t % a.tc * (CT * 32) + 4 * (lane >> 5);   // the lane's first channel there
    const TailOfThread tail = ask_tail(a, ct * a.tc * (CT * 32), a.tc * (CT * 32));
    // every wave comes here once, wherever its tile takes it
    const auto staged = [&] {
        stage_tails(a, tails, tail, a.tc * (CT * 32));
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    };
    v16i total[CT][NT] = {};
    if (live && kb0 < kb1) {
        const int8_t *w = a.blob + (size_t)(c0 >> 5) * (a.KB * mode_block(MODE));
        int high = 0;
        if constexpr (!mode_i8(MODE)) {
            const uint32_t last = p0 + NT * 32 - 1;
            high = any_high(a, p0, last < a.pixels ? last : a.pixels - 1, lane);
            if (high & 2) digit4<MODE, CT, NT>(a, part[wave], lane, w, kb0, kb1, px, at);
            if (high) contract<MODE, CT, NT, true>(a, total, w, kb0, kb1, px, px01, at, lane, staged);
            if (high & 2)
#pragma unroll
                for (int c = 0; c < CT; ++c)
#pragma unroll
                    for (int p = 0; p < NT; ++p)
#pragma unroll
                        for (int i = 0; i < 16; ++i) total[c][p][i] += part[wave][(c * NT + p) * 16 + i][lane];
        }
        if (!high) contract<MODE, CT, NT, false>(a, total, w, kb0, kb1, px, px01, at, lane, staged);
    } else {
        staged();
    }
    const bool folded = !mode_i8(MODE) && WAVES == 4 && ks == 1 && !a.y && !(tails.odd[0] | tails.odd[1]);
    const int chl = c0 + 4 * (lane >> 5);
    if (ks == 1) {
        if (!live) return;
        // units of 16 channels x 32 pixels; every residual is on its way before the first value is stored
        OutAt o[NT];
        float res[CT * 2 * NT][8];
#pragma unroll
        for (int p = 0; p < NT; ++p) o[p] = out_at(a, at[p], pix[p]);
        if (a.residual)
#pragma unroll
            for (int u = 0; u < CT * 2 * NT; ++u) load_residual(a, res[u], chl + u / NT * 16, o[u % NT]);
        if (folded) {
#pragma unroll
            for (int c = 0; c < CT * 2; ++c) {
                asm volatile("" ::: "memory");   // the constants of one unit at a time
                ChannelTail tl;
#pragma unroll
                for (int i = 0; i < kUnit; ++i) {
                    const int ch = tail0 + c * 16 + 8 * (i >> 2) + (i & 3);
                    tl.add[i] = tails.add[ch];
                    tl.scale[i] = tails.scale1[ch];
                    tl.shift[i] = tails.shift1[ch];
                }
#pragma unroll
                for (int p = 0; p < NT; ++p) {
                    int32_t v[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = total[c >> 1][p][(c & 1) * 8 + i] + tl.add[i];
                    store_tail_folded(a, tl, v, res[c * NT + p], chl + c * 16, o[p]);
                }
            }
            return;
        }
#pragma unroll
        for (int c = 0; c < CT * 2; ++c) {
            ChannelTail tl;
            load_tail(tails, tl, tail0 + c * 16);
#pragma unroll
            for (int p = 0; p < NT; ++p) {
                int32_t v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = total[c >> 1][p][(c & 1) * 8 + i];
                store_tail<false>(a, tl, v, res[c * NT + p], chl + c * 16, o[p]);
            }
        }
        return;
    }
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int p = 0; p < NT; ++p)
#pragma unroll
            for (int i = 0; i < 16; ++i) part[wave][(c * NT + p) * 16 + i][lane] = total[c][p][i];
    __syncthreads();
    if (!live) return;
    // the ks waves of a tile share its epilogue, in halves of 32 x 32 values
    constexpr int all = CT * NT * 2;
    const int units = all > ks ? all / ks : 1;
    for (int u = kpart * units; u < (kpart + 1) * units && u < all; ++u) {
        const int ch = chl + (u >> 1) / NT * 32 + (u & 1) * 16;
        const uint32_t pp = p0 + (u >> 1) % NT * 32 + (lane & 31);
        const OutAt o = out_at(a, pixel_at(a, pp), pp);
        ChannelTail tl;
        float res[8];
        load_tail(tails, tl, tail0 + ch - chl);
        if (a.residual) load_residual(a, res, ch, o);
        int32_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            v[i] = 0;
            for (int s = 0; s < ks; ++s) v[i] += part[t * ks + s][u * 8 + i][lane];
        }
        store_tail<false>(a, tl, v, res, ch, o);
    }
}

// A convolution with a max pooling behind it (a ResNet's stem).
struct MfmaPool {
    int pk, ps, pp;             // window, stride, padding
    int POH, POW;               // pooled rows and columns
    int th, tw, PH, PW;         // of a workgroup: its pooled rows and columns, and the convolution's that they take
    int tiles_h, tiles_w;
    FastDiv by_pw, by_tw, by_tiles_w, by_tiles_h;
};
constexpr int kPoolPixels = 256, kPoolStride = 68;   // words per pixel: 64 channels, and 4 to spread rows over the banks

// A workgroup forms the sums of 64 channels x a rectangle of pixels (32 at a time per wave, as mfma_kernel does), leaves them
// in LDS and pools from there, so that the sums are neither written nor read: with a pass of its own they were, 4 bytes each,
// and the padded result was laid out by a third.  Rectangles overlap by pk - ps rows and columns: 15 x 17 pixels give 7 x 8
// windows of 3 x 3 with stride 2, an eighth of the products done twice.  The affine step is monotonic in the sum (every
// rounding is), so a window's value is that of its largest sum, or smallest where the scale is negative, which are kept
// inverted.  us, layer, pooling pass and layout pass before, and this: 64 images of 224 x 224, 3 -> 64 channels, 7 x 7, shifts to
// 14: 162 + 68 + 23 and 170; 8-bit activations 87 + 61 + 17 and 88; 128 images, shifts to 2: 164 + 110 + 54 (two layers read it)
// and 123.  What bounds it: vector instructions, about 700 for 32 pixels x 64 channels beside 56 or 140 products.
template <int MODE, bool K3>
__global__ __launch_bounds__(256, 2) void mfma_pool_kernel(MfmaArgs a, MfmaPool m)
{
    __shared__ int32_t sums[kPoolPixels * kPoolStride];
    __shared__ ChannelTails<64> tails;
    __shared__ int32_t flips[64];   // all ones where the smallest sum counts
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t wg = blockIdx.x;
    const uint32_t per = gridDim.x >> 3;
    if (wg < per * 8) wg = (wg & 7) * per + (wg >> 3);
    uint32_t rest = div_by_uniform(wg, a.by_ctiles);
    const int c0 = (int)(wg - rest * a.ctiles) * 64;
    const uint32_t tiles = div_by_uniform(rest, m.by_tiles_w);
    const int w0 = (int)(rest - tiles * m.tiles_w) * m.tw;
    const uint32_t n = div_by_uniform(tiles, m.by_tiles_h);
    const int h0 = (int)(tiles - n * m.tiles_h) * m.th;
    const int r0 = h0 * m.ps - m.pp, q0 = w0 * m.ps - m.pp;   // the rectangle's first row and column
    const int pixels = m.PH * m.PW;
    stage_tails(a, tails, ask_tail(a, c0, 64), 64);
    if (threadIdx.x < 64) flips[threadIdx.x] = tails.scale[threadIdx.x] < 0.0f ? -1 : 0;
    __syncthreads();
    const int8_t *w = a.blob + (size_t)(c0 >> 5) * (a.KB * mode_block(MODE));
    int high = 0;
    if constexpr (!mode_i8(MODE)) {
        const int first = r0 < 0 ? 0 : r0, last = r0 + m.PH < a.OH ? r0 + m.PH - 1 : a.OH - 1;
        high = any_high(a, (n * a.OH + first) * a.OW, (n * a.OH + last) * a.OW + a.OW - 1, lane);
    }
    for (int t = wave; t * 32 < pixels; t += 4) {
        const int pos = t * 32 + (lane & 31);
        const uint32_t clamped = pos < pixels ? pos : pixels - 1, r = div_by(clamped, m.by_pw);
        int oh = r0 + (int)r, ow = q0 + (int)(clamped - r * m.PW);
        oh = oh < 0 ? 0 : oh < a.OH ? oh : a.OH - 1;
        ow = ow < 0 ? 0 : ow < a.OW ? ow : a.OW - 1;
        const PixelAt at[1] = {{n, (uint32_t)oh, (uint32_t)ow}};
        const uint32_t row = (n * a.lay.Hp + oh * a.sh + a.crop_h) * a.lay.rstride, col = ow * a.sw + a.crop_w;
        const uint32_t px[1] = {row + col * a.lay.cp + (lane >> 5) * 16};
        const uint32_t px01[1] = {row + col * a.lay.px01 + (lane >> 5) * a.lay.half01};
        v16i total[2][1];
        const auto none = [] {};
        int32_t (*slot)[64] = (int32_t (*)[64])(sums + t * 32 * kPoolStride);   // this tile's own place, before its sums
        if constexpr (mode_i8(MODE)) {
            contract<MODE, 2, 1, false>(a, total, w, 0, a.KB, px, px01, at, lane, none);
        } else if (high) {
            if (high & 2) digit4<MODE, 2, 1>(a, slot, lane, w, 0, a.KB, px, at);
            contract<MODE, 2, 1, true>(a, total, w, 0, a.KB, px, px01, at, lane, none);
            if (high & 2)
#pragma unroll
                for (int c = 0; c < 2; ++c)
#pragma unroll
                    for (int i = 0; i < 16; ++i) total[c][0][i] += slot[c * 16 + i][lane];
        } else {
            contract<MODE, 2, 1, false, true>(a, total, w, 0, a.KB, px, px01, at, lane, none);
        }
        asm volatile("" ::: "memory");   // the constants are read here, not kept in 96 registers through the loop
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int ch = u * 16 + 4 * (lane >> 5);
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                v4i v = *(const v4i *)(tails.add + ch + 8 * g);
                const v4i flip = *(const v4i *)(flips + ch + 8 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = (total[u >> 1][0][(u & 1) * 8 + g * 4 + i] + v[i]) ^ flip[i];
                *(v4i *)(sums + pos * kPoolStride + ch + 8 * g) = v;
            }
        }
    }
    __syncthreads();
    // a wave pools 16 of the channels
    const int ch = wave * 16 + 4 * (lane >> 5), windows = m.th * m.tw;
    if (c0 + wave * 16 >= a.N) return;
    ChannelTail tl;
    load_tail(tails, tl, ch);
    for (int g = 0; g < windows; g += 32) {
        const int idx = g + (lane & 31), clamped = idx < windows ? idx : windows - 1;
        const int i0 = (int)div_by((uint32_t)clamped, m.by_tw), j0 = clamped - i0 * m.tw;
        const int oh = h0 + i0, ow = w0 + j0;
        int32_t best[kUnit];
#pragma unroll
        for (int i = 0; i < kUnit; ++i) best[i] = INT32_MIN;
        // rows and columns outside the image: the nearest one inside, which is in the window too
        const auto row = [&](int i) {
            const int r = oh * m.ps - m.pp + i;
            return ((r < 0 ? 0 : r < a.OH ? r : a.OH - 1) - r0) * m.PW;
        };
        const auto column = [&](int j) {
            const int c = ow * m.ps - m.pp + j;
            return (c < 0 ? 0 : c < a.OW ? c : a.OW - 1) - q0;
        };
        const auto take = [&](int at) {
            const v4i v0 = *(const v4i *)(sums + at * kPoolStride + ch), v1 = *(const v4i *)(sums + at * kPoolStride + ch + 8);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                best[k] = v0[k] > best[k] ? v0[k] : best[k];
                best[4 + k] = v1[k] > best[4 + k] ? v1[k] : best[4 + k];
            }
        };
        if constexpr (K3) {
            int c[3];
#pragma unroll
            for (int j = 0; j < 3; ++j) c[j] = column(j);
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const int r = row(i);
#pragma unroll
                for (int j = 0; j < 3; ++j) take(r + c[j]);
            }
        } else {
            for (int i = 0; i < m.pk; ++i) {
                const int r = row(i);
                for (int j = 0; j < m.pk; ++j) take(r + column(j));
            }
        }
        OutAt o;
        o.in = idx < windows && oh < m.POH && ow < m.POW;
        o.p = o.in ? (n * m.POH + oh) * m.POW + ow : 0;
        o.i = (size_t)n * a.ostride_n + (oh * m.POW + ow);
        const size_t qrow = (size_t)(n * a.qHp + oh + a.qph);
        o.j = a.qflags ? qrow * a.qlay.rstride + (ow + a.qpw) * a.qlay.cp
                       : ((size_t)n * a.N * a.qHp + oh + a.qph) * a.qWp + ow + a.qpw;
        o.j01 = qrow * a.qlay.rstride + (ow + a.qpw) * a.qlay.px01;
        const float res[kUnit] = {};
        ChannelTail plain = tl;
#pragma unroll
        for (int i = 0; i < kUnit; ++i) {
            best[i] ^= flips[ch + 8 * (i >> 2) + (i & 3)];
            plain.add[i] = 0;   // it is in the sums
        }
        store_tail<true>(a, plain, best, res, c0 + ch, o);
    }
}

// Zeros for flags that a launch gathers.
__global__ __launch_bounds__(256) void mfma_clear_kernel(uint32_t *__restrict__ words, long count)
{
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < count; i += (long)gridDim.x * 256) words[i] = 0;
}

// The padding of the next layer's input.
template <typename Q>
__global__ __launch_bounds__(256) void mfma_border_kernel(Q *__restrict__ q, long planes, int Hp, int Wp, int ph, int pw)
{
    const int rows = 2 * ph * Wp, side = 2 * pw * (Hp - 2 * ph), per = rows + side;
    const long total = planes * per;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
        const long plane = i / per;
        int r = (int)(i - plane * per), h, w;
        if (r < rows) {
            h = r / Wp;
            w = r - h * Wp;
            if (h >= ph) h += Hp - 2 * ph;
        } else {
            r -= rows;
            h = r / (2 * pw);
            w = r - h * 2 * pw;
            h += ph;
            if (w >= pw) w += Wp - 2 * pw;
        }
        q[(plane * Hp + h) * Wp + w] = 0;
    }
}

// ... and of its operands, in pieces of 16 bytes: whole rows above and below, both ends of the columns of the others.
// For buffers that no caller zeroed once (first use, and captured graphs, which own theirs).
__global__ __launch_bounds__(256) void mfma_operand_border_kernel(int8_t *__restrict__ q, MfmaX lay, int ph, int pw)
{
    // digits 0 and 1 of 16-channel blocks lie side by side: one segment of two pieces a pixel in place of two of one
    const bool joined = lay.digits > 1 && lay.cp == 16;
    const int segments = lay.cb * lay.digits, pieces = lay.dstride >> 4, wide = lay.cp >> 4;
    for (long row = blockIdx.x; row < lay.rows; row += gridDim.x) {
        v4i *r = (v4i *)(q + (size_t)row * lay.rstride);
        const int h = (int)(row % lay.Hp);
        if (h < ph || h >= lay.Hp - ph) {
            for (int i = threadIdx.x; i < lay.rstride >> 4; i += 256) r[i] = v4i{};
        } else {
            const int side = pw * wide;
            for (int i = threadIdx.x; i < segments * 2 * side; i += 256) {
                const int segment = i / (2 * side), j = i - segment * 2 * side;
                const int digit = segment % lay.digits;
                if (joined && digit < 2) {
                    // digit 0's share clears the left columns, digit 1's the right ones
                    const int base = (segment - digit) * pieces;
                    r[base + (digit == 0 ? j : 2 * (lay.Wp - pw) + j)] = v4i{};
                } else {
                    r[segment * pieces + (j < side ? j : (lay.Wp - 2 * pw) * wide + j)] = v4i{};
                }
            }
        }
    }
}

// ks waves to a tile; with `groups` (ks 1, CT 2), whole tiles for that many groups of four pixel tiles, and the pixel tiles
// that are left shared four ways.
template <int MODE, int CT, int NT, int WAVES>
static int launch_tiles(MfmaArgs &a, int ks, long groups, hipStream_t st)
{
    const int ctiles = ceil_div(a.N, CT * 32), tiles = ceil_div((int)a.pixels, NT * 32);
    a.ks = ks;
    a.tc = CT == 1 && WAVES / a.ks >= 2 && ctiles > 1 ? 2 : 1;
    a.ctiles = ceil_div(ctiles, a.tc);
    a.by_ctiles = fast_div((uint32_t)a.ctiles);
    const int pw = WAVES / a.ks / a.tc;
    long grid = (long)a.ctiles * ceil_div(tiles, pw);
    a.whole = (uint32_t)grid;
    if (groups > 0) {
        a.whole = (uint32_t)(groups * a.ctiles);
        a.tail_tile = (uint32_t)(groups * pw);
        grid = a.whole + (tiles - groups * pw) * (long)a.ctiles;
    }
    hipLaunchKernelGGL((mfma_kernel<MODE, CT, NT, WAVES>), dim3((unsigned)grid), dim3(WAVES * 64), 0, st, a);
    return launch_status();
}

// Whole tiles would give some CUs a workgroup more than others: all get the same number, and the tiles that are left, which
// a fraction of the chip would work on alone, are shared four ways.  Groups of four pixel tiles that stay whole; 0: not so.
// What is left may be more the longer the reduction is (it pays for four starts and the meeting), and short reductions gain
// only where a round is a good part of the launch.  us without and with, 64 channels, hand-off (left in tiles a CU):
//   1280 tiles (1)     blocks 4: 15.4 12.5   9: 19.9 15.6   18: 28.2 21.4   36: 41.7 33.3   72: 81.2 71.1
//   1536 and 2560 (2)  4: 15.6 18.3, 21.9 22.6   9: 20.0 24.0, 28.2 28.2   18: 28.6 27.5, 41.5 38.6   36: 43.8 40.1, 79.8 69.8
//   1792 (3)           9: 20.3 24.2   18: 28.8 31.4   36: 48.2 48.1   72: 101 98
// ResNet layers, 3 x 3, 64 images, of 64, 128, 256 channels, whose tiles are 49 times a power of two: 89 80, 80 66, 74 71; 8-bit
// 42 38, 41 33, 37 34; 128 images of 256 channels of 14 x 14 134 117, 8-bit 68 54; 1024 -> 256, 1 x 1, 8-bit: 37 30.
static long even_groups(const MfmaArgs &a, long cus)
{
    const long ctiles = ceil_div(a.N, 64), tiles = ceil_div((int)a.pixels, 32), grid = ctiles * ((tiles + 3) / 4);
    if (grid <= cus || (a.KB < 8 && grid > 4 * cus)) return 0;
    const long groups = grid / cus * cus / ctiles, left = (tiles - groups * 4) * ctiles;
    return left > 0 && left <= (a.KB >= 32 ? 3 : a.KB >= 16 ? 2 : 1) * cus ? groups : 0;
}

// Waves that share a tile's reduction, of `blocks` blocks.  Waves in one workgroup also share a tile's epilogue, which is most
// of a short reduction's time, so few tiles always take four; more tiles take as many as fit a workgroup a CU (two, three
// with the registers of 8-bit activations), if the reduction pays for its parts' start and their meeting in LDS; and a long
// one is cut in two while that fills slots which whole tiles leave empty.  Measured with 1, 2 and 4 parts, hand-off to the
// next layer (us; 256 CUs, tiles of 64 channels x 32 pixels):
//   int32, blocks  512 tiles        768               1024              1536              2560              4096
//     2            10.6  9.3  8.5*  10.9 11.1 14.2                                                          (*: 384)
//     4            11.8 10.2  9.4   12.0 12.2 14.6    12.4 12.5 16.7    16.6 19.3 23.8    23.9 28.2 37.5    29.9 41.3 57.3
//     9            14.4 11.6 10.9   14.7 14.7 16.9    15.2 15.4 19.6    21.6 23.1 28.0    30.3 34.0 43.8    39.4 50.0 67.4
//     18           19.4 14.6 13.3   20.8 19.5 20.3    21.6 20.6 24.1    30.1 29.5 33.8    43.7 44.2 53.2    62.2 71.9 88.2
//     36           30.4 20.7 18.7   31.1 28.4 26.6    32.3 29.7 32.8    47.8 43.8 46.4    84.1 80.8 86.5     121  133  143
//   8-bit
//     4             7.4  7.5  6.7    7.5  8.2  7.6     7.6  8.4 11.0     9.2  9.4 13.2    11.4 15.0 20.5    15.1 21.2 29.8
//     9             8.7  8.2  7.5    8.8  9.4  8.3     8.9  9.5 11.9    11.4 11.3 14.5    14.9 17.6 22.4    19.3 25.7 34.1
//     18           11.2  9.4  8.6   11.4 11.3 10.1    11.5 11.6 13.5    15.9 15.2 17.2    21.4 22.1 26.9    27.4 32.3 40.8
//     36           16.3 11.9 10.6   16.6 15.6 13.1    17.7 16.6 17.4    24.4 21.2 22.8    33.3 32.0 35.8    44.3 48.0 55.0
static int reduction_parts(long tiles, long cus, int blocks, bool i8)
{
    if (tiles <= 2 * cus || (tiles <= 3 * cus && blocks >= (i8 ? 9 : 32))) return 4;
    if (tiles <= 6 * cus) return blocks >= 16 ? 2 : 1;
    return !i8 && blocks >= 32 && tiles > 8 * cus && tiles < 16 * cus ? 2 : 1;
}

template <int MODE>
static int launch_mfma(MfmaArgs &a, hipStream_t st)
{
    const long cus = device_cus();
    const bool pair = a.N > 32;
    const long tiles = pair ? (long)ceil_div(a.N, 64) * ceil_div((int)a.pixels, 32) : (long)ceil_div((int)a.pixels, 64);
    // Fewer than a tile for every other CU: half the tile, and the reduction in eight parts (64 and 128 tiles, us with four
    // parts and these: 4 blocks 8.0, 7.8; 18: 9.9, 9.1; 36: 11.9, 10.5; 144: 28.4, 21.0; 256 tiles: 30.9, 41.2).
    if (tiles <= cus / 2) return launch_tiles<MODE, 1, 1, 8>(a, 8, 0, st);
    const long groups = pair ? even_groups(a, cus) : 0;
    const int ks = groups ? 1 : reduction_parts(tiles, cus, a.KB, mode_i8(MODE));
    return pair ? launch_tiles<MODE, 2, 1, 4>(a, ks, groups, st) : launch_tiles<MODE, 1, 2, 4>(a, ks, 0, st);
}

// Workgroups of a fused pooling launch, two a CU, one after another: how long it takes, in rounds -- one tile of 32 pixels for
// each of a workgroup's four waves -- of a CU that has two of them.  A round without a second workgroup takes 0.8 of that.
static double pool_rounds(long workgroups, int tiles, long cus)
{
    const long rest = workgroups % (2 * cus);
    return ceil_div(tiles, 4) * (workgroups / (2 * cus) + (rest == 0 ? 0.0 : rest <= cus ? 0.8 : 1.0));
}

// The rectangle of pooled pixels of a workgroup, whose convolution takes at most kPoolPixels: the one whose launch takes the
// fewest rounds, of these the one with the fewest tiles, and the largest of those.  Returns the rounds.
static double pool_tile(MfmaPool &m, long images, long cus)
{
    double best = 0;
    long least = 0, fewest = 0;
    for (int limit = kPoolPixels; limit >= 128; limit /= 2)
        for (int th = 1; th <= m.POH; ++th) {
            const long PH = (long)(th - 1) * m.ps + m.pk;
            if (PH * m.pk > limit) break;
            long tw = (limit / PH - m.pk) / m.ps + 1;   // the widest, then as wide as that many in a row need to be
            if (tw > m.POW) tw = m.POW;
            const int down = ceil_div(m.POH, th), across = ceil_div(m.POW, (int)tw);
            tw = ceil_div(m.POW, across);
            const long PW = (tw - 1) * m.ps + m.pk, rectangles = (long)down * across;
            const int tiles = (int)((PH * PW + 31) / 32);
            const double rounds = pool_rounds(images * rectangles, tiles, cus);
            const long spent = rectangles * tiles;
            if (best > 0 && (rounds > best || (rounds == best && (spent > least || (spent == least && rectangles >= fewest))))) continue;
            best = rounds;
            least = spent;
            fewest = rectangles;
            m.th = th;
            m.tw = (int)tw;
            m.PH = (int)PH;
            m.PW = (int)PW;
            m.tiles_h = down;
            m.tiles_w = across;
        }
    return best;
}

// Whether a convolution and the max pooling behind it take less time as one launch than as sums, a pooling pass and, as a
// rule, a layout pass for the layer that reads the result: an estimate of both, in us, fitted to 240 shapes and 160 drawn ones.
// The single launch multiplies pixels that rectangles share more than once, leaves waves idle in rectangles of odd sizes, and
// never cuts a reduction: a round (pool_rounds) takes `block` per block of the reduction and 4.  The separate one writes and
// reads the sums, 4 ns a tile, reads each as often as windows overlap, 0.4 ps a value more than the single launch does from LDS,
// and has two more launches: 12, between what they take in a graph (7) and what they take the host (14).  Nor is it done before
// the host has issued all of it, kPoolHost: 24 on the host of the table below, 37 on a slower one, where one launch takes 25 (us
// there, 1 image: 32 -> 96 channels of 13 x 13, 5 x 5: 39 28; 512 -> 256, 1 x 1, 3 x 3 windows stride 1: 40 31; 64 -> 96 of 16 x 16,
// 5 x 5 stride 1: 38 29; 8-bit 128 -> 40 of 27 x 27, 3 x 3 / 2: 38 26; 2 images 256 -> 96 of 6 x 6: 38 27).  us separate, fused,
// issued one after another, with the next layer's operands (* fused; 3 x 3 convolutions, 2 x 2 windows unless said otherwise;
// int32, then 8-bit activations, shifts to 14):
//   7 x 7 stem of 224 x 224, 3 x 3 stride 2    1 image  24 14*  25 10*     8  40 30*  32 15*     64  224 156*  122 79*
//   64 -> 64 channels of 224 x 224             1  40 29*  28 14*           8  175 146*  103 70*
//   64 -> 128 of 112 x 112                     1  28 19*  24 10*           8  95 79*  59 37*     64  726 555*  460 246*
//   128 -> 256 of 56 x 56                      1  26 29   25 14*           8  83 81*  50 38*     64  579 520*  306 238*
//   256 -> 512 of 28 x 28                      1  25 50   25 23*           8  83 79*  48 37*     64  500 522   260 245*
//   512 -> 512 of 28 x 28                      1  37 117  24 41            8  144 154  75 74*    64  932 1060  462 479*
//   512 -> 512 of 14 x 14                      1  25 116  24 39            8  52 115  31 41      64  253 309   130 146
//   256 -> 256 of 13 x 13, 3 x 3 stride 2      1  25 49   24 23*           8  25 49   24 23*     64  75 77     44 36*
//   64 -> 192 of 27 x 27, 5 x 5 then 3 x 3 / 2 1  24 37   24 18*           8  38 38   25 18*     64  151 166   84 78
//   32 images, 64 -> 64 of 32 x 32, stride 1   3 x 3  41 32*  32 15*       5 x 5  63 43*  55 24*     11 x 11  147 105*  138 61*
//     512 -> 64                                3 x 3  101 159  58 74       5 x 5  124 242  81 95     11 x 11  209 619   166 289
//   128 images, 64 -> 128 of 16 x 16  44 28*  34 13*       128 -> 256 of 8 x 8  43 42  30 20*       512 -> 512 of 2 x 2  29 228  24 83
constexpr double kPoolHost = 24.0;
static bool pool_pays(const MfmaPool &m, int mode, int KB, long images, long pixels, int ctiles, long cus)
{
    MfmaPool tile = m;
    const double block = mode == kI32S15 ? 0.95 : mode == kI32S7 ? 0.9 : mode == kI32S4 ? 0.5 : mode == kI8S8 ? 0.36 : 0.23;
    const double tiles = (pixels + 31) / 32 * (double)ctiles;
    const double looks = (double)images * ctiles * 64 * m.POH * m.POW * m.pk * m.pk;
    const double fused = pool_tile(tile, images * ctiles, cus) * (KB * block + 4.0);
    const double separate = 12.0 + (tiles / (8.0 * cus) + 0.07) * KB * block + tiles * 0.004 + looks * 0.4e-6;
    return fused <= (separate > kPoolHost ? separate : kPoolHost);
}

template <int MODE>
static int launch_pool(MfmaArgs &a, MfmaPool &m, unsigned grid, hipStream_t st)
{
    if (m.pk == 3)
        hipLaunchKernelGGL((mfma_pool_kernel<MODE, true>), dim3(grid), dim3(256), 0, st, a, m);
    else
        hipLaunchKernelGGL((mfma_pool_kernel<MODE, false>), dim3(grid), dim3(256), 0, st, a, m);
    return launch_status();
}

template <int SRC, bool I8>
static int launch_prepare(const PrepArgs &a, bool matrix, hipStream_t st)
{
    const dim3 grid((unsigned)((a.lay.rows + a.rpw - 1) / a.rpw), (unsigned)a.lay.fy);
    if (matrix)
        hipLaunchKernelGGL((mfma_prepare_kernel<SRC, I8, true, 16>), grid, dim3(256), 0, st, a);
    else if (a.lay.cp >= 16)
        hipLaunchKernelGGL((mfma_prepare_kernel<SRC, I8, false, 16>), grid, dim3(256), 0, st, a);
    else if (a.lay.cp == 8)
        hipLaunchKernelGGL((mfma_prepare_kernel<SRC, I8, false, 8>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((mfma_prepare_kernel<SRC, I8, false, 4>), grid, dim3(256), 0, st, a);
    return launch_status();
}

// The mode of a layer, or -1: the largest shift among its non-zero weights and the activations' width decide.
static int mode_of(int max_shift, int x_bytes)
{
    if (max_shift < 0 || max_shift > 31) return -1;
    if (x_bytes == 1) return max_shift <= 3 ? kI8S4 : kI8S8;
    if (x_bytes != 4) return -1;
    return max_shift <= 3 ? kI32S4 : max_shift <= 6 ? kI32S7 : max_shift <= 14 ? kI32S15 : -1;
}

// The formats that the conversions take (ds_quantize_f32_i32, ds_quantize_pad_f32_i8).
static bool format_ok(int I, int F, int bytes)
{
    return F >= 0 && (bytes == 1 ? I >= 2 && I + F <= 8 : I >= 1 && I + F <= 32);
}

}  // namespace ds

using namespace ds;

DS_EXPORT size_t ds_mfma_weight_bytes(int N, int C, int FH, int FW, int max_shift, int x_bytes)
{
    const int mode = mode_of(max_shift, x_bytes);
    if (mode < 0 || N <= 0 || C <= 0 || FH <= 0 || FW <= 0) return 0;
    if ((double)C * FH * FW > kMfmaMaxK) return 0;
    const MfmaGeom g = mfma_geom(N, C, FH, FW);
    if ((double)g.kb * mode_block(mode) > (double)(1u << 30)) return 0;   // 32-bit offsets within a tile
    return mfma_blob_corr(g, mode) + (size_t)g.ntiles * 32 * 4;
}

DS_EXPORT int ds_mfma_tile_weights_i32(const int32_t *w_ref, void *blob, int N, int C, int FH, int FW, int bits,
                                       int max_shift, int x_bytes, ds_stream_t stream)
{
    if (!w_ref || !blob) return DS_EINVAL;
    if (bits < 1 || bits > 6) return DS_EBITS;
    if (ds_mfma_weight_bytes(N, C, FH, FW, max_shift, x_bytes) == 0) return DS_EINVAL;
    const int mode = mode_of(max_shift, x_bytes);
    const MfmaGeom g = mfma_geom(N, C, FH, FW);
    hipStream_t st = (hipStream_t)stream;
    const long total = (long)g.ntiles * g.kb * 64;
    hipLaunchKernelGGL(mfma_tile_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st, w_ref, (int8_t *)blob, N, C,
                       FH, FW, bits, mode, g.cp, g.cb, g.taps, g.fwg, g.kb, total);
    int rc = launch_status();
    if (rc != DS_OK || !mode_i8(mode)) return rc;
    hipLaunchKernelGGL(mfma_corr_kernel, dim3((unsigned)(g.ntiles * 32)), dim3(64), 0, st, w_ref,
                       (int32_t *)((char *)blob + mfma_blob_corr(g, mode)), N, C * FH * FW, bits, mode);
    return launch_status();
}

// Bytes of the prepared activations of a padded Nb x C x Hp x Wp input (a matrix of M rows and K columns: Nb =
// ceil(M / 64), C = K, Hp = 1, Wp = 64); 0 where this path does not serve the layer.
DS_EXPORT size_t ds_mfma_input_bytes(int Nb, int C, int Hp, int Wp, int FH, int FW, int x_bytes)
{
    if (Nb <= 0 || C <= 0 || Hp <= 0 || Wp <= 0 || FH <= 0 || FW <= 0 || (x_bytes != 1 && x_bytes != 4)) return 0;
    if (Hp < FH || Wp < FW || (double)Nb * Hp >= kMaxRows) return 0;
    const MfmaGeom g = mfma_geom(1, C, FH, FW);
    const double bytes = (double)Nb * Hp * Wp * g.cb * g.cp * (x_bytes == 1 ? 1 : kDigits);
    if (bytes > 2.0e9 || (double)Nb * C * Hp * Wp > 2.0e9) return 0;
    const MfmaX x = mfma_x(Nb, C, Hp, Wp, g, x_bytes == 1);
    const size_t by_row = (size_t)x.rows * x.fy, by_tile = ((size_t)x.rows * Wp / 32 + 1) * x.c16;
    return x.planes + align_up(by_row > by_tile ? by_row : by_tile, 256);
}

DS_EXPORT int ds_mfma_prepare(const void *x, int source, void *dst, int Nb, int C, int H, int W, int ph, int pw, int FH,
                              int FW, int matrix_rows, int x_bytes, int mode, int I, int F, ds_stream_t stream)
{
    if (!x || !dst || ph < 0 || pw < 0 || ph > kMaxPad || pw > kMaxPad) return DS_EINVAL;
    if (H <= 0 || W <= 0 || H > (1 << 30) || W > (1 << 30)) return DS_EINVAL;
    const bool matrix = matrix_rows > 0;
    if (matrix && (H != 1 || W != 64 || ph || pw || Nb != ceil_div(matrix_rows, 64))) return DS_EINVAL;
    if (source < kSrcF32 || source > kSrcI8 || (source == kSrcI32 && x_bytes != 4) || (source == kSrcI8 && x_bytes != 1))
        return DS_EINVAL;
    if (source == kSrcF32 && (!format_ok(I, F, x_bytes) || (mode != DS_Q_ROUND_TO_FIXED && (mode != DS_Q_CAST || x_bytes == 1))))
        return DS_EINVAL;
    const int Hp = H + 2 * ph, Wp = W + 2 * pw;
    if (ds_mfma_input_bytes(Nb, C, Hp, Wp, FH, FW, x_bytes) == 0) return DS_EINVAL;
    PrepArgs a{};
    const MfmaGeom g = mfma_geom(1, C, FH, FW);
    a.lay = mfma_x(Nb, C, Hp, Wp, g, x_bytes == 1);
    a.x = x;
    a.dst = (int8_t *)dst;
    a.flags = (uint8_t *)dst + a.lay.planes;
    a.C = C;
    a.H = H;
    a.W = W;
    a.ph = ph;
    a.pw = pw;
    a.M = matrix_rows;
    a.K = C;
    a.vec = matrix && source != kSrcI8 && C % 4 == 0 && (uintptr_t)x % 16 == 0;
    a.per = a.lay.cbf * Wp * (a.lay.cp == 32 ? 2 : 1);
    a.rpw = a.per >= 256 ? 1 : 256 / a.per;
    a.by_per = fast_div((uint32_t)a.per);
    a.by_wp = fast_div((uint32_t)Wp);
    a.by_hp = fast_div((uint32_t)Hp);
    a.spec = make_spec(I, F, mode);
    hipStream_t st = (hipStream_t)stream;
    if (source == kSrcI8) return launch_prepare<kSrcI8, true>(a, matrix, st);
    if (source == kSrcI32) return launch_prepare<kSrcI32, false>(a, matrix, st);
    return x_bytes == 1 ? launch_prepare<kSrcF32, true>(a, matrix, st) : launch_prepare<kSrcF32, false>(a, matrix, st);
}

// ds_mfma_conv2d and ds_mfma_conv2d_pool (pool_k > 0).
static int mfma_conv2d_any(const void *prepared, const void *blob, const int32_t *bias, int32_t *y, float *out, void *q,
                           const float *scale, const float *shift, const float *residual, int Nb, int C, int Hp, int Wp,
                           int O, int FH, int FW, int sh, int sw, int crop_h, int crop_w, int prep_FH, int prep_FW,
                           int matrix_rows, int max_shift, int x_bytes, int F_in, int relu, int I, int F, int ph, int pw,
                           int q_bytes, int q_FH, int q_FW, int prep_tiles, int prep_ph, int prep_pw, int pool_k, int pool_s,
                           int pool_p, ds_stream_t stream)
{
    const int border_kept = q_bytes & DS_Q_BORDER_KEPT;
    const bool operands = (q_bytes & DS_Q_OPERANDS) != 0;
    q_bytes &= 0xff;
    if (!prepared || !blob || (!y && !out && !q) || (y && (out || q))) return DS_EINVAL;
    if (sh <= 0 || sw <= 0 || crop_h < 0 || crop_w < 0 || ph < 0 || pw < 0) return DS_EINVAL;
    if (crop_h > kMaxPad || crop_w > kMaxPad || ph > kMaxPad || pw > kMaxPad) return DS_EINVAL;
    if (q && ((q_bytes != 1 && q_bytes != 4) || !format_ok(I, F, q_bytes))) return DS_EINVAL;
    if (!y && (F_in < 0 || F_in > 31)) return DS_EINVAL;
    const int mode = mode_of(max_shift, x_bytes);
    if (mode < 0 || ds_mfma_weight_bytes(O, C, FH, FW, max_shift, x_bytes) == 0) return DS_EINVAL;
    if (ds_mfma_input_bytes(Nb, C, Hp, Wp, prep_FH, prep_FW, x_bytes) == 0) return DS_EINVAL;
    const MfmaGeom g = mfma_geom(O, C, FH, FW);
    if (g.cp != mfma_geom(O, C, prep_FH, prep_FW).cp) return DS_EINVAL;   // prepared for another grouping of taps
    const int Hc = Hp - 2 * crop_h, Wc = Wp - 2 * crop_w;
    if (Hc < FH || Wc < FW) return DS_EINVAL;
    MfmaArgs a{};
    a.lay = mfma_x(Nb, C, Hp, Wp, g, x_bytes == 1);
    a.x = (const int8_t *)prepared;
    a.flags = (const uint8_t *)prepared + a.lay.planes;
    if (prep_tiles) {
        if (prep_ph < 0 || prep_pw < 0 || Hp <= 2 * prep_ph || Wp <= 2 * prep_pw || g.cp < 16) return DS_EINVAL;
        a.lay.tiles = 1;
        a.lay.th = Hp - 2 * prep_ph;
        a.lay.tw = Wp - 2 * prep_pw;
        a.lay.tph = prep_ph;
        a.lay.tpw = prep_pw;
    }
    a.blob = (const int8_t *)blob;
    a.corr = mode_i8(mode) ? (const int32_t *)((const char *)blob + mfma_blob_corr(g, mode)) : nullptr;
    a.bias = bias;
    a.y = y;
    a.out = out;
    a.q = q;
    a.scale = scale;
    a.shift = shift;
    a.residual = residual;
    a.N = O;
    a.KB = g.kb;
    a.FH = FH;
    a.fwg = g.fwg;
    a.tapstep = g.taps * g.cp;
    a.tapstep01 = g.taps * a.lay.px01;
    a.sh = sh;
    a.sw = sw;
    a.crop_h = crop_h;
    a.crop_w = crop_w;
    a.OH = (Hc - FH) / sh + 1;
    a.OW = (Wc - FW) / sw + 1;
    const double pixels = (double)Nb * a.OH * a.OW;
    if (pixels > 1.0e9 || (double)O * pixels > 8.0e9) return DS_EINVAL;
    a.matrix = matrix_rows > 0;
    a.pixels = a.matrix ? (uint32_t)matrix_rows : (uint32_t)pixels;
    if (a.matrix && ((double)matrix_rows > pixels || q)) return DS_EINVAL;
    MfmaPool m{};
    int rows = a.OH, columns = a.OW;   // of the result
    if (pool_k) {
        if (!ds_mfma_pool_serves(a.OH, a.OW, pool_k, pool_s, pool_p) || a.matrix || y || residual || pixels * O * 4 >= 2147483648.0)
            return DS_EINVAL;
        m.pk = pool_k;
        m.ps = pool_s;
        m.pp = pool_p;
        m.POH = rows = (a.OH + 2 * pool_p - pool_k) / pool_s + 1;
        m.POW = columns = (a.OW + 2 * pool_p - pool_k) / pool_s + 1;
    }
    a.ostride_c = a.matrix ? 1 : rows * columns;
    a.ostride_n = (long)a.ostride_c * O;
    a.relu = relu;
    a.q_bytes = q_bytes;
    a.qph = ph;
    a.qpw = pw;
    a.qHp = rows + 2 * ph;
    a.qWp = columns + 2 * pw;
    if (q && (double)a.qHp * a.qWp > 2147483647.0) return DS_EINVAL;
    a.inv = ldexpf(1.0f, -F_in);
    a.unfold = ldexpf(1.0f, F_in);
    a.q_only = q && !out && !residual && relu && I != 1;
    a.qfold = a.q_only ? ldexpf(1.0f, F) : 1.0f;
    a.qspec = make_spec(I, F, DS_Q_ROUND_TO_FIXED);
    a.by_image = fast_div((uint32_t)(a.OH * a.OW));
    a.by_row = fast_div((uint32_t)a.OW);
    hipStream_t st = (hipStream_t)stream;
    if (operands) {
        if (!q || a.matrix || ds_mfma_input_bytes(Nb, O, a.qHp, a.qWp, q_FH, q_FW, q_bytes) == 0)
            return DS_EINVAL;
        const MfmaGeom qg = mfma_geom(1, O, q_FH, q_FW);
        if (qg.cp < 16) return DS_EINVAL;
        a.qlay = mfma_x(Nb, O, a.qHp, a.qWp, qg, q_bytes == 1);
        a.qflags = (uint8_t *)q + a.qlay.planes;
        if (!border_kept && (ph || pw)) {
            const unsigned blocks = (unsigned)(a.qlay.rows < 4096 ? a.qlay.rows : 4096);
            hipLaunchKernelGGL(mfma_operand_border_kernel, dim3(blocks), dim3(256), 0, st, (int8_t *)q, a.qlay, ph, pw);
        }
    } else if (q && !border_kept && (ph || pw)) {
        const long cells = (long)Nb * O * (2L * ph * a.qWp + 2L * pw * rows);
        const unsigned blocks = (unsigned)((cells + 255) / 256 < 4096 ? (cells + 255) / 256 : 4096);
        if (q_bytes == 1)
            hipLaunchKernelGGL((mfma_border_kernel<int8_t>), dim3(blocks), dim3(256), 0, st, (int8_t *)q, (long)Nb * O, a.qHp,
                               a.qWp, ph, pw);
        else
            hipLaunchKernelGGL((mfma_border_kernel<int32_t>), dim3(blocks), dim3(256), 0, st, (int32_t *)q, (long)Nb * O, a.qHp,
                               a.qWp, ph, pw);
    }
    if (pool_k) {
        a.ctiles = ceil_div(O, 64);
        a.by_ctiles = fast_div((uint32_t)a.ctiles);
        pool_tile(m, (long)Nb * a.ctiles, device_cus());
        const long grid = (long)Nb * m.tiles_h * m.tiles_w * a.ctiles;
        m.by_pw = fast_div((uint32_t)m.PW);
        m.by_tw = fast_div((uint32_t)m.tw);
        m.by_tiles_w = fast_div((uint32_t)m.tiles_w);
        m.by_tiles_h = fast_div((uint32_t)m.tiles_h);
        if (operands && q_bytes == 4) {
            const long words = (long)(align_up(((size_t)Nb * rows * columns / 32 + 1) * a.qlay.c16, 4) / 4);
            hipLaunchKernelGGL(mfma_clear_kernel, dim3((unsigned)(words / 256 < 1024 ? words / 256 + 1 : 1024)), dim3(256), 0, st,
                               (uint32_t *)a.qflags, words);
        }
        switch (mode) {
        case kI32S15: return launch_pool<kI32S15>(a, m, (unsigned)grid, st);
        case kI32S7: return launch_pool<kI32S7>(a, m, (unsigned)grid, st);
        case kI32S4: return launch_pool<kI32S4>(a, m, (unsigned)grid, st);
        case kI8S8: return launch_pool<kI8S8>(a, m, (unsigned)grid, st);
        default: return launch_pool<kI8S4>(a, m, (unsigned)grid, st);
        }
    }
    switch (mode) {
    case kI32S15: return launch_mfma<kI32S15>(a, st);
    case kI32S7: return launch_mfma<kI32S7>(a, st);
    case kI32S4: return launch_mfma<kI32S4>(a, st);
    case kI8S8: return launch_mfma<kI8S8>(a, st);
    default: return launch_mfma<kI8S4>(a, st);
    }
}

DS_EXPORT int ds_mfma_conv2d(const void *prepared, const void *blob, const int32_t *bias, int32_t *y, float *out, void *q,
                             const float *scale, const float *shift, const float *residual, int Nb, int C, int Hp, int Wp,
                             int O, int FH, int FW, int sh, int sw, int crop_h, int crop_w, int prep_FH, int prep_FW,
                             int matrix_rows, int max_shift, int x_bytes, int F_in, int relu, int I, int F, int ph, int pw,
                             int q_bytes, int q_FH, int q_FW, int prep_tiles, int prep_ph, int prep_pw,
                             ds_stream_t stream)
{
    return mfma_conv2d_any(prepared, blob, bias, y, out, q, scale, shift, residual, Nb, C, Hp, Wp, O, FH, FW, sh, sw, crop_h,
                           crop_w, prep_FH, prep_FW, matrix_rows, max_shift, x_bytes, F_in, relu, I, F, ph, pw, q_bytes, q_FH,
                           q_FW, prep_tiles, prep_ph, prep_pw, 0, 0, 0, stream);
}

// ds_mfma_conv2d and ds_mfma_conv2d_pool with their arguments in two arrays.
DS_EXPORT int ds_mfma_conv2d_packed(const void *const *p, const int32_t *d, ds_stream_t stream)
{
    if (!p || !d) return DS_EINVAL;
    return mfma_conv2d_any(p[0], p[1], (const int32_t *)p[2], (int32_t *)p[3], (float *)p[4], (void *)p[5], (const float *)p[6],
                           (const float *)p[7], (const float *)p[8], d[0], d[1], d[2], d[3], d[4], d[5], d[6], d[7], d[8], d[9],
                           d[10], d[11], d[12], d[13], d[14], d[15], d[16], d[17], d[18], d[19], d[20], d[21], d[22], d[23],
                           d[24], d[25], d[26], d[27], d[28], d[29], d[30], stream);
}

// The max pooling windows that the fused launch has a form for: at least one pixel of the image in each, and a convolution
// rectangle that fits a workgroup.
DS_EXPORT int ds_mfma_pool_serves(int OH, int OW, int pool_k, int pool_s, int pool_p)
{
    if (pool_k < 1 || pool_s < 1 || pool_p < 0 || 2 * (long)pool_p > pool_k || pool_k > 11) return 0;
    return OH > 0 && OW > 0 && OH + 2 * (long)pool_p >= pool_k && OW + 2 * (long)pool_p >= pool_k;
}

DS_EXPORT int ds_mfma_pool_pays(int Nb, int C, int OH, int OW, int O, int FH, int FW, int max_shift, int x_bytes, int pool_k,
                                int pool_s, int pool_p)
{
    if (Nb <= 0 || !ds_mfma_pool_serves(OH, OW, pool_k, pool_s, pool_p)) return 0;
    if (ds_mfma_weight_bytes(O, C, FH, FW, max_shift, x_bytes) == 0) return 0;
    const double pixels = (double)Nb * OH * OW;
    if (pixels * O * 4 >= 2147483648.0) return 0;
    MfmaPool m{};
    m.pk = pool_k;
    m.ps = pool_s;
    m.pp = pool_p;
    m.POH = (OH + 2 * pool_p - pool_k) / pool_s + 1;
    m.POW = (OW + 2 * pool_p - pool_k) / pool_s + 1;
    return pool_pays(m, mode_of(max_shift, x_bytes), mfma_geom(O, C, FH, FW).kb, Nb, (long)pixels, ceil_div(O, 64), device_cus());
}

DS_EXPORT int ds_mfma_conv2d_pool(const void *prepared, const void *blob, const int32_t *bias, float *out, void *q,
                                  const float *scale, const float *shift, int Nb, int C, int Hp, int Wp, int O, int FH, int FW,
                                  int sh, int sw, int prep_FH, int prep_FW, int max_shift, int x_bytes, int F_in, int relu,
                                  int I, int F, int ph, int pw, int q_bytes, int q_FH, int q_FW, int prep_tiles, int prep_ph,
                                  int prep_pw, int pool_k, int pool_s, int pool_p, ds_stream_t stream)
{
    if (pool_k < 1) return DS_EINVAL;
    return mfma_conv2d_any(prepared, blob, bias, nullptr, out, q, scale, shift, nullptr, Nb, C, Hp, Wp, O, FH, FW, sh, sw, 0, 0,
                           prep_FH, prep_FW, 0, max_shift, x_bytes, F_in, relu, I, F, ph, pw, q_bytes, q_FH, q_FW, prep_tiles,
                           prep_ph, prep_pw, pool_k, pool_s, pool_p, stream);
}
