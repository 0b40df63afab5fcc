// ff_conv_generic.hip -- any conv geometry the tuned kernel table does not
// hold (the reference's im2col + GEMM path takes every shape:
// kernels/conv2d_nhwc.c:150-220): an implicit GEMM with the geometry in
// registers instead of template parameters.
//
// 64- or 128-wide output tiles, four waves of 32x32x32 i8 MFMAs.  Channel
// counts that are multiples of 16 load the A operand (16-byte channel runs
// of the NHWC input) and the B operand (packed weights) straight into a
// double-buffered LDS ring (conv_generic_dma_kernel); other channel counts
// stage it through registers, in 8-byte runs or byte by byte (any channel
// count; the 3-channel input layer quantizes fp32 faces or maps uint8 pixels
// on the fly).  The epilogue is the tuned kernels' per element (in-scale,
// ws, bias, residual, PReLU, round half away, with the x86 out-of-range case
// unless FFK_EPI_IN_RANGE), then X, its even pixels only or BN(X) through the
// channel's table.  No LDS reuse of the input patch: each tap's run is read
// from L2 / HBM for every output pixel.
#include "ff_conv_table.h"
#include "ff_numerics.h"
#include "ff_wavek.h"

#include <algorithm>

namespace {

struct GenGeom {
    int cin, cout, kh, kw, stride, pad, hin, win, hout, wout;
    int ktot;       // kh * kw * cin
    int kpad;       // ktot rounded up to whole 64-byte weight steps
    int d_ci, d_tw, d_th;    // 64 = d_ci + cin * (d_tw + kw * d_th): one K step in (channel, tap column, tap row)
    int row_skip;        // (win - kw) * cin: elements a tap-row step skips
    unsigned mag_hw, mag_wo; // multipliers of the divisions by hout*wout (below 128) and wout, 0: divide
    unsigned in_bytes;   // the launch's int8 input tensor (below 2 GiB)
    int vec;             // bytes per access of the int8 outputs and the residual
};

// A thread's position k in the reduction order (kh*KW + kw)*Cin + ci: tap
// row th, tap column tw, channel ci, and off = (th*Win + tw)*Cin + ci, the
// input element's offset from the output pixel's tap (0, 0) element.
struct KCursor {
    int k, ci, th, tw, off;
};

__device__ __forceinline__ KCursor kcursor_at(const GenGeom& g, int k) {
    KCursor c;
    const int tap = k / g.cin;
    c.k = k;
    c.ci = k - tap * g.cin;
    c.th = tap / g.kw;
    c.tw = tap - c.th * g.kw;
    c.off = (c.th * g.win + c.tw) * g.cin + c.ci;
    return c;
}

// The cursor one 64-element K step on, without branches: each digit of the
// mixed-radix position wraps at most once.  (The K loop's address arithmetic is
// what its waves issue between MFMAs: with a loop over the wraps, 64-bit row
// divisions before it and four-way bounds checks, 3x3 256->256 @20 at 64 faces
// took 28.7 us, now 24.6; 5x5 63.4, now 55-57.)
__device__ __forceinline__ void kcursor_next(KCursor& c, const GenGeom& g) {
    c.k += 64;
    c.ci += g.d_ci;
    const bool w0 = c.ci >= g.cin;
    c.ci -= w0 ? g.cin : 0;
    c.tw += g.d_tw + w0;
    const bool w1 = c.tw >= g.kw;
    c.tw -= w1 ? g.kw : 0;
    const int dth = g.d_th + w1;
    c.th += dth;
    c.off += 64 + dth * g.row_skip;
}

// Image and in-image position of the tile's pixel m0 + r: b0, rem0 those of
// the tile's first pixel (uniform), r < 128.
__device__ __forceinline__ void gen_pixel(const GenGeom& g, int hw, int b0, int rem0, int r, int& b, int& oh, int& ow) {
    unsigned rem = (unsigned)(rem0 + r);
    b = b0;
    if (hw >= 128) {                                  // at most one image further
        const bool w = rem >= (unsigned)hw;
        rem -= w ? hw : 0;
        b += w;
    } else {
        const unsigned q = g.mag_hw ? __umulhi(rem, g.mag_hw) : rem;       // (hw 1: rem images on)
        b += (int)q;
        rem -= q * hw;
    }
    oh = (int)(g.mag_wo ? __umulhi(rem, g.mag_wo) : rem / (unsigned)g.wout);
    ow = (int)rem - oh * g.wout;
}

// Moves the cursor n elements on without a division: each channel wrap is
// the next tap (the next pixel of the row: off runs on), each tap-column
// wrap the next tap row (off skips Win - KW pixels).
__device__ __forceinline__ void kcursor_step(KCursor& c, const GenGeom& g, int n) {
    c.k += n;
    c.ci += n;
    c.off += n;
    while (c.ci >= g.cin) {
        c.ci -= g.cin;
        if (++c.tw == g.kw) {
            c.tw = 0;
            c.th++;
            c.off += (g.win - g.kw) * g.cin;
        }
    }
}

// The 16 A-operand bytes from cursor c on of the output pixel whose tap (0, 0)
// is input pixel (ih0, iw0) at element offset base (channel counts that are
// multiples of 16 take conv_generic_dma_kernel instead).
// RUN 8: two taps' 8-byte runs (Cin % 8 == 0) through the int8 input's
// buffer resource r_in, where padding, rows past the batch and k past K take
// the out-of-range offset and read zeros.  RUN 0: byte by byte (any Cin, and
// the 3-channel input layer, which quantizes fp32 faces or maps uint8
// pixels), zeros there by branch.
template <int RUN>
__device__ __forceinline__ v4i gather_a(const ConvArgs& a, const GenGeom& g, __amdgpu_buffer_rsrc_t r_in,
                                        const void* x, bool mrow, long long base, int ih0, int iw0, KCursor c) {
    static_assert(RUN == 8 || RUN == 0, "16-byte runs: conv_generic_dma_kernel");
    if constexpr (RUN == 8) {
        v4i v;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h) kcursor_step(c, g, 8);
            const int ih = ih0 + c.th, iw = iw0 + c.tw;
            const bool in = mrow && c.k < g.ktot && ih >= 0 && ih < g.hin && iw >= 0 && iw < g.win;
            const unsigned off = in ? (unsigned)(base + c.off) : FF_OOB;
            const auto u = __builtin_amdgcn_raw_buffer_load_b64(r_in, off, 0, 0);
            v[2 * h] = (int)u[0];
            v[2 * h + 1] = (int)u[1];
        }
        return v;
    } else {
        v4i v = {0, 0, 0, 0};
        if (!mrow) return v;
        const bool stem = g.cin == 3;
        const bool rgb8 = stem && (a.flags & FFK_IN_RGB8);
        // (global-space pointers: the input may come through the I/O
        // descriptor, whose pointer the compiler cannot place)
        typedef const __attribute__((address_space(1))) int8_t* gi8;
        typedef const __attribute__((address_space(1))) uint8_t* gu8;
        typedef const __attribute__((address_space(1))) float* gf32;
        for (int e = 0; e < 16; e++) {
            if (e) kcursor_step(c, g, 1);
            int q = 0;
            if (c.k < g.ktot) {
                const int ih = ih0 + c.th, iw = iw0 + c.tw;
                if (ih >= 0 && ih < g.hin && iw >= 0 && iw < g.win) {
                    const long long off = base + c.off;
                    if (!stem) q = ((gi8)x)[off];
                    else if (rgb8) q = a.in_lut[c.ci * 256 + ((gu8)x)[off]];
                    else q = ff::quant_input(((gf32)x)[off], a.in_inv[c.ci]);
                }
            }
            v[e >> 2] |= (int)((uint32_t)(uint8_t)q << (8 * (e & 3)));
        }
        return v;
    }
}

// Epilogue.  The MFMAs run with the weights as the row operand, so a lane
// ends with one pixel (column lane%32) and, per 32-channel block, four groups
// of four consecutive channels: group r/4 holds channels (r/4)*8 + (lane/32)*4
// + r%4.  Each group is requantized and packed into one dword of the wave's
// staging tile, which then leaves as 16-byte chunks of a pixel's channels.
// (Stored straight from registers a 128x128 tile was 64 byte stores per lane
// of 32 bytes a row, and the BN output a table gather per element: 3x3 96->96
// @45 PReLU at 33 faces 27.4 us, now 17.0; 96->128 @35 residual+BN at 196 faces
// 129 us, now 60.)

// Channels per vector of the int8 tensors' accesses: 16, 8 or 4 bytes, the
// largest that divides the channel count and every base address; else 1
// (row_bytes).
__device__ __forceinline__ v4i chunk_load(const int8_t* p, int left, int vec) {
    v4i v = {0, 0, 0, 0};
    if (vec == 16) {
        if (left >= 16) v = *reinterpret_cast<const v4i*>(p);
        return v;
    }
    if (vec == 8) {
        typedef int v2i __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (left >= 8 * h + 8) {
                const v2i u = *reinterpret_cast<const v2i*>(p + 8 * h);
                v[2 * h] = u[0];
                v[2 * h + 1] = u[1];
            }
        return v;
    }
#pragma unroll
    for (int h = 0; h < 4; h++)
        if (left >= 4 * h + 4) v[h] = *reinterpret_cast<const int*>(p + 4 * h);
    return v;
}

__device__ __forceinline__ void chunk_store(int8_t* p, v4i v, int left, int vec) {
    if (vec == 16) {
        if (left >= 16) *reinterpret_cast<v4i*>(p) = v;
    } else if (vec == 8) {
        typedef int v2i __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int h = 0; h < 2; h++)
            if (left >= 8 * h + 8) *reinterpret_cast<v2i*>(p + 8 * h) = v2i{v[2 * h], v[2 * h + 1]};
    } else {
#pragma unroll
        for (int h = 0; h < 4; h++)
            if (left >= 4 * h + 4) *reinterpret_cast<int*>(p + 4 * h) = v[h];
    }
}

// The thread and its lane, opaque: addresses made from them are computed where
// they are used, not kept in registers across the requant (which spilled).
__device__ __forceinline__ int gen_tid() {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    return tid;
}
__device__ __forceinline__ int gen_lane() { return gen_tid() & 63; }

// Any channel count and address (vec 1): bytes, a lane per channel, so that an
// access is whole rows of the block's channels: as many rows as fit 64 lanes
// with each row's channels rounded up to a power of two.  (16 channels a lane,
// as bytes or as unaligned vectors, took twice the time or more of a whole
// launch: 1x1 256->131 @45 at 31 faces 47.5 us, now 22.9; 3x3 192->131
// residual+BN @56 at 49 faces 251, 108.)  The block: `rows` of up to ROWS
// pixels, `chans` of up to CW channels; v = get(row, channel) for a place of
// the block, put(row, channel, v).
template <int ROWS, int CW, typename G, typename P>
__device__ __forceinline__ void row_bytes(long long rows, int chans, G get, P put) {
    const int end = (int)(rows < ROWS ? rows : ROWS), w = chans < CW ? chans : CW;
    constexpr int U = 4;                               // accesses in flight
    if (end <= 0 || w <= 0) return;
    const int sh = w > 1 ? 32 - __builtin_clz(w - 1) : 0;
    const int lane = gen_lane(), step = 64 >> sh;
    const int row0 = lane >> sh, ch = lane & ((1 << sh) - 1);
    for (int r = 0; r < end; r += U * step) {
        int8_t v[U];
#pragma unroll
        for (int u = 0; u < U; u++) v[u] = get(min(r + u * step + row0, end - 1), min(ch, w - 1));
#pragma unroll
        for (int u = 0; u < U; u++)
            if (r + u * step + row0 < end && ch < w) put(r + u * step + row0, ch, v[u]);
    }
}

constexpr int GEN_NPRM = 5;                           // parameter rows the epilogue reads
constexpr int gen_stage_bytes(int MI, int NJ) { return MI * 32 * (NJ * 32 + 16); }

// The tile's parameter rows [GEN_NPRM][BN] -> LDS (before the K loop, whose
// barriers make them visible)
template <int BN>
__device__ __forceinline__ void gen_params(const ConvArgs& a, const GenGeom& g, int n0, float* prm) {
    if (a.out_i32) return;
    constexpr int rows[GEN_NPRM] = {FFK_P_WS, FFK_P_BIAS, FFK_P_SLOPE, FFK_P_ADDSCALE, FFK_P_INV};
#pragma unroll
    for (int r = 0; r < GEN_NPRM; r++)
        for (int c = threadIdx.x; c < BN; c += blockDim.x)
            prm[r * BN + c] = n0 + c < g.cout ? a.params[rows[r] * g.cout + n0 + c] : 0.0f;
}

// The BN tables go through LDS 64 at a time (pitch FF_LUT_PITCH): round j
// holds those of the j-th 32-channel block of both wave columns (all 128 of a
// tile at once would leave two workgroups per CU instead of four: 320->192
// 5x5 @65 at 8 faces, 530 workgroups, 187 us against 129).  A thread's four
// 16-byte pieces of round j:
constexpr int GEN_LUT_BYTES = 64 * FF_LUT_PITCH;

template <int NJ>
__device__ __forceinline__ void gen_lut_load(const ConvArgs& a, const GenGeom& g, int n0, int j, v4i (&t)[4]) {
    const int tid = gen_tid();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = k * 256 + tid;
        const int c = i >> 4, n = n0 + (c >> 5) * (NJ * 32) + j * 32 + (c & 31);
        typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1)));
        t[k] = v4i{0, 0, 0, 0};
        if (n < g.cout) t[k] = *reinterpret_cast<const v4i_any*>(a.bn_lut + (size_t)n * 256 + (i & 15) * 16);
    }
}

__device__ __forceinline__ void gen_lut_store(const v4i (&t)[4], int8_t* lut) {
    const int tid = gen_tid();
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const int i = k * 256 + tid;
        *reinterpret_cast<v4i*>(lut + (i >> 4) * FF_LUT_PITCH + (i & 15) * 16) = t[k];
    }
}

// Four int32 saturated to int8, packed (v_ashr_pk_i8_i32 saturates two).  An
// in-range requant value truncated to int32 and then saturated is the value
// the fp32 clamp before the truncation gives: the bounds are integers.
__device__ __forceinline__ uint32_t pack_sat_i8(int a, int b, int c, int d) {
    const uint32_t lo = (uint16_t)__builtin_amdgcn_ashr_pk_i8_i32((unsigned)a, (unsigned)b, 0);
    const uint32_t hi = (uint16_t)__builtin_amdgcn_ashr_pk_i8_i32((unsigned)c, (unsigned)d, 0);
    return __builtin_amdgcn_perm(hi, lo, 0x05040100u);
}

// The epilogue's three parts are separate functions, so that its five forms
// (gen_requant) share the code of the other two: a small launch's epilogue runs
// once, from code that is not in the instruction cache yet.

// The residual of the wave's MI x NJ blocks at tile (m0, n0 + wc) -> its
// staging tile
template <int MI, int NJ>
__device__ __forceinline__ void gen_residual(const ConvArgs& a, const GenGeom& g, long long m0, int n, int8_t* stage) {
    constexpr int P = NJ * 32 + 16;                    // staging row pitch
    constexpr int CH = NJ * 2, RPI = 64 / CH;          // 16-byte chunks per row, rows per chunk access
    const int lane = gen_lane();
    if (g.vec == 1) {
        const int8_t* src = a.add_src + (size_t)m0 * g.cout + n;
        row_bytes<MI * 32, NJ * 32>(a.M - m0, g.cout - n, [&](int row, int ch) { return src[row * g.cout + ch]; },
                                    [&](int row, int ch, int8_t v) { stage[row * P + ch] = v; });
    } else {
        constexpr int U = 4;                           // chunks in flight
        constexpr int N = MI * 32 / RPI;
        auto fetch = [&](int vec) {
#pragma unroll
            for (int k0 = 0; k0 < N; k0 += U) {
                v4i v[U];
#pragma unroll
                for (int u = 0; u < U && k0 + u < N; u++) {
                    const int nc = n + (lane % CH) * 16;
                    const long long m = m0 + lane / CH + (k0 + u) * RPI;
                    v[u] = v4i{0, 0, 0, 0};
                    if (m < a.M && nc < g.cout) v[u] = chunk_load(a.add_src + (size_t)m * g.cout + nc, g.cout - nc, vec);
                }
#pragma unroll
                for (int u = 0; u < U && k0 + u < N; u++)
                    *reinterpret_cast<v4i*>(stage + (lane / CH + (k0 + u) * RPI) * P + (lane % CH) * 16) = v[u];
                asm volatile("" ::: "memory");
            }
        };
        if (g.vec == 16) fetch(16);
        else fetch(g.vec);
    }
    __builtin_amdgcn_wave_barrier();                   // (the wave's own tile: its LDS accesses run in order)
}

// The wave's blocks (channels wc.. of the tile) -> int8 in its staging tile,
// which holds the residual.  prm: the tile's parameter rows.  RANGE and PRELU
// as in wave_epi_i8 (0 / 1 with the flags read at run time: the general
// form).  PIPE: a group's
// parameters are read one group ahead of its arithmetic (not beside the BN
// tables in flight: 128 registers keep four workgroups per CU).
template <int MI, int NJ, int BN, int RANGE, int PRELU, bool PIPE>
__device__ __forceinline__ void gen_requant(const v16i (&acc)[MI][NJ], const ConvArgs& a, int wc, int8_t* stage,
                                            const float* prm) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    constexpr int P = NJ * 32 + 16;
    const int lane = threadIdx.x & 63;
    const int lc = lane & 31, lh = lane >> 5;
    const bool add = RANGE != 2 && (a.flags & FFK_EPI_ADD), prelu = PRELU && (a.flags & FFK_EPI_PRELU);
    const bool insc = RANGE == 0 && (a.flags & FFK_EPI_INSCALE);
    struct Prm { v4f ws, bias, inv, slope, adds; };
    auto params = [&](int t) {                         // of group t: channels (t/4)*32 + (t%4)*8 + lh*4 ..
        const float* pr = prm + wc + (t >> 2) * 32 + (t & 3) * 8 + lh * 4;
        Prm p;
        p.ws = *reinterpret_cast<const v4f*>(pr);
        p.bias = *reinterpret_cast<const v4f*>(pr + BN);
        p.inv = *reinterpret_cast<const v4f*>(pr + 4 * BN);
        if (prelu) p.slope = *reinterpret_cast<const v4f*>(pr + 2 * BN);
        if (add) p.adds = *reinterpret_cast<const v4f*>(pr + 3 * BN);
        return p;
    };
    Prm nxt = params(0);
#pragma unroll
    for (int t = 0; t < NJ * 4; t++) {
        const int j = t >> 2, q = t & 3;
        const Prm p = nxt;
        if (PIPE && t + 1 < NJ * 4) nxt = params(t + 1);
#pragma unroll
        for (int i = 0; i < MI; i++) {
            uint32_t* d = reinterpret_cast<uint32_t*>(stage + (i * 32 + lc) * P + j * 32 + q * 8 + lh * 4);
            const uint32_t res = add ? *d : 0u;
            int v[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float f = (float)acc[i][j][q * 4 + e];
                if (insc) f = f * a.in_scale;
                f = f * p.ws[e];
                f = f + p.bias[e];
                if (add) f = ff::add_residual(f, (int32_t)(int8_t)(res >> (8 * e)), p.adds[e]);
                if (PRELU == 1 && prelu) f = ff::prelu(f, p.slope[e]);
                if (PRELU == 2 && prelu) f = ff::prelu_le1(f, p.slope[e]);
                if (RANGE == 0) {
                    v[e] = ff::requant_haz(f * p.inv[e]);
                } else {                               // (truncated here, clamped by the pack)
                    const float h = RANGE == 2 ? __builtin_fmaf(f, p.inv[e], copysignf(0.5f, f))
                                               : f * p.inv[e] + copysignf(0.5f, f * p.inv[e]);
                    v[e] = (int)h;
                }
            }
            *d = pack_sat_i8(v[0], v[1], v[2], v[3]);
        }
        asm volatile("" ::: "memory");                 // one group at a time: bounds the live parameters
        if (!PIPE && t + 1 < NJ * 4) nxt = params(t + 1);
    }
    __builtin_amdgcn_wave_barrier();
}

// The wave's staging tile -> X, or X at its even pixels
template <int MI, int NJ>
__device__ __forceinline__ void gen_store_x(const ConvArgs& a, const GenGeom& g, long long m0, int n, const int8_t* stage) {
    constexpr int P = NJ * 32 + 16, CH = NJ * 2, RPI = 64 / CH;
    const int lane = gen_lane();
    if (a.flags & FFK_OUT_X_EVEN) {
        const unsigned hw = (unsigned)(g.hout * g.wout);
#pragma unroll 1
        for (int k = 0; k < MI * 32 / RPI; k++) {
            const int row = lane / CH + k * RPI, ch = (lane % CH) * 16;
            const long long m = m0 + row;
            if (m >= a.M || n + ch >= g.cout) continue;
            const unsigned bb = (unsigned)m / hw, rem = (unsigned)m - bb * hw;
            const unsigned oh = rem / (unsigned)g.wout, ow = rem - oh * g.wout;
            if ((oh | ow) & 1) continue;
            const long long px = ((long long)bb * (g.hout / 2) + (oh >> 1)) * (g.wout / 2) + (ow >> 1);
            int8_t* dst = a.out + (size_t)px * g.cout + n + ch;
            if (g.vec > 1) chunk_store(dst, *reinterpret_cast<const v4i*>(stage + row * P + ch), g.cout - n - ch, g.vec);
            else
                for (int e = 0; e < min(16, g.cout - n - ch); e++) dst[e] = stage[row * P + ch + e];
        }
        return;
    }
    auto flush = [&](int vec) {
#pragma unroll
        for (int k = 0; k < MI * 32 / RPI; k++) {
            const int row = lane / CH + k * RPI, ch = (lane % CH) * 16;
            const long long m = m0 + row;
            if (m >= a.M || n + ch >= g.cout) continue;
            chunk_store(a.out + (size_t)m * g.cout + n + ch, *reinterpret_cast<const v4i*>(stage + row * P + ch),
                        g.cout - n - ch, vec);
        }
    };
    if (g.vec == 16) {
        flush(16);
    } else if (g.vec > 1) {
        flush(g.vec);
    } else {
        int8_t* dst = a.out + (size_t)m0 * g.cout + n;
        row_bytes<MI * 32, NJ * 32>(a.M - m0, g.cout - n, [&](int row, int ch) { return stage[row * P + ch]; },
                                    [&](int row, int ch, int8_t v) { dst[row * g.cout + ch] = v; });
    }
}

// BN(X) of the staging tile's j-th 32-channel block, through the round's
// tables (those of this wave's column at `lut`); the block is not read again
template <int MI, int NJ>
__device__ __forceinline__ void gen_bn_round(const ConvArgs& a, const GenGeom& g, long long m0, int n0, int j,
                                             int8_t* stage, const int8_t* lut) {
    constexpr int P = NJ * 32 + 16;
    const int lane = gen_lane();
    const int ch = (lane & 1) * 16, n = n0 + j * 32 + ch;
    auto flush = [&](int vec) {
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int row = i * 32 + (lane >> 1);
        const long long m = m0 + row;
        if (m >= a.M || n >= g.cout) continue;
        v4i* s = reinterpret_cast<v4i*>(stage + row * P + j * 32 + ch);
        const v4i v = *s;
        const int8_t* L = lut + ch * FF_LUT_PITCH + 128;
        v4i w;
#pragma unroll
        for (int d = 0; d < 4; d++) {
            uint32_t b[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                b[e] = (uint8_t)L[(d * 4 + e) * FF_LUT_PITCH + (int8_t)((uint32_t)v[d] >> (8 * e))];
            const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);
            const uint32_t hi = __builtin_amdgcn_perm(b[3], b[2], 0x0c0c0400u);
            w[d] = (int)__builtin_amdgcn_perm(hi, lo, 0x05040100u);
        }
        if (vec > 1) chunk_store(a.out_bn + (size_t)m * g.cout + n, w, g.cout - n, vec);
        else *s = w;
    }
    };
    if (g.vec == 16) {
        flush(16);
    } else if (g.vec > 1) {
        flush(g.vec);
    } else {
        flush(1);
        __builtin_amdgcn_wave_barrier();
        int8_t* dst = a.out_bn + (size_t)m0 * g.cout + n0 + j * 32;
        row_bytes<MI * 32, 32>(a.M - m0, g.cout - n0 - j * 32, [&](int row, int c) { return stage[row * P + j * 32 + c]; },
                               [&](int row, int c, int8_t v) { dst[row * g.cout + c] = v; });
    }
}

// All of it after the K loop: smem is the workgroup's LDS (the operands are
// consumed), gen_epi_bytes of it.
constexpr int GEN_RAW_BYTES = 4 * 16 * 36 * 4;        // (raw sums)
constexpr int gen_epi_bytes(int BM, int BN, bool LUT) {
    const int e = 4 * gen_stage_bytes(BM / 64, BN / 64) + (LUT ? GEN_LUT_BYTES : 0);
    return e > GEN_RAW_BYTES ? e : GEN_RAW_BYTES;
}

// Workgroups per CU the registers have to allow: what each tile's K loop
// needs (at 130 registers 24->256 5x5 @45 at 52 faces took 46.6 us, 39.4 at 124)
constexpr int gen_occupancy(int BM, int BN, bool LUT, int RUN) {
    const int blocks = BM / 64 * (BN / 64);
    return blocks == 4 ? (RUN != 16 && LUT ? 3 : 4) : blocks == 2 ? 5 : 6;
}

template <int BM, int BN, bool LUT>
__device__ __forceinline__ void gen_epilogue(const v16i (&acc)[BM / 64][BN / 64], const ConvArgs& a, const GenGeom& g,
                                             long long m0, int n0, int wr, int wc, int8_t* smem, const float* prm) {
    constexpr int MI = BM / 64, NJ = BN / 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (a.out_i32) {
        // raw sums: 16 pixels of a 32-channel block at a time through the wave's
        // LDS, so that a store is two rows of 32 channels (straight from
        // registers, 16 bytes of each of 32 rows, 1x1 256->132 @45 at 31 faces
        // took 20.0 us, now 18.9)
        constexpr int RP = 36, RAW = GEN_RAW_BYTES / 4; // row pitch (int32), bytes of a wave
        int32_t* st = reinterpret_cast<int32_t*>(smem + wave * RAW);
        const int lc = lane & 31, lh = lane >> 5;
        __syncthreads();                               // every wave is done with the operands
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    if (lc >> 4 == h)
#pragma unroll
                        for (int q = 0; q < 4; q++)
                            *reinterpret_cast<v4i*>(st + (lc & 15) * RP + q * 8 + lh * 4) =
                                v4i{acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]};
                    __builtin_amdgcn_wave_barrier();
                    const long long mb = m0 + wr + i * 32 + h * 16;
                    const int n = n0 + wc + j * 32 + lc;
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const int row = k * 2 + lh;
                        const int32_t v = st[row * RP + lc];
                        if (mb + row < a.M && n < g.cout) a.out_i32[(size_t)(mb + row) * g.cout + n] = v;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
        return;
    }
    int8_t* lut = smem + 4 * gen_stage_bytes(MI, NJ);
    int8_t* stage = smem + wave * gen_stage_bytes(MI, NJ);
    v4i t[4];
    if constexpr (LUT) gen_lut_load<NJ>(a, g, n0, 0, t);
    __syncthreads();                                   // every wave is done with the operands
    const int f = a.flags;
    const bool pr = (f & FFK_EPI_PRELU) != 0;
    const bool rng = (f & FFK_EPI_IN_RANGE) && !(f & FFK_EPI_INSCALE) && (!pr || (f & FFK_EPI_PRELU_LE1));
    const bool fma = rng && (f & FFK_EPI_FMA_TAIL) && !(f & FFK_EPI_ADD);
    if (f & FFK_EPI_ADD) gen_residual<MI, NJ>(a, g, m0 + wr, n0 + wc, stage);
    // (one-block tiles: 62 registers instead of 78, eight workgroups per CU: the
    // input layer, 3->64 5x5 @112 at 64 faces, 175 -> 165 us)
    constexpr bool PIPE = !LUT && MI * NJ > 1;
#define FF_GEN_EPI(RG, PR) gen_requant<MI, NJ, BN, RG, PR, PIPE>(acc, a, wc, stage, prm)
    if (!rng) FF_GEN_EPI(0, 1);
    else if (fma && pr) FF_GEN_EPI(2, 2);
    else if (fma) FF_GEN_EPI(2, 0);
    else if (pr) FF_GEN_EPI(1, 2);
    else FF_GEN_EPI(1, 0);
#undef FF_GEN_EPI
    if (a.out) gen_store_x<MI, NJ>(a, g, m0 + wr, n0 + wc, stage);
    if constexpr (LUT) {
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            if (j) __syncthreads();                    // the last round's tables are read
            gen_lut_store(t, lut);
            if (j + 1 < NJ) gen_lut_load<NJ>(a, g, n0, j + 1, t);
            __syncthreads();
            gen_bn_round<MI, NJ>(a, g, m0 + wr, n0 + wc, j, stage, lut + (wc / (NJ * 32)) * 32 * FF_LUT_PITCH);
        }
    }
}

// Channel counts that are not multiples of 16: BM x BN output tiles (64 or
// 128 each) of four waves in a 2 x 2 grid, each
// wave MI x NJ 32x32 blocks; per 64-byte K step every thread stages 16 bytes
// of BM/64 A rows (output pixels) and of BN/64 B rows (output channels) in
// LDS, then each wave runs 2 * MI * NJ 32x32x32 MFMAs; the next step's loads
// are in flight meanwhile.  A 128-wide tile halves the gathers of the other
// operand per MAC: every staged A row serves BN output channels, every B row
// BM output pixels.
template <int RUN, int BM, int BN, bool LUT>
__global__ __launch_bounds__(256, gen_occupancy(BM, BN, LUT, RUN)) void conv_generic_kernel(ConvArgs a, GenGeom g) {
    constexpr int AR = BM / 64, BR = BN / 64;          // operand rows each thread stages
    constexpr int MI = BM / 64, NJ = BN / 64;          // 32x32 blocks per wave (2 x 2 waves)
    // one 64-byte K step per barrier pair (two or four steps' pieces staged
    // at once, their loads in flight together, measured 7-48 % slower:
    // fewer waves per SIMD, the gathers' VALU work back to back)
    constexpr int PITCH = 80;                          // LDS row pitch of the staged operands
    constexpr int LDS_K = (BM + BN) * PITCH, LDS_E = gen_epi_bytes(BM, BN, LUT);
    __shared__ __align__(16) int8_t smem[LDS_K > LDS_E ? LDS_K : LDS_E];
    __shared__ __align__(16) float prm[GEN_NPRM * BN];
    int8_t* As = smem;
    int8_t* Bs = smem + BM * PITCH;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tiles_n = (g.cout + BN - 1) / BN;
    // Workgroups go round-robin over the 8 XCDs: give each XCD a contiguous
    // run of tiles (N fastest), so the tiles that gather the same pixels
    // share one L2.
    const unsigned nb = gridDim.x, bid = blockIdx.x;
    const unsigned t = (nb & 7) == 0 ? (bid & 7) * (nb >> 3) + (bid >> 3) : bid;
    const long long m0 = (long long)(t / tiles_n) * BM;
    const int n0 = (int)(t % tiles_n) * BN;
    const int hw = g.hout * g.wout;
    const void* x = g.cin != 3 ? (const void*)a.in : a.in_f32 ? (const void*)a.in_f32 : (const void*)a.io->in;

    const int r = tid >> 2, kq = (tid & 3) * 16;
    bool mrow[AR];
    int ih0[AR], iw0[AR];
    long long base[AR];          // element offset of the row's tap (0, 0) input pixel
    const int b0 = (int)((unsigned)m0 / (unsigned)hw), rem0 = (int)((unsigned)m0 - (unsigned)b0 * hw);
#pragma unroll
    for (int i = 0; i < AR; i++) {
        mrow[i] = m0 + r + 64 * i < a.M;
        int b, oh, ow;
        gen_pixel(g, hw, b0, rem0, r + 64 * i, b, oh, ow);
        ih0[i] = oh * g.stride - g.pad;
        iw0[i] = ow * g.stride - g.pad;
        base[i] = (((long long)b * g.hin + ih0[i]) * g.win + iw0[i]) * g.cin;
    }
    KCursor cur = kcursor_at(g, kq);
    const __amdgpu_buffer_rsrc_t r_in = ff_rsrc(a.in, RUN ? g.in_bytes : 0u);
    const int wr = (wave >> 1) * (BM / 2), wc = (wave & 1) * (BN / 2);
    auto load_b = [&](int k0, int i) {
        const int ncol = n0 + r + 64 * i;
        v4i v = {0, 0, 0, 0};
        if (ncol < g.cout) v = *reinterpret_cast<const v4i*>(a.w + ((size_t)(k0 >> 6) * g.cout + ncol) * 64 + kq);
        return v;
    };

    v16i acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0;
    v4i ra[AR], rb[BR];
#pragma unroll
    for (int i = 0; i < AR; i++) ra[i] = gather_a<RUN>(a, g, r_in, x, mrow[i], base[i], ih0[i], iw0[i], cur);
#pragma unroll
    for (int i = 0; i < BR; i++) rb[i] = load_b(0, i);
    gen_params<BN>(a, g, n0, prm);
    for (int k0 = 0; k0 < g.kpad; k0 += 64) {
        __syncthreads();                                  // the previous step's fragments are read
#pragma unroll
        for (int i = 0; i < AR; i++) *reinterpret_cast<v4i*>(As + (r + 64 * i) * PITCH + kq) = ra[i];
#pragma unroll
        for (int i = 0; i < BR; i++) *reinterpret_cast<v4i*>(Bs + (r + 64 * i) * PITCH + kq) = rb[i];
        __syncthreads();
        if (k0 + 64 < g.kpad) {
            kcursor_next(cur, g);
#pragma unroll
            for (int i = 0; i < AR; i++) ra[i] = gather_a<RUN>(a, g, r_in, x, mrow[i], base[i], ih0[i], iw0[i], cur);
#pragma unroll
            for (int i = 0; i < BR; i++) rb[i] = load_b(k0 + 64, i);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
            v4i A[MI], B[NJ];
#pragma unroll
            for (int i = 0; i < MI; i++)
                A[i] = *reinterpret_cast<const v4i*>(As + (wr + i * 32 + (lane & 31)) * PITCH + h * 32 + (lane >> 5) * 16);
#pragma unroll
            for (int j = 0; j < NJ; j++)
                B[j] = *reinterpret_cast<const v4i*>(Bs + (wc + j * 32 + (lane & 31)) * PITCH + h * 32 + (lane >> 5) * 16);
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(B[j], A[i], acc[i][j], 0, 0, 0);
        }
    }

    gen_epilogue<BM, BN, LUT>(acc, a, g, m0, n0, wr, wc, smem, prm);
}

// Cin % 16 == 0 (16-byte channel runs): the same tiles with the operands
// loaded straight into a GEN_NST-deep LDS ring (direct-to-LDS buffer loads:
// no register staging, the loads of GEN_NST - 1 steps in flight; two stages,
// 16-32 KB, leave room for four or five workgroups per CU, which measured
// 15-25 % faster than three or four stages with fewer workgroups).  A stage is
// BM + BN 64-byte rows in 256-byte lines of four rows, the 16-byte slot of
// (row r, piece p) ((r%4)*4 + p) XOR (r/4 % 4), as in conv_dma_kernel: the
// 16 rows a ds_read_b128 lane group reads land in 16 distinct slots.  A lane
// fetches the same piece p of its rows at every step (the swizzle picks
// which), so one K cursor per thread serves all its A rows; padding, rows
// past the batch, k past K and channels past Cout read zeros through the
// out-of-range offset.
constexpr int GEN_NST = 2;

template <int BM, int BN, bool LUT>
__global__ __launch_bounds__(256, gen_occupancy(BM, BN, LUT, 16)) void conv_generic_dma_kernel(ConvArgs a, GenGeom g) {
    constexpr int MI = BM / 64, NJ = BN / 64;          // 32x32 blocks per wave (2 x 2 waves)
    constexpr int A_BYTES = BM * 64, B_BYTES = BN * 64, STAGE = A_BYTES + B_BYTES;
    constexpr int A_LD = A_BYTES / (256 * 16), B_LD = B_BYTES / (256 * 16);
    constexpr int LPS = A_LD + B_LD;                   // loads per thread and stage
    static_assert((GEN_NST - 2) * LPS < 64, "vmcnt range");
    constexpr int LDS_K = GEN_NST * STAGE, LDS_E = gen_epi_bytes(BM, BN, LUT);
    // (one array for all of it: beside a second one the compiler waits for every
    // load into LDS before it reads LDS, so that no load overlaps the step
    // before it: 512->33 7x7 s2 @5 at 2 faces 124 us, 101 with one; 320->33 7x7
    // @35 at 21 faces 117, 101; 5x5 256->256 @14 at 256 faces, four workgroups
    // per CU, the same)
    constexpr int LDS = LDS_K > LDS_E ? LDS_K : LDS_E;
    __shared__ __align__(1024) int8_t smem[LDS + GEN_NPRM * BN * 4];
    float* prm = reinterpret_cast<float*>(smem + LDS);
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int tiles_n = (g.cout + BN - 1) / BN;
    const unsigned nb = gridDim.x, bid = blockIdx.x;
    const unsigned t = (nb & 7) == 0 ? (bid & 7) * (nb >> 3) + (bid >> 3) : bid;
    const long long m0 = (long long)(t / tiles_n) * BM;
    const int n0 = (int)(t % tiles_n) * BN;
    const int hw = g.hout * g.wout;
    const int nsteps = g.kpad / 64;
    const __amdgpu_buffer_rsrc_t r_in = ff_rsrc(a.in, g.in_bytes);
    const __amdgpu_buffer_rsrc_t r_w = ff_rsrc(a.w, (unsigned)(nsteps * g.cout * 64));

    // this thread's pieces: wave load j of wave w fills lines (4j + w)*4 ..
    // +3 of a stage's A (B) rows; lane L takes line +L/16, slot L%16, which
    // holds piece p = slot%4 XOR ... of row 4*line + slot/4
    const int sl = (lane & 15) ^ ((lane >> 4) & 3);
    const int p = sl & 3;
    int a_base[A_LD], a_ih0[A_LD], a_iw0[A_LD];
    const int b0 = (int)((unsigned)m0 / (unsigned)hw), rem0 = (int)((unsigned)m0 - (unsigned)b0 * hw);
#pragma unroll
    for (int j = 0; j < A_LD; j++) {
        const int r = ((j * 4 + wave) * 4 + (lane >> 4)) * 4 + (sl >> 2);
        int b, oh, ow;
        gen_pixel(g, hw, b0, rem0, r, b, oh, ow);
        const int ih = oh * g.stride - g.pad;
        a_iw0[j] = ow * g.stride - g.pad;
        a_base[j] = ((b * g.hin + ih) * g.win + a_iw0[j]) * g.cin;
        a_ih0[j] = m0 + r < a.M ? ih : -(1 << 28);     // a row past the batch fails every bounds check
    }
    unsigned b_off[B_LD];
#pragma unroll
    for (int j = 0; j < B_LD; j++) {
        const int n = n0 + ((j * 4 + wave) * 4 + (lane >> 4)) * 4 + (sl >> 2);
        b_off[j] = n < g.cout ? (unsigned)(n * 64 + p * 16) : FF_OOB;
    }
    // A step's A offsets.  64-row tiles are taken where there is about one
    // workgroup per CU and nothing else hides the chain of their arithmetic: they
    // are computed a step ahead, in the shadow of the fragment reads (512->33
    // 7x7 s2 @5 at 2 faces 101 -> 91 us, 320->33 7x7 @35 at 21 faces 101 ->
    // 90).  128-row tiles compute them at the loads: other workgroups of the
    // CU run meanwhile, and two more live registers cost more (5x5 256->256 @14
    // at 256 faces 102 us, 107 a step ahead).
    constexpr bool AHEAD = BM == 64;
    KCursor cur = kcursor_at(g, p * 16);
    auto a_offset = [&](int j) {
        const bool v = cur.k < g.ktot && (unsigned)(a_ih0[j] + cur.th) < (unsigned)g.hin &&
                       (unsigned)(a_iw0[j] + cur.tw) < (unsigned)g.win;
        return v ? (unsigned)(a_base[j] + cur.off) : FF_OOB;
    };
    unsigned a_off[A_LD] = {};
    auto ahead = [&]() {
        if constexpr (AHEAD) {
#pragma unroll
            for (int j = 0; j < A_LD; j++) a_off[j] = a_offset(j);
            kcursor_next(cur, g);
        }
    };
    ahead();
    auto issue = [&](int st, int buf) {
        int8_t* sb = smem + buf * STAGE;
#pragma unroll
        for (int j = 0; j < A_LD; j++)
            bdma16(r_in, AHEAD ? a_off[j] : a_offset(j), 0u, sb + (j * 4 + wave) * 1024);
        const unsigned wst = (unsigned)(st * g.cout * 64);
#pragma unroll
        for (int j = 0; j < B_LD; j++)
            bdma16(r_w, b_off[j], wst, sb + A_BYTES + (j * 4 + wave) * 1024);
        if constexpr (!AHEAD) kcursor_next(cur, g);
    };

    const int wm = wave >> 1, wn = wave & 1;
    const int a_rd = dma_slot(wm * MI * 32 + (lane & 31), lane >> 5);
    const int b_rd = A_BYTES + dma_slot(wn * NJ * 32 + (lane & 31), lane >> 5);
    v16i acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0;
#pragma unroll
    for (int u = 0; u < GEN_NST - 1; u++) {
        if (u < nsteps) issue(u, u);
        ahead();
    }
    gen_params<BN>(a, g, n0, prm);
    int rbuf = 0;                                      // ring slot of step s
    for (int st = 0; st < nsteps; st++) {
        if (st + GEN_NST - 2 < nsteps) dma_wait_barrier<(GEN_NST - 2) * LPS>();
        else dma_wait_barrier<0>();
        if (st + GEN_NST - 1 < nsteps) issue(st + GEN_NST - 1, rbuf == 0 ? GEN_NST - 1 : rbuf - 1);
        const int8_t* sb = smem + rbuf * STAGE;
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            v4i af[MI], bf[NJ];
#pragma unroll
            for (int i = 0; i < MI; i++) af[i] = *reinterpret_cast<const v4i*>(sb + ((a_rd + i * 2048) ^ (ks * 32)));
#pragma unroll
            for (int j = 0; j < NJ; j++) bf[j] = *reinterpret_cast<const v4i*>(sb + ((b_rd + j * 2048) ^ (ks * 32)));
            if (ks == 0) ahead();
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(bf[j], af[i], acc[i][j], 0, 0, 0);
        }
        rbuf = rbuf == GEN_NST - 1 ? 0 : rbuf + 1;
    }
    gen_epilogue<BM, BN, LUT>(acc, a, g, m0, n0, wm * (BM / 2), wn * (BN / 2), smem, prm);
}

// Tile shape of a launch: 128-wide in N above 64 output channels, 128-high
// in M where that still gives the 256 CUs a workgroup each, except for the
// 3-channel input layer, whose byte gather runs faster on 64-row tiles.
struct GenTile { int bm, bn; };

GenTile gen_tile(long long M, int cin, int cout) {
    GenTile t;
    t.bn = cout > 64 ? 128 : 64;
    const long long tiles_n = (cout + t.bn - 1) / t.bn;
    t.bm = cin != 3 && ((M + 127) / 128) * tiles_n >= 256 ? 128 : 64;
    return t;
}

// Grids of 64-row tiles up to one workgroup per CU and reductions of this many
// 64-byte steps run on the wave-split kernel's tiles (ff_conv_wavek.hip): eight
// waves instead of four, each with its own K steps and no barrier between them.
// (us, four-wave tiles -> these: 5x5 s2 160->192 @7 residual+BN at 20 faces, 63
// steps on 10 workgroups, 30.4 -> 14.6; 3x3 s2 160->384 @10 at 3 faces, 23
// steps, 13.0 -> 8.2; 3x3 96->96 @45 at 8 faces, 14 steps on 254 workgroups,
// 10.0 -> 7.8.  A four-stage ring in the four-wave tiles: 27.1, 12.6, 10.2,
// and slower at 400 workgroups.)
constexpr int GEN_WK_MIN_STEPS = 12;

template <int RUN, int BM, int BN, bool LUT>
void launch_tile(dim3 gd, hipStream_t s, const ConvArgs& a, const GenGeom& g) {
    if constexpr (RUN == 16) hipLaunchKernelGGL((conv_generic_dma_kernel<BM, BN, LUT>), gd, dim3(256), 0, s, a, g);
    else hipLaunchKernelGGL((conv_generic_kernel<RUN, BM, BN, LUT>), gd, dim3(256), 0, s, a, g);
}

template <int RUN, bool LUT>
void launch_run(GenTile t, dim3 gd, hipStream_t s, const ConvArgs& a, const GenGeom& g) {
    if (t.bm == 128 && t.bn == 128) launch_tile<RUN, 128, 128, LUT>(gd, s, a, g);
    else if (t.bm == 128) launch_tile<RUN, 128, 64, LUT>(gd, s, a, g);
    else if (t.bn == 128) launch_tile<RUN, 64, 128, LUT>(gd, s, a, g);
    else launch_tile<RUN, 64, 64, LUT>(gd, s, a, g);
}

// (kernels with the BN tables in LDS are separate: the tables of 128 channels
// take 34 KB)
template <int RUN>
void launch_run(GenTile t, dim3 gd, hipStream_t s, const ConvArgs& a, const GenGeom& g) {
    if ((a.flags & FFK_EPI_BN) && !a.out_i32) launch_run<RUN, true>(t, gd, s, a, g);
    else launch_run<RUN, false>(t, gd, s, a, g);
}

}  // namespace

// Workgroups of the generic kernel for M output pixels (one per tile).
long long ff_conv_generic_grid(long long M, int cin, int cout) {
    const GenTile t = gen_tile(M, cin, cout);
    return ((M + t.bm - 1) / t.bm) * ((cout + t.bn - 1) / t.bn);
}

int ff_conv_generic_launch(const ConvArgs& a, const ffk_conv_desc* d, hipStream_t s) {
    GenGeom g;
    g.cin = d->cin; g.cout = d->cout; g.kh = d->kh; g.kw = d->kw; g.stride = d->stride; g.pad = d->pad;
    g.hin = d->hin; g.win = d->win;
    g.hout = (d->hin + 2 * d->pad - d->kh) / d->stride + 1;
    g.wout = (d->win + 2 * d->pad - d->kw) / d->stride + 1;
    g.ktot = d->kh * d->kw * d->cin;
    g.kpad = (g.ktot + FF_KSTEP - 1) / FF_KSTEP * FF_KSTEP;
    g.d_ci = FF_KSTEP % g.cin;
    g.d_tw = FF_KSTEP / g.cin % g.kw;
    g.d_th = FF_KSTEP / g.cin / g.kw;
    g.row_skip = (g.win - g.kw) * g.cin;
    // multiplication by ceil(2^32 / d) divides m exactly while m * d < 2^32;
    // m is below 128 + 128 for the first, below hout*wout for the second
    auto mag = [](long long d) { return d < 2 ? 0u : (unsigned)((0x100000000ll + d - 1) / d); };
    const long long px = (long long)g.hout * g.wout;
    g.mag_hw = px < 128 ? mag(px) : 0u;
    g.mag_wo = px * g.wout < 0x100000000ll ? mag(g.wout) : 0u;
    // channel runs are read as 8- / 16-byte vectors: they need the run's
    // alignment in memory (a tensor base that is not 16-byte aligned takes
    // the byte gather)
    const int run = (d->cin == 3 || d->cin % 8 || ((uintptr_t)d->in & 15)) ? 0 : d->cin % 16 ? 8 : 16;
    uintptr_t bits = (uintptr_t)d->cout | (uintptr_t)d->out | (uintptr_t)d->out_bn;
    if (d->flags & FFK_EPI_ADD) bits |= (uintptr_t)d->add_src;
    g.vec = bits & 3 ? 1 : bits & 4 ? 4 : bits & 8 ? 8 : 16;
    // The channel-run gathers address the int8 input with 32-bit offsets: a
    // batch whose input or output tensor reaches 2 GiB runs as several
    // launches over consecutive image ranges (images are independent).  The
    // byte gather uses 64-bit addresses and takes the batch in one launch.
    const long long px_out = (long long)g.hout * g.wout;
    const long long in_img = (long long)d->hin * d->win * d->cin;
    const long long img = std::max<long long>(in_img, px_out * d->cout);
    const int slice = run == 0 ? d->batch : (int)std::min<long long>(d->batch, 0x7fffffffLL / img);
    if (slice < 1) {
        ffk_set_error("conv: one image's tensors reach 2 GiB%s%s", nullptr, nullptr);
        return FFK_ERR_ARG;
    }
    const bool x_even = (d->flags & FFK_OUT_X_EVEN) != 0;
    for (int b0 = 0; b0 < d->batch; b0 += slice) {
        const int nb = std::min(slice, d->batch - b0);
        ConvArgs as = a;
        as.M = (int)((long long)nb * px_out);
        const size_t o = (size_t)b0 * px_out * d->cout;
        if (run) as.in = a.in + (size_t)b0 * in_img;
        if (a.add_src) as.add_src = a.add_src + o;
        if (a.out) as.out = a.out + (x_even ? o / 4 : o);     // even/even pixels: a quarter
        if (a.out_bn) as.out_bn = a.out_bn + o;
        if (a.out_i32) as.out_i32 = a.out_i32 + o;
        g.in_bytes = run ? (unsigned)(nb * in_img) : 0u;
        const long long grid = ff_conv_generic_grid(as.M, d->cin, d->cout);
        if (grid > 0x7fffffffLL) {
            ffk_set_error("conv: batch too large for the generic kernel%s%s", nullptr, nullptr);
            return FFK_ERR_ARG;
        }
        const GenTile t = gen_tile(as.M, d->cin, d->cout);
        const dim3 gd((unsigned)grid);
        // (its vectors hold four channels and it fetches BN tables in 16-byte pieces, where the
        // tiles here take them at any address; its pixel arithmetic needs M * hout*wout below 2^32,
        // its K arithmetic K * cin)
        const bool lut_ok = !(d->flags & FFK_EPI_BN) || d->out_i32 || ((uintptr_t)d->bn_lut & 15) == 0;
        if (run == 16 && t.bm == 64 && grid <= FF_WK_MAX_WG && g.kpad / FF_KSTEP >= GEN_WK_MIN_STEPS && g.vec >= 4 &&
            lut_ok && as.M * px_out < 0x100000000ll && (long long)g.kpad * g.cin < 0x100000000ll) {
            const int rc = ff_wk_generic(as, d, t.bn, s);
            if (rc != FFK_OK) return rc;
            continue;
        }
        if (run == 0) launch_run<0>(t, gd, s, as, g);
        else if (run == 8) launch_run<8>(t, gd, s, as, g);
        else launch_run<16>(t, gd, s, as, g);
        const int rc = ffk_check_launch("generic conv launch");
        if (rc != FFK_OK) return rc;
    }
    return FFK_OK;
}
