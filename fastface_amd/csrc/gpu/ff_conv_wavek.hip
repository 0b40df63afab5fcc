// ff_conv_wavek.hip -- small grids: an output tile's K reduction shared by the
// eight waves of one workgroup (conv_wk_kernel), for the convs of small
// batches (FFK_LATENCY) and the FC head.
//
// What bounds a small launch is its chain of dependent steps: the launch
// itself (1.6 us a node in a graph of dependent launches, measured with a
// 64-byte fill), one memory round trip, the K loop, the epilogue.  With one
// 64x64 tile per four waves, a face's 256->256 14x14 layer is 16 tiles of 72
// serial K steps; sharing K among workgroups instead (split-K) shortens the
// chain but adds a round trip of int32 partial tiles through memory and an
// arrival count, 2.6 us of such a launch's 6.2.  Here a workgroup takes a
// smaller tile (16x32 to 64x64 outputs) so that about every CU has one, and
// its eight waves take every eighth 64-byte K step each, on their own:
//   * each wave streams its steps' operands into a private LDS ring
//     (direct-to-LDS buffer loads, whole 64-byte rows per lane quad, so the
//     fetches are coalesced; the same 16-row fragments loaded straight into
//     registers, 16 rows per 16 lanes, moved about half the bytes per cycle)
//     and waits for its own loads only: no barrier in the K loop;
//   * v_mfma_i32_16x16x64_i8 with the weights as the row operand: a lane
//     ends with four consecutive channels of one pixel, so partial tiles go
//     to LDS and results to memory as vectors of channels;
//   * one barrier, then every thread sums its outputs' eight partials from
//     LDS and runs the epilogue on four channels at a time, with the
//     parameters, residual bytes and BN tables fetched before the K loop.
// Measured (us per launch in a graph of 30, warm L2, split-K or 64x64 tiles
// before -> now): 256->256 @14 residual+BN 6.9 -> 3.9 at 1 face, 9.3 -> 5.1
// at 8; 512->512 @7 7.7 -> 4.9 at 1, 10.6 -> 6.9 at 16.  The tiles stop
// paying past one workgroup per CU (1x1 64->64 @56 at 8 faces as 784 tiles
// of 32x64: 9.5 us where 64x64 tiles of four waves take 4.2), which is where
// the launch rule stops.
//
// The FC head (K = 25088, 392 steps) also splits K over workgroups, four
// ways where that fits the CUs, through the split-K workspace: 12 faces
// 20.4 -> 6.9 us against the matvec, 100 faces 28.5 -> 9.6 and 512 faces
// 30.3 -> 22.7 against 128x128 tiles split eight ways (32 to 128
// workgroups).  Where the matvec and, past 704 faces, those tiles are the
// faster ones: fc_kernel.
#include "ff_conv_table.h"
#include "ff_numerics.h"
#include "ff_wavek.h"

#include <algorithm>

namespace {

// m / d by multiplication, mag = ceil(2^32 / d) (0 stands for d == 1): exact
// for every m with m * d < 2^32 (mag * d exceeds 2^32 by less than d, so the
// error m * (mag * d - 2^32) / (d * 2^32) stays below 1 / d).  The largest m
// of each divisor is checked where the kernel is chosen: block indices by
// grid_fits, pixels and K positions by the conv rules (choose_launch,
// ffk_conv_s2_shortcut, ff_conv_generic_launch).
__device__ __forceinline__ unsigned fdiv(unsigned m, unsigned mag) { return mag ? __umulhi(m, mag) : m; }

// four floats or sums in the caller's memory, which is aligned to one
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4f_mem __attribute__((ext_vector_type(4), aligned(4)));
typedef int v4i_mem __attribute__((ext_vector_type(4), aligned(4)));

constexpr int KW = 8;                                       // waves per workgroup

// A tile of MT*16 pixels and NH column halves (or one) of NT*16 channels:
// every wave has MT x NT 16x16 MFMA blocks, KG waves share a half's K steps.
template <int MT, int NT, int NH>
struct WkTile {
    static constexpr int BM = MT * 16, BN = NH * NT * 16, KG = KW / NH;
    static constexpr int PITCH = NT * 16 + 4;               // int32 row pitch of a partial tile
    static constexpr int NTH = KW * 64;
    static constexpr int GROUPS = BM * BN / 4;              // 4 consecutive channels of a pixel each
    static constexpr int GPT = (GROUPS + NTH - 1) / NTH;    // groups per thread
    static constexpr int C4 = BN / 4;                       // groups per pixel
    static constexpr int PART = KW * BM * PITCH * 4;
    // BN tables in LDS; with two halves the partial tiles leave no room, and
    // the lookups read them from memory
    static constexpr bool LUT_LDS = NH == 1;
    static constexpr int LUT_LD = LUT_LDS ? (BN * FF_LUT_PITCH + 1023) / 1024 : 0;
    static_assert(NTH % C4 == 0, "a thread keeps its channels");
};

struct WkPos {
    unsigned tile, sp;
    int m0, n0, s_beg, s_end;
};

__device__ __forceinline__ WkPos wk_pos(const WkGeom& g, int BM, int BN) {
    WkPos p;
    const unsigned bid = blockIdx.x;
    const unsigned rest = fdiv(bid, g.mag_tn);
    const unsigned tn = bid - rest * g.tiles_n;
    const unsigned tm = fdiv(rest, g.mag_split);
    p.sp = rest - tm * g.split;
    p.tile = tm * g.tiles_n + tn;
    p.m0 = (int)tm * BM;
    p.n0 = (int)tn * BN;
    p.s_beg = (int)p.sp * g.per_split;
    p.s_end = min(g.ksteps, p.s_beg + g.per_split);
    return p;
}

// tap-(0,0) input position of output pixel m
__device__ __forceinline__ void wk_pixel(const ConvArgs& a, const WkGeom& g, int m, int& base, int& ih, int& iw) {
    const unsigned mm = (unsigned)min(m, a.M - 1);
    const unsigned b = fdiv(mm, g.mag_hw);
    const unsigned rem = mm - b * g.hw;
    const unsigned oh = fdiv(rem, g.mag_wo);
    const unsigned ow = rem - oh * g.wout;
    const int r = (int)(oh * g.stride) - g.pad;
    iw = (int)(ow * g.stride) - g.pad;
    base = (((int)b * g.hin + r) * g.win + iw) * g.cin;
    ih = m < a.M ? r : -(1 << 28);
}

// tap row, tap column and element offset of K step s (a 64-channel run of
// one tap), or, SPAN (channel counts that are multiples of 16 only), of its
// 16-byte piece q; false past the reduction's end
template <bool SPAN>
__device__ __forceinline__ bool wk_tap(const WkGeom& g, int s, int q, int& kh, int& kw, int& koff) {
    if constexpr (SPAN) {
        const unsigned k = (unsigned)s * 64 + q * 16;
        const unsigned tap = fdiv(k, g.mag_cin);
        kh = (int)fdiv(tap, g.mag_kw);
        kw = (int)tap - kh * g.kw;
        koff = (kh * g.win + kw) * g.cin + (int)(k - tap * g.cin);
        return (int)k < g.ktot;
    } else {
        const unsigned tap = fdiv((unsigned)s, g.mag_cs);
        kh = (int)fdiv(tap, g.mag_kw);
        kw = (int)tap - kh * g.kw;
        koff = (kh * g.win + kw) * g.cin + (s - (int)tap * g.csteps) * 64;
        return true;
    }
}

// The second conv of a launch: none, or the 1x1 shortcut (over the compact
// block input, csteps K steps, at most one a wave) that adds the first's
// int8 result (ffk_conv_s2_shortcut).
struct WkOne {
    static constexpr bool PAIR = false;
};
struct WkPair {
    static constexpr bool PAIR = true;
    ConvArgs b;
    int cin, csteps;
};

// epilogue operands of a thread's channels, loaded ahead of the reduction
template <int GPT>
struct WkEpi {
    v4f ws, bias, slope, adds, inv;
    int add[GPT];
};

template <int MT, int NT, int NH, bool FC, bool PAIR>
__device__ __forceinline__ void wk_prefetch(const ConvArgs& a, const WkGeom& g, const WkPos& p, WkEpi<WkTile<MT, NT, NH>::GPT>& e,
                                            int8_t* lut_s, int wave) {
    typedef WkTile<MT, NT, NH> T;
    const int tid = threadIdx.x, lane = tid & 63;
    const int nc = p.n0 + (tid % T::C4) * 4;
    e.ws = e.bias = e.slope = e.adds = e.inv = v4f{0, 0, 0, 0};
    if constexpr (FC) {
        if (nc < g.cout) {
            e.ws = *reinterpret_cast<const v4f_mem*>(a.fc_ws + nc);
            e.bias = *reinterpret_cast<const v4f_mem*>(a.fc_bias + nc);
        }
    } else if (!a.out_i32 && nc < g.cout) {
        const float* P = a.params + nc;
        e.ws = *reinterpret_cast<const v4f_mem*>(P + FFK_P_WS * g.cout);
        e.bias = *reinterpret_cast<const v4f_mem*>(P + FFK_P_BIAS * g.cout);
        e.inv = *reinterpret_cast<const v4f_mem*>(P + FFK_P_INV * g.cout);
        if (a.flags & FFK_EPI_PRELU) e.slope = *reinterpret_cast<const v4f_mem*>(P + FFK_P_SLOPE * g.cout);
        if (a.flags & FFK_EPI_ADD) e.adds = *reinterpret_cast<const v4f_mem*>(P + FFK_P_ADDSCALE * g.cout);
        if ((a.flags & FFK_EPI_ADD) && !PAIR) {            // (a pair's residual is its own first result)
            const __amdgpu_buffer_rsrc_t r_add = ff_rsrc(a.add_src, (unsigned)a.M * g.cout);
#pragma unroll
            for (int q = 0; q < T::GPT; q++)
                e.add[q] = (int)__builtin_amdgcn_raw_buffer_load_b32(
                    r_add, (unsigned)(p.m0 + (tid + q * T::NTH) / T::C4) * g.cout + nc, 0, 0);
        }
    }
    if constexpr (!FC && T::LUT_LDS) {
        if ((a.flags & FFK_EPI_BN) && !a.out_i32) {        // BN tables of the tile's channels -> LDS
            constexpr int SPR = FF_LUT_PITCH / 16;
            const __amdgpu_buffer_rsrc_t r_lut = ff_rsrc(a.bn_lut, (unsigned)g.cout * 256);
#pragma unroll
            for (int k = 0; k < (T::LUT_LD + KW - 1) / KW; k++) {
                const int blk = k * KW + wave;
                if (blk < T::LUT_LD) {
                    const int slot = blk * 64 + lane;
                    const int c = slot / SPR, pc = slot - c * SPR;
                    bdma16(r_lut, pc < 16 && c < T::BN && p.n0 + c < g.cout ? (unsigned)((p.n0 + c) * 256 + pc * 16) : FF_OOB,
                           0, lut_s + blk * 1024);
                }
            }
        }
    }
}

// Partial tiles of the waves -> sums -> (exchange) -> epilogue and stores.
// A pair: `a` is the shortcut, `first` the first conv, `acc2` the shortcut's
// partial of the waves that took one of its K steps (`mine` >= 0).
template <int MT, int NT, int NH, bool FC, typename X>
__device__ __forceinline__ void wk_finish(const v4i (&acc)[MT][NT], const ConvArgs& a, const WkGeom& g, const WkPos& p,
                                          const WkEpi<WkTile<MT, NT, NH>::GPT>& ep, int8_t* smem, const int8_t* lut_s, int wave,
                                          const ConvArgs& first, const X& x2, const v4i (&acc2)[MT][NT], int mine) {
    typedef WkTile<MT, NT, NH> T;
    constexpr int GPT = T::GPT, GROUPS = T::GROUPS, NTH = T::NTH, C4 = T::C4, PITCH = T::PITCH, BM = T::BM;
    const int tid = threadIdx.x, lane = tid & 63;
    const int lr = lane & 15, lq = lane >> 4;
    const int c4 = tid % C4;
    const int nc = p.n0 + c4 * 4;
    const bool nok = nc < g.cout;
    {
        int32_t* ps = reinterpret_cast<int32_t*>(smem) + wave * BM * PITCH;
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int j = 0; j < NT; j++)
                *reinterpret_cast<v4i*>(ps + (i * 16 + lr) * PITCH + j * 16 + lq * 4) = acc[i][j];
    }
    __syncthreads();
    v4i sum[GPT];
    int resid[GPT];
#pragma unroll
    for (int q = 0; q < GPT; q++) resid[q] = X::PAIR ? 0 : ep.add[q];
#pragma unroll
    for (int q = 0; q < GPT; q++) {
        const int gi = tid + q * NTH;
        sum[q] = v4i{0, 0, 0, 0};
        if (GROUPS % NTH == 0 || gi < GROUPS) {
            // wave w holds half w % NH of K group w / NH
            const int half = c4 / (C4 / NH);
            const int32_t* ps = reinterpret_cast<const int32_t*>(smem) + (half * BM + gi / C4) * PITCH + (c4 - half * (C4 / NH)) * 4;
#pragma unroll
            for (int w = 0; w < T::KG; w++) sum[q] += *reinterpret_cast<const v4i*>(ps + w * NH * BM * PITCH);
        }
    }
    if constexpr (X::PAIR) {
        // the first conv's int8 results, then the shortcut's sums
        v4f ws = {}, bias = {}, inv = {};
        if (nok) {
            ws = *reinterpret_cast<const v4f_mem*>(first.params + FFK_P_WS * g.cout + nc);
            bias = *reinterpret_cast<const v4f_mem*>(first.params + FFK_P_BIAS * g.cout + nc);
            inv = *reinterpret_cast<const v4f_mem*>(first.params + FFK_P_INV * g.cout + nc);
        }
        __syncthreads();                                     // the first partial tiles are read
        int32_t* ps = reinterpret_cast<int32_t*>(smem);
        if (mine >= 0)
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    *reinterpret_cast<v4i*>(ps + (mine * BM + i * 16 + lr) * PITCH + j * 16 + lq * 4) = acc2[i][j];
        __syncthreads();
#pragma unroll
        for (int q = 0; q < GPT; q++) {
            const int gi = tid + q * NTH;
            uint32_t v = 0;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                float f = (float)sum[q][e];
                f = f * ws[e];
                f = f + bias[e];
                v |= (uint32_t)(uint8_t)ff::requant_haz(f * inv[e]) << (8 * e);
            }
            resid[q] = (int)v;
            sum[q] = v4i{0, 0, 0, 0};
            if (GROUPS % NTH == 0 || gi < GROUPS)
                for (int w = 0; w < x2.csteps; w++)
                    sum[q] += *reinterpret_cast<const v4i*>(ps + (w * BM + gi / C4) * PITCH + c4 * 4);
        }
    }
    if (FC && g.split > 1) {
        // the partial tiles of the K ranges, exchanged as in conv_i8_kernel:
        // device-scope (sc1) stores, waited for before the barrier and the
        // arrival count; the last workgroup to arrive sums them all
        constexpr int CPOL_SC1 = 16;
        const __amdgpu_buffer_rsrc_t r_ws = ff_rsrc(a.ws, gridDim.x * (unsigned)(GROUPS * 16));
        const unsigned base = p.tile * (unsigned)g.split * (GROUPS * 16);
#pragma unroll
        for (int q = 0; q < GPT; q++) {
            const int gi = tid + q * NTH;
            if (GROUPS % NTH == 0 || gi < GROUPS)
                __builtin_amdgcn_raw_buffer_store_b128(sum[q], r_ws, base + p.sp * (GROUPS * 16) + gi * 16, 0, CPOL_SC1);
        }
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        int* last = reinterpret_cast<int*>(smem);
        if (tid == 0)
            last[0] = __hip_atomic_fetch_add(&a.counters[p.tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
                      (unsigned)(g.split - 1);
        __syncthreads();
        if (!last[0]) return;
        if (tid == 0) __hip_atomic_store(&a.counters[p.tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int q = 0; q < GPT; q++) sum[q] = v4i{0, 0, 0, 0};
        for (int s = 0; s < g.split; s++) {
#pragma unroll
            for (int q = 0; q < GPT; q++) {
                const int gi = tid + q * NTH;
                if (GROUPS % NTH == 0 || gi < GROUPS)
                    sum[q] += __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                                                          r_ws, base + s * (GROUPS * 16) + gi * 16, 0, CPOL_SC1));
            }
        }
    }
    if constexpr (FC) {
        float* out = a.out_f32 ? a.out_f32 : a.io->out;
#pragma unroll
        for (int q = 0; q < GPT; q++) {
            const int gi = tid + q * NTH;
            const int m = p.m0 + gi / C4;
            if ((GROUPS % NTH == 0 || gi < GROUPS) && m < a.M && nok) {
                v4f o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = ff::fc_out(sum[q][e], a.in_scale, ep.ws[e], ep.bias[e]);
                *reinterpret_cast<v4f_mem*>(out + (size_t)m * g.cout + nc) = o;
            }
        }
        return;
    }
    const bool xe = (a.flags & FFK_OUT_X_EVEN) != 0;
    const __amdgpu_buffer_rsrc_t r_x = ff_rsrc(a.out, a.out ? (unsigned)(xe ? a.M / 4 : a.M) * g.cout : 0u);
    const __amdgpu_buffer_rsrc_t r_bn = ff_rsrc(a.out_bn, (a.flags & FFK_EPI_BN) ? (unsigned)a.M * g.cout : 0u);
    const __amdgpu_buffer_rsrc_t r_lut = ff_rsrc(a.bn_lut, (a.flags & FFK_EPI_BN) ? (unsigned)g.cout * 256 : 0u);
#pragma unroll
    for (int q = 0; q < GPT; q++) {
        const int gi = tid + q * NTH;
        if (GROUPS % NTH != 0 && gi >= GROUPS) break;
        const int m = p.m0 + gi / C4;
        if (m >= a.M || !nok) continue;
        if (a.out_i32) {
            *reinterpret_cast<v4i_mem*>(a.out_i32 + (size_t)m * g.cout + nc) = sum[q];
            continue;
        }
        uint32_t x = 0, bn = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            float f = (float)sum[q][e];
            if (a.flags & FFK_EPI_INSCALE) f = f * a.in_scale;
            f = f * ep.ws[e];
            f = f + ep.bias[e];
            if (a.flags & FFK_EPI_ADD) f = ff::add_residual(f, (int32_t)(int8_t)((uint32_t)resid[q] >> (8 * e)), ep.adds[e]);
            if (a.flags & FFK_EPI_PRELU) f = ff::prelu(f, ep.slope[e]);
            const int v = ff::requant_haz(f * ep.inv[e]);
            x |= (uint32_t)(uint8_t)v << (8 * e);
            if (a.flags & FFK_EPI_BN) {
                if constexpr (T::LUT_LDS) bn |= (uint32_t)(uint8_t)lut_s[(c4 * 4 + e) * FF_LUT_PITCH + v + 128] << (8 * e);
                else bn |= (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(r_lut, (unsigned)((nc + e) * 256 + v + 128), 0, 0) << (8 * e);
            }
        }
        unsigned xo = (unsigned)m * g.cout + nc;
        if (xe) {
            const unsigned b = fdiv((unsigned)m, g.mag_hw);
            const unsigned rem = (unsigned)m - b * g.hw;
            const unsigned oh = fdiv(rem, g.mag_wo), ow = rem - oh * g.wout;
            xo = ((oh | ow) & 1) ? FF_OOB : ((b * (g.hout / 2) + (oh >> 1)) * (g.wout / 2) + (ow >> 1)) * g.cout + nc;
        }
        __builtin_amdgcn_raw_buffer_store_b32(x, r_x, xo, 0, 0);
        if (a.flags & FFK_EPI_BN) __builtin_amdgcn_raw_buffer_store_b32(bn, r_bn, (unsigned)m * g.cout + nc, 0, 0);
    }
}

// MT x NT: the tile in 16x16 MFMA blocks.  D: stages of each wave's ring (a
// stage is one 64-byte K step of the tile's MT*16 pixel rows and NT*16 weight
// rows, 1 KB per 16 rows): two for the 32-channel tiles, one for the others,
// whose stages are larger (256->256 @14 at 8 faces: one 4.75 us, two 4.92;
// more stages were slower everywhere, the eight waves' loads already cover
// the latency).
// SPAN: K steps may span taps (wk_tap).  FC: the head as a 1x1 conv over 1x1
// images.
// X: WkPair, or one conv.
template <int MT, int NT, int NH, int D, bool SPAN, bool FC, typename X>
__global__ __launch_bounds__(KW * 64) void conv_wk_kernel(ConvArgs a, WkGeom g, X x2) {
    typedef WkTile<MT, NT, NH> T;
    constexpr int KG = T::KG;
    constexpr int LPS = MT + NT, STAGE = LPS * 1024;         // loads per lane, bytes per stage
    constexpr int RING = KW * D * STAGE;
    constexpr int MAIN = RING > T::PART ? RING : T::PART;
    static_assert((D - 1) * LPS < 64, "vmcnt range");
    __shared__ __align__(1024) int8_t smem[MAIN + (FC ? 0 : T::LUT_LD * 1024)];
    int8_t* lut_s = smem + MAIN;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const WkPos p = wk_pos(g, T::BM, T::BN);
    const __amdgpu_buffer_rsrc_t r_in = ff_rsrc(a.in, g.in_bytes);
    const __amdgpu_buffer_rsrc_t r_w = ff_rsrc(a.w, (unsigned)g.ksteps * g.cout * 64);
    // A 1 KB load fills four 256-byte lines of four rows: lane L takes line
    // L/16, slot L%16, whose row and 16-byte piece follow the swizzle of
    // conv_dma_kernel (dma_slot), conflict-free for the fragment reads.
    const int sl = (lane & 15) ^ ((lane >> 4) & 3);
    const int row = (lane >> 4) * 4 + (sl >> 2), q = sl & 3;
    int p_base[MT], p_ih[MT], p_iw[MT];
#pragma unroll
    for (int i = 0; i < MT; i++) {
        const int m = p.m0 + i * 16 + row;
        if constexpr (FC) {
            p_base[i] = m < a.M ? m * g.cin + q * 16 : -1;
        } else {
            wk_pixel(a, g, m, p_base[i], p_ih[i], p_iw[i]);
            if (!SPAN) p_base[i] += q * 16;
        }
    }
    unsigned w_off[NT];
#pragma unroll
    for (int j = 0; j < NT; j++) {
        const int n = p.n0 + (wave % NH) * (NT * 16) + j * 16 + row;
        w_off[j] = n < g.cout ? (unsigned)(n * 64 + q * 16) : FF_OOB;
    }
    int8_t* ring = smem + wave * D * STAGE;
    // this wave's K steps: s_beg + kg + t*KG, t < cnt
    const int kg = wave / NH;
    const int main_cnt = (p.s_end - p.s_beg - kg + KG - 1) / KG;
    int cnt = main_cnt, mine = -1;
    if constexpr (X::PAIR) {
        // the shortcut's steps follow the first conv's in the same order: the
        // waves after its last step take them, as their last
        const int i = (kg - p.s_end) & (KG - 1);
        if (i < x2.csteps) { mine = i; cnt++; }
    }
    auto issue = [&](int t, int slot) {
        const int s = p.s_beg + kg + t * KG;
        if constexpr (X::PAIR) {
            if (t == main_cnt) {
                const __amdgpu_buffer_rsrc_t r_in2 = ff_rsrc(x2.b.in, (unsigned)a.M * x2.cin);
                const __amdgpu_buffer_rsrc_t r_w2 = ff_rsrc(x2.b.w, (unsigned)x2.csteps * g.cout * 64);
                int8_t* sb = ring + slot * STAGE;
#pragma unroll
                for (int j = 0; j < NT; j++) bdma16(r_w2, w_off[j], (unsigned)mine * (unsigned)(g.cout * 64), sb + (MT + j) * 1024);
#pragma unroll
                for (int i = 0; i < MT; i++)
                    bdma16(r_in2, (unsigned)((p.m0 + i * 16 + row) * x2.cin + mine * 64 + q * 16), 0, sb + i * 1024);
                return;
            }
        }
        const unsigned wst = (unsigned)s * (unsigned)(g.cout * 64);
        int8_t* sb = ring + slot * STAGE;
#pragma unroll
        for (int j = 0; j < NT; j++) bdma16(r_w, w_off[j], wst, sb + (MT + j) * 1024);
        if constexpr (FC) {
#pragma unroll
            for (int i = 0; i < MT; i++)
                bdma16(r_in, p_base[i] >= 0 ? (unsigned)(p_base[i] + s * 64) : FF_OOB, 0, sb + i * 1024);
        } else {
            int kh, kw, koff;
            const bool kin = wk_tap<SPAN>(g, s, q, kh, kw, koff);
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const bool v = kin && (unsigned)(p_ih[i] + kh) < (unsigned)g.hin && (unsigned)(p_iw[i] + kw) < (unsigned)g.win;
                bdma16(r_in, v ? (unsigned)(p_base[i] + koff) : FF_OOB, 0, sb + i * 1024);
            }
        }
    };
    v4i acc[MT][NT], acc2[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[i][j] = acc2[i][j] = v4i{0, 0, 0, 0};
    WkEpi<T::GPT> ep;
    const ConvArgs& last = [&]() -> const ConvArgs& {
        if constexpr (X::PAIR) return x2.b;
        else return a;
    }();
    wk_prefetch<MT, NT, NH, FC, X::PAIR>(last, g, p, ep, lut_s, wave);
#pragma unroll
    for (int u = 0; u < D; u++)
        if (u < cnt) issue(u, u);
    const int rd = dma_slot(lane & 15, lane >> 4);
    int slot = 0;
    for (int t = 0; t < cnt; t++) {
        if (t + D <= cnt) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * LPS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        const int8_t* sb = ring + slot * STAGE + rd;
        v4i fp[MT], fw[NT];
#pragma unroll
        for (int i = 0; i < MT; i++) fp[i] = *reinterpret_cast<const v4i*>(sb + i * 1024);
#pragma unroll
        for (int j = 0; j < NT; j++) fw[j] = *reinterpret_cast<const v4i*>(sb + (MT + j) * 1024);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage is read: its slot is free
        if (t + D < cnt) issue(t + D, slot);
        if (X::PAIR && t == main_cnt) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc2[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[j], fp[i], acc2[i][j], 0, 0, 0);
        } else {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int j = 0; j < NT; j++)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fw[j], fp[i], acc[i][j], 0, 0, 0);
        }
        slot = slot + 1 == D ? 0 : slot + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // every load into LDS has landed
    __syncthreads();                                         // the rings are free: partial tiles go there
    wk_finish<MT, NT, NH, FC>(acc, last, g, p, ep, smem, lut_s, wave, a, x2, acc2, mine);
}

unsigned magic(unsigned d) { return d <= 1 ? 0u : (unsigned)((0x100000000ull + d - 1) / d); }

// The tiles, smallest first.
struct WkTileSize { int bm, bn; };
constexpr WkTileSize WK_TILES[WK_NTILES] = {{16, 32}, {32, 32}, {32, 64}, {48, 64}, {64, 64}};

// A grid whose blocks wk_pos can divide exactly (tiles_n, then split) and
// whose threads the launch can count.
bool grid_fits(long long tiles, long long tiles_n, int split) {
    const long long wgs = tiles * split, lim = 0xffffffffLL;
    return wgs <= lim / (KW * 64) && wgs <= lim / tiles_n && wgs <= lim / split;
}

template <bool FC, typename X>
int wk_launch(const ConvArgs& a, WkGeom& g, int tile, int split, hipStream_t s, const X& x) {
    const WkTileSize& ts = WK_TILES[tile];
    g.tiles_n = (g.cout + ts.bn - 1) / ts.bn;
    g.split = split;
    g.per_split = (g.ksteps + split - 1) / split;
    g.mag_tn = magic(g.tiles_n);
    g.mag_split = magic(split);
    const dim3 gd((unsigned)(ff_wk_tiles(tile, a.M, g.cout) * split)), bd(KW * 64);
    switch (tile) {
    case 0: hipLaunchKernelGGL((conv_wk_kernel<1, 2, 1, 2, false, FC, X>), gd, bd, 0, s, a, g, x); break;
    case 1: hipLaunchKernelGGL((conv_wk_kernel<2, 2, 1, 2, false, FC, X>), gd, bd, 0, s, a, g, x); break;
    case 2: hipLaunchKernelGGL((conv_wk_kernel<2, 4, 1, 1, false, FC, X>), gd, bd, 0, s, a, g, x); break;
    case 3: hipLaunchKernelGGL((conv_wk_kernel<3, 4, 1, 1, false, FC, X>), gd, bd, 0, s, a, g, x); break;
    default:
        // (a pair's second accumulators do not fit a 64x64 tile's registers)
        if constexpr (!X::PAIR) hipLaunchKernelGGL((conv_wk_kernel<4, 4, 1, 1, false, FC, X>), gd, bd, 0, s, a, g, x);
        break;
    }
    return ffk_check_launch(FC ? "fc launch" : "conv launch");
}

}  // namespace

long long ff_wk_tiles(int tile, long long M, int cout) {
    const WkTileSize& ts = WK_TILES[tile];
    return ((M + ts.bm - 1) / ts.bm) * ((cout + ts.bn - 1) / ts.bn);
}

// The smallest tile whose grid stays within `max_wg` workgroups, or -1.  A
// tile is taken from the K length on where its eight partial tiles cost less
// than the waves' shorter K loops save (us, the default kernels -> this one):
// 16x32 always (1x1 64->128 @28 at 1 face 3.5 -> 3.1), 32x32 and 32x64 from 9
// steps (64->64 @56 at 1 face 4.6 -> 3.8, at 2 faces 4.7 -> 4.1; the 1x1
// 128->256 @14 at 3 faces 3.8 -> 3.8), 48x64 and 64x64 from 36 (256->256 @14
// at 12 faces 7.7 -> 6.4, at 20 7.9 -> 7.1; the 18 steps of 128->256 @28 at
// 4 faces 5.1 -> 5.5, of 128->128 @56 at 8 4.8 -> 5.5).
int ff_wk_pick(long long M, int cout, int ksteps, int max_wg) {
    constexpr int min_steps[WK_NTILES] = {1, 9, 9, 36, 36};
    for (int t = 0; t < WK_NTILES; t++)
        if (ff_wk_tiles(t, M, cout) <= max_wg) return ksteps >= min_steps[t] ? t : -1;
    return -1;
}

namespace {
WkGeom conv_geom(const ConvArgs& a, const ffk_conv_desc* d) {
    WkGeom g = {};
    g.cin = d->cin; g.cout = d->cout; g.kw = d->kw; g.stride = d->stride; g.pad = d->pad;
    g.hin = d->hin; g.win = d->win;
    g.hout = (d->hin + 2 * d->pad - d->kh) / d->stride + 1;
    g.wout = (d->win + 2 * d->pad - d->kw) / d->stride + 1;
    g.hw = g.hout * g.wout;
    g.csteps = d->cin / FF_KSTEP;
    g.ktot = d->kh * d->kw * d->cin;
    g.ksteps = (g.ktot + FF_KSTEP - 1) / FF_KSTEP;
    g.mag_hw = magic(g.hw); g.mag_wo = magic(g.wout); g.mag_kw = magic(d->kw); g.mag_cs = magic(g.csteps);
    g.mag_cin = magic(g.cin);
    g.in_bytes = (unsigned)((size_t)(a.M / g.hw) * d->hin * d->win * d->cin);
    return g;
}
}  // namespace

int ff_wk_conv(const ConvArgs& a, const ffk_conv_desc* d, int tile, hipStream_t s) {
    WkGeom g = conv_geom(a, d);
    return wk_launch<false>(a, g, tile, 1, s, WkOne{});
}

// A stride-2 conv and the 1x1 shortcut that adds its result, as one launch:
// the launch saved (3 to 5 us in a
// chain) outweighs the shortcut's few K steps and a second exchange of partial
// tiles.  Measured on whole calls: 1 face 250 -> 240 us (four pairs), 8 faces
// 372 -> 364 (two), 20 faces 484 -> 479.
int ff_wk_pair(const ConvArgs& a, const ConvArgs& b, const ffk_conv_desc* c, const ffk_conv_desc* sc, int tile,
               hipStream_t s) {
    WkGeom g = conv_geom(a, c);
    return wk_launch<false>(a, g, tile, 1, s, WkPair{b, sc->cin, sc->cin / FF_KSTEP});
}

// A conv without a tuned kernel (16-byte channel runs) on 64x64 or 64x128
// tiles, one per workgroup.
int ff_wk_generic(const ConvArgs& a, const ffk_conv_desc* d, int bn, hipStream_t s) {
    WkGeom g = conv_geom(a, d);
    g.tiles_n = (g.cout + bn - 1) / bn;
    g.split = 1;
    g.per_split = g.ksteps;
    g.mag_tn = magic(g.tiles_n);
    const dim3 gd((unsigned)(((long long)a.M + 63) / 64 * g.tiles_n)), bd(KW * 64);
    const bool span = g.cin % FF_KSTEP != 0;
    if (bn == 64 && span) hipLaunchKernelGGL((conv_wk_kernel<4, 4, 1, 1, true, false, WkOne>), gd, bd, 0, s, a, g, WkOne{});
    else if (bn == 64) hipLaunchKernelGGL((conv_wk_kernel<4, 4, 1, 1, false, false, WkOne>), gd, bd, 0, s, a, g, WkOne{});
    else if (span) hipLaunchKernelGGL((conv_wk_kernel<4, 4, 2, 1, true, false, WkOne>), gd, bd, 0, s, a, g, WkOne{});
    else hipLaunchKernelGGL((conv_wk_kernel<4, 4, 2, 1, false, false, WkOne>), gd, bd, 0, s, a, g, WkOne{});
    return ffk_check_launch("generic conv launch");
}

// The FC head: four K ranges where a tile's grid then fits the CUs, two with
// the 64x64 tiles above that (513 to 1024 faces of 512 outputs), else one.
// (Measured with 1, 2, 4, 7, 8, 14, 16 and 28 ranges at 1-2000 faces: four is
// the fastest up to 512; more ranges pay more for the exchange than their
// shorter loops save.)  ws_bytes: the workspace at hand; a plan that needs
// more runs whole K on the smallest tile that fits the CUs.
WkFcPlan ff_wk_fc_plan(int batch, int n, int k, size_t ws_bytes) {
    for (int split = 4; split >= 2; split /= 2)
        for (int t = split == 2 ? WK_NTILES - 1 : 0; t < WK_NTILES; t++) {
            const long long wgs = ff_wk_tiles(t, batch, n) * split;
            if (wgs > FF_WK_MAX_WG) continue;
            const size_t need = FF_SPLIT_COUNTER_BYTES + (size_t)wgs * WK_TILES[t].bm * WK_TILES[t].bn * sizeof(int32_t);
            if (need <= ws_bytes) return {t, split, need};
        }
    for (int t = 0; t < WK_NTILES; t++)
        if (ff_wk_tiles(t, batch, n) <= FF_WK_MAX_WG) return {t, 1, 0};
    return {WK_NTILES - 1, 1, 0};
}

// Heads this kernel takes: buffers below 2 GiB, vectors of four outputs, and
// a grid that fits (65537 column tiles of 64 fail from the second row tile
// on).  A plan with fewer workgroups than FF_WK_MAX_WG always fits, so the
// whole-K plan of the most tiles decides.
bool ff_wk_fc_fits(int batch, int n, int k) {
    const long long lim = 0x7fffffffLL;
    if ((n & 3) || (long long)batch * k > lim || (long long)n * k > lim) return false;
    const WkFcPlan p = ff_wk_fc_plan(batch, n, k, 0);
    const int bn = WK_TILES[p.tile].bn;
    return grid_fits(ff_wk_tiles(p.tile, batch, n), (n + bn - 1) / bn, p.split);
}

int ff_wk_fc(const ffk_fc_desc* d, hipStream_t s) {
    const WkFcPlan p = ff_wk_fc_plan(d->batch, d->n, d->k, d->workspace ? d->workspace_bytes : 0);
    ConvArgs a = {};
    a.in = d->a;
    a.w = d->w;
    a.fc_ws = d->ws;
    a.fc_bias = d->bias;
    a.io = d->io;
    a.out_f32 = d->out;
    a.M = d->batch;
    a.in_scale = d->a_scale;
    if (p.split > 1) {
        a.counters = (unsigned*)d->workspace;
        a.ws = (int32_t*)((int8_t*)d->workspace + FF_SPLIT_COUNTER_BYTES);
    }
    WkGeom g = {};
    g.cin = d->k; g.cout = d->n;
    g.ksteps = d->k / FF_KSTEP;
    g.in_bytes = (unsigned)((size_t)d->batch * d->k);
    return wk_launch<true>(a, g, p.tile, p.split, s, WkOne{});
}
