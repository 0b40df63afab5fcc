// ff_wavek.h -- the wave-split kernel's geometry and host interface
// (ff_conv_wavek.hip).
#pragma once
#include "ff_conv_table.h"

struct WkGeom {
    int cin, cout, kw, stride, pad, hin, win, hout, wout, hw;
    int ktot, ksteps, csteps;       // the reduction, its 64-byte K steps, those of one tap
    int tiles_n, split, per_split;  // column tiles, K ranges, steps per range
    unsigned mag_hw, mag_wo, mag_kw, mag_cs, mag_cin, mag_tn, mag_split;   // divisors' multipliers
    unsigned in_bytes;
};

constexpr int WK_NTILES = 5;        // 16x32, 32x32, 32x64, 48x64, 64x64 (pixels x channels)
// Grids up to one workgroup per CU; of each half where two halves of a batch
// run at once (FFK_SHARED_GPU), up to half of that.
constexpr int FF_WK_MAX_WG = 256;
constexpr int FF_WK_MAX_WG_SHARED = 128;

long long ff_wk_tiles(int tile, long long M, int cout);
int ff_wk_pick(long long M, int cout, int ksteps, int max_wg);
int ff_wk_conv(const ConvArgs& a, const ffk_conv_desc* d, int tile, hipStream_t s);
int ff_wk_pair(const ConvArgs& a, const ConvArgs& b, const ffk_conv_desc* c, const ffk_conv_desc* sc, int tile,
               hipStream_t s);
int ff_wk_generic(const ConvArgs& a, const ffk_conv_desc* d, int bn, hipStream_t s);

struct WkFcPlan { int tile, split; size_t ws_bytes; };
WkFcPlan ff_wk_fc_plan(int batch, int n, int k, size_t ws_bytes);
bool ff_wk_fc_fits(int batch, int n, int k);
int ff_wk_fc(const ffk_fc_desc* d, hipStream_t s);
