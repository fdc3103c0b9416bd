// gemm_cost.h — estimated times (us) of the GEMM kernels, by which the planner (abi.hip) picks
// one.  Host code over sizes alone.
//
// The lines are least-squares fits to 500 layers with each kernel forced in turn (batch 2-60000,
// widths 24-4096, whole, ragged and odd; the GEMM with its epilogue and the copies, reductions
// and error kernels that the route needs).  They hold within ~10% (direct-to-LDS, fp32 register-
// staged), ~13% (K-splitting) and ~20% (fp16 register-staged).  The route that sizes take where
// the others are not ahead is direct-to-LDS where its grid fills the GPU, else register-staged;
// on those layers the choice is 3% (forward, dX) and 6% (dW) behind the best route on average and
// 1 call in 100 is more than 3% behind that route.  Ragged k no longer costs a hidden error its
// fused epilogue (65536 x 1024 below 1000: 507 -> 335 us), nor a long batch a dW its split
// (fp16 6741 x 2304 -> 1984: 167 -> 114; fp32 65536 x 1024 -> 1024: 1517 -> 1117).
#pragma once

#include <cmath>

#include "launch.h"

namespace skl {

// Another route's estimate has to be below this share of that route's: of a dW on direct-to-LDS
// tiles more, where a share of 0.97 puts 4 of 300 dWs on a route 1.2-1.46x slower.
constexpr double ROUTE_MARGIN = 0.97, DW_DMA_MARGIN = 0.85;

// What becomes of an output element: the forward's caches (three with the fused activation;
// with a norm the prenorm alone, which takes the larger tiles 0.45-0.7 of that), a plain fp32
// store, the hidden error in the epilogue (without and with a norm), the optimiser step.
enum class Work : uint32_t { Fwd, Store, Err, ErrNorm, Dw };

inline double kilo_tiles(const GemmLaunch &g, uint32_t t) {   // in units of 256 tiles: one per CU
    return (double)((g.M + t - 1) / t) * ((g.N + t - 1) / t) / 256.0;
}
inline double mega_out(const GemmLaunch &g) { return (double)g.M * g.N * 1e-6; }
// us per million elements of the optimiser's state in one pass, and of a reduction of s planes
inline double state_us(const GemmLaunch &g) { return (g.dtype == 1 ? 26.0 : 16.0) / 7.0; }
inline double reduce_us(const GemmLaunch &g, uint32_t s) { return ((g.dtype == 1 ? 26.0 : 16.0) + 8.0 * s) / 4.5; }
// the element-wise hidden-error kernel behind a GEMM that stored the sum
inline double err_us(const GemmLaunch &g, bool norm) { return norm ? 5.0 + 5.5 * mega_out(g) : 4.0 + 3.7 * mega_out(g); }

// ---- K-splitting kernel -----------------------------------------------------------------
// The larger of two lines: what one workgroup takes (lat us per k-tile of 128 bytes) and the
// GPU's rate (units of 256 workgroups times `rate` us per k-tile and `out` for the epilogue; one
// CU with one more than others sets the time of the first few units).  A dW's operands are both
// transposed in LDS: its own slopes.  64x64 tiles of 1 or 2 waves are taken only where they fill
// one round: one line.
struct WaveLine {
    uint32_t tile, waves;
    double lat, rate, lat_dw, rate_dw;
    double fix[5], out[5];   // by Work
};
// fp16, rows on 4-byte boundaries; fp16 through registers; fp32
constexpr WaveLine WAVE_F16[] = {
    {16, 16, 0.048, 0.044, 0.156, 0.153, {3.5, 2.6, 3.5, 3.6, 4.2}, {2.1, 1.40, 2.50, 3.0, 1.0}},
    {32, 4, 0.100, 0.082, 0.195, 0.166, {3.6, 2.6, 3.6, 3.9, 4.3}, {1.0, 0.58, 1.55, 2.0, 0.0}},
    {64, 4, 0.204, 0.190, 0.254, 0.235, {5.6, 3.6, 5.7, 6.8, 5.7}, {2.1, 1.20, 3.50, 5.4, 0.0}},
    {64, 2, 0.740, 0.000, 0.890, 0.000, {10.8, 5.5, 17.0, 25.0, 4.6}, {}},
};
constexpr WaveLine WAVE_REG[] = {
    {16, 16, 0.078, 0.085, 0.162, 0.206, {3.3, 3.0, 3.5, 3.5, 4.8}, {2.0, 1.80, 3.00, 3.6, 1.0}},
    {32, 8, 0.163, 0.134, 0.217, 0.243, {4.0, 3.6, 4.6, 5.1, 5.5}, {1.2, 1.10, 2.00, 2.5, 0.1}},
    {64, 4, 0.441, 0.295, 0.492, 0.354, {7.4, 5.1, 7.1, 8.6, 7.9}, {2.9, 1.70, 3.90, 5.5, 0.0}},
};
constexpr WaveLine WAVE_F32[] = {
    {16, 16, 0.057, 0.056, 0.100, 0.096, {2.8, 2.7, 3.5, 3.5, 4.6}, {2.00, 1.50, 2.5, 2.7, 1.1}},
    {32, 8, 0.153, 0.142, 0.157, 0.153, {3.8, 2.8, 4.2, 4.3, 5.1}, {1.25, 0.90, 1.7, 2.1, 0.5}},
    {64, 8, 0.520, 0.529, 0.525, 0.532, {5.8, 4.4, 6.4, 6.8, 7.0}, {4.30, 3.10, 6.0, 7.2, 1.7}},
    {64, 4, 0.553, 0.529, 0.562, 0.536, {6.2, 4.3, 6.6, 7.5, 7.1}, {2.90, 1.80, 4.1, 5.4, 0.4}},
    {64, 2, 1.950, 0.000, 1.920, 0.000, {16.0, 8.3, 20.8, 30.8, 13.7}, {}},
    {64, 1, 3.850, 0.000, 0.000, 0.000, {22.5, 12.5, 35.0, 51.0, 0.0}, {}},
};

inline double wave_us(const GemmLaunch &g, const WaveLine &l, Work w, uint32_t splits) {
    const uint32_t bk = g.dtype == 1 ? 64 : 32, i = (uint32_t)w;
    const bool dw = w == Work::Dw;
    const double kt = (double)((g.K + bk - 1) / bk) / splits, e = mega_out(g);
    double units = kilo_tiles(g, l.tile) * splits;
    if (units > 1.0 && units < 3.0) {
        units = std::ceil(units);
        if (g.dtype == 1 && !dw) units -= units < 2.5 ? 0.45 : 0.25;   // as measured: 1.25-1.75 as 1.55
    }
    double us = l.fix[i] + std::fmax((dw ? l.lat_dw : l.lat) * kt, units * ((dw ? l.rate_dw : l.rate) * kt + l.out[i]));
    if (dw) us += splits == 1 ? e * state_us(g) : 3.0 + e * reduce_us(g, splits);
    // three caches leave these tiles at ~1.5 TB/s (22073 x 760, K 64: 70 us)
    if (w == Work::Fwd) us = std::fmax(us, e * (g.dtype == 1 ? 4.2 : 5.8) * (g.fwd.fuse_act ? 1.0 : 0.6));
    return us;
}

// ... on the tiles and waves that the launcher takes.
inline double wave_us(const GemmLaunch &g, Work w, uint32_t tile, uint32_t splits) {
    const bool reg = !wave_dword_rows(g);
    const WaveLine *l = g.dtype == 0 ? WAVE_F32 : reg ? WAVE_REG : WAVE_F16;
    const uint32_t waves = gemm_wave_waves(g, tile);
    while (l->tile != tile || l->waves != waves) ++l;
    return wave_us(g, *l, w, splits);
}

// ---- the other kernels ------------------------------------------------------------------
// fix + k-tiles x the larger of `lat` and `rate` per unit of 256 tiles and `round` per round of
// them + out per million elements
struct TileLine {
    double fix, lat, rate, round, out;
};
inline double tile_us(const TileLine &l, double kt, double units, double e) {
    return l.fix + kt * std::fmax(l.lat, l.rate * units + l.round * std::ceil(units)) + l.out * e;
}

// Register-staged kernels on 128x128 tiles, or 64x64 (small: fp32 grids below 192 of them).
// vec: 16-byte rows (else they are gathered element by element).
inline double staged_us(const GemmLaunch &g, Work w, uint32_t splits, bool small, bool vec) {
    const bool f16 = g.dtype == 1;
    const double kt = (double)((g.K + (f16 ? 63 : 31)) / (f16 ? 64 : 32)) / splits, e = mega_out(g);
    const double units = kilo_tiles(g, small ? 64 : 128) * splits;
    if (w == Work::Dw) {
        static const TileLine dw[5][2] = {   // fp16 whole, split; fp32 whole, split, small
            {{17.9, 5.20, 0.00, 4.80, 1.7}, {17.2, 1.14, 0.19, 0.60, 0.0}},
            {{10.8, 3.40, 0.58, 3.80, 0.0}, {5.4, 1.29, 0.50, 0.00, 0.0}},
            {{5.1, 0.70, 0.00, 2.97, 1.5}, {24.3, 0.70, 0.22, 1.89, 0.0}},
            {{7.3, 3.15, 0.54, 2.40, 0.0}, {7.8, 0.88, 0.04, 2.03, 0.0}},
            {{9.0, 0.97, 1.00, 0.00, 10.8}, {8.2, 0.94, 0.59, 0.15, 0.6}}};
        return tile_us(dw[f16 ? splits > 1 : small ? 4 : 2 + (splits > 1)][vec], kt, units, e) +
               (splits > 1 ? 3.0 + e * reduce_us(g, splits) : e * state_us(g));
    }
    static const TileLine lines[3][2][2] = {   // [fp16, fp32, fp32 small][forward][vec]
        {{{2.8, 3.20, 0.00, 2.10, 1.4}, {4.1, 0.72, 0.00, 0.52, 0.7}},
         {{10.9, 3.60, 0.65, 3.00, 4.4}, {10.4, 1.00, 0.00, 0.55, 1.4}}},
        {{{7.9, 0.70, 0.28, 2.72, 0.0}, {6.1, 2.05, 0.13, 1.89, 0.5}},
         {{5.7, 0.70, 0.00, 3.20, 2.4}, {8.9, 0.00, 0.49, 1.78, 1.2}}},
        {{{2.4, 1.16, 0.26, 0.78, 1.6}, {2.8, 0.72, 0.01, 0.58, 0.7}},
         {{5.7, 1.20, 0.35, 0.68, 4.9}, {4.6, 0.82, 0.10, 0.58, 1.35}}}};
    TileLine l = lines[f16 ? 0 : small ? 2 : 1][w == Work::Fwd][vec];
    if (w == Work::Fwd && !g.fwd.fuse_act) l.out *= 0.45;
    return tile_us(l, kt, units, e);
}

// Direct-to-LDS kernel on (padded) whole tiles: rounds of 256 256x256 tiles times 128 k, the
// copies, the output.  A dW's `rounds` is the planner's estimate of its loop in us.
inline double dma_us(const GemmLaunch &g, Work w, double rounds, double pad_us, uint32_t splits) {
    static const struct { double fix, round, pad, out; } l[5] = {{9.3, 2.27, 1.44, 1.7}, {4.6, 2.67, 0.53, 0.86},
                                                                 {0.0, 2.83, 0.42, 3.15}, {0.0, 2.97, 0.03, 5.4},
                                                                 {0.0, 0.76, 0.86, 1.56}};
    const auto &p = l[(uint32_t)w];
    const double e = mega_out(g), us = p.fix + p.round * rounds + p.pad * pad_us;
    if (w == Work::Dw) return us + e * state_us(g) * p.out + (splits > 1 ? 3.0 + e * 4.0 * splits / 4.5 : 0.0);
    return us + e * p.out * (w == Work::Fwd && !g.fwd.fuse_act ? 0.45 : 1.0);
}

// ... and on 128x128 tiles over operands as stored (rag: not whole tiles).
inline double dma128_us(const GemmLaunch &g, Work w, bool rag) {
    static const TileLine whole[4] = {{8.2, 0.57, 0.476, 0.0, 0.97}, {3.4, 0.433, 0.462, 0.0, 0.55},
                                      {11.6, 0.506, 0.506, 0.0, 2.54}, {17.4, 0.62, 0.514, 0.0, 4.5}};
    static const TileLine ragged[2] = {{9.7, 0.50, 0.50, 0.0, 1.4}, {5.1, 0.434, 0.551, 0.0, 0.63}};
    TileLine l = rag ? ragged[w == Work::Store] : whole[(uint32_t)w];
    if (w == Work::Fwd && !g.fwd.fuse_act) l.out *= 0.7;
    return tile_us(l, (double)((g.K + 63) / 64), kilo_tiles(g, 128), mega_out(g));
}

// The hidden error of a layer below at most 16 outputs in the error kernel itself (elements, or
// rows where they are narrow: 44376 x 64 fp32 55 us, 117 with RMSNorm).
inline double err_skinny_us(const GemmLaunch &g, bool norm) {
    const bool f16 = g.dtype == 1;
    const double rows = g.M * 1e-3, e = mega_out(g);
    return norm ? 7.5 + std::fmax((f16 ? 5.5 : 6.2) * e, (f16 ? 1.0 : 2.0) * rows)
                : 6.5 + std::fmax((f16 ? 3.7 : 4.2) * e, (f16 ? 0.75 : 1.05) * rows);
}

// A dW of at most 16 columns is a stream over X.  The streaming kernel: 4.3 TB/s (fp16) and 4.8
// (fp32) and the reduction's serial walk over its slices.  The K-splitting kernel cannot be
// faster than ~5 TB/s, or 2.8 where rows are not 16-byte aligned or, in fp16, the odd pitch of
// either operand takes it through registers.  Streaming kernel against it: f16 4096 x 4096 ->
// 10 19 us, 16; 16384 x 2048 -> 10 26, 23; 9406 x 38336 -> 8 180, 144; 18807 x 29256 -> 7 255,
// 408; f32 42395 x 4032 -> 5 141, 117; 93006 x 5038 -> 11 403, 918.
inline double skinny_us(const GemmLaunch &g) {
    const double bytes = (double)g.M * g.K * (g.dtype == 1 ? 2.0 : 4.0);
    return 8.0 + bytes / (g.dtype == 1 ? 4.3e6 : 4.8e6) + 0.06 * skinny_dw_slices(g.K, g.M);
}
inline double narrow_wave_us(const GemmLaunch &g) {
    const uint32_t esz = g.dtype == 1 ? 2 : 4;
    const bool rows16 = (uint64_t)g.lda * esz % 16 == 0 && (reinterpret_cast<uintptr_t>(g.A) & 15u) == 0 && wave_dword_rows(g);
    return 6.0 + (double)g.M * g.K * esz / (rows16 ? 5.0e6 : 2.8e6);
}

}  // namespace skl
