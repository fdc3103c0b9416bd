// gemm_wave.hip — launcher and tile choice of the K-splitting GEMM kernel (gemm_wave.h).
#include <cmath>

#include "epilogue.h"
#include "gemm_wave.h"
#include "launch.h"

namespace skl {

// Output rows of every tensor start on a 4-element boundary.
template <typename T> static bool epi_rows4(const GemmLaunch &g) {
    auto ok = [](const void *p, size_t esz) { return (reinterpret_cast<uintptr_t>(p) & (4 * esz - 1)) == 0; };
    switch (g.op) {
    case Op::Fwd:
        return g.fwd.ldc % 4 == 0 && ok(g.fwd.bias, sizeof(T)) && ok(g.fwd.z_out, sizeof(T)) &&
               (!g.fwd.fuse_act || (ok(g.fwd.predrop, sizeof(T)) && ok(g.fwd.out, sizeof(T)) &&
                                    (!g.fwd.use_dropout || ok(g.fwd.mask, sizeof(T)))));
    case Op::InputGrad:
    case Op::DwPartial: return g.st.ldc % 4 == 0 && g.st.split_stride % 4 == 0 && ok(g.st.out, 4);
    case Op::DwOpt:
        return g.opt.ldc % 4 == 0 && ok(g.opt.master, 4) && ok(g.opt.dv, 4) && ok(g.opt.dm, 4) &&
               ok(g.opt.param, sizeof(T));
    default: return false;
    }
}

// Tiles: rows = columns = 16, 32 or 64, with the waves that share a workgroup's K.
// 16 waves of 16x16 and 4 or 8 of 32x32 or 64x64 put 64-128 KB of loads in flight per CU.
// 64x64 tiles keep two waves per SIMD resident, so the fewer waves share a tile, the more
// tiles one round holds: 4 waves and 512 tiles, or where that makes the grid one round at
// least three quarters full, 2 waves and 1024 (4096 x 1024, K 1024: f16 21.5 -> 19.9 us, f32
// 79 -> 73; a grid of 512 so: 43 -> 68, a pair of waves per CU sits on two of its SIMDs) and
// in fp32 1 wave and 2048 (8192 x 1024, K 1024: 154 -> 143).  Up to 256 tiles fp32 takes 8
// waves (1024 x 1024 dW over 4096 rows: 76 -> 70).
static uint32_t wave_share(uint32_t dtype, uint64_t tiles64) {
    if (tiles64 > 768 && tiles64 <= 1024) return 2;
    if (dtype == 0 && tiles64 > 1536 && tiles64 <= 2048) return 1;
    if (dtype == 0 && tiles64 <= 256) return 8;
    return 4;
}
static uint64_t tiles_of(const GemmLaunch &g, uint32_t t) {
    return (uint64_t)((g.M + t - 1) / t) * ((g.N + t - 1) / t);
}

template <typename T, class Epi, bool AK, bool BK, bool REG, int MB, int W, int S, int WPE>
static hipError_t run_wave_t(const GemmLaunch &g, const typename Epi::Params &p0, hipStream_t s) {
    GemmShape sh{};
    sh.M = g.M;
    sh.N = g.N;
    sh.K = g.K;
    sh.lda = g.lda;
    sh.ldb = g.ldb;
    sh.tiles_m = (g.M + 16 * MB - 1) / (16 * MB);
    sh.tiles_n = (g.N + 16 * MB - 1) / (16 * MB);
    sh.k_per_split = gemm_wave_slice(g.K, g.splits);
    sh.nv = epi_rows4<T>(g) ? 1u : 0u;
    const uint32_t splits = (g.K + sh.k_per_split - 1) / sh.k_per_split;
    if (splits > 1 && g.op != Op::DwPartial) return hipErrorInvalidValue;
    const uint32_t tiles = sh.tiles_m * sh.tiles_n;
    typename Epi::Params p = p0;
    uint32_t more = 0;
    if constexpr (std::is_same<typename Epi::Params, OptEpi>::value) {
        if (p.vec_blocks) {
            // The parameter update: columns per workgroup as given for 256 threads, in
            // workgroups of its own where the last round of tiles leaves room for them
            // (1024 x 1024 dW over 2048 rows: 22 -> 19 us), else behind the tiles (2048 x
            // 1000, 512 tiles in one full round: 48 us a step in a second round, 45 so).
            constexpr uint32_t slots = MB == 1 ? 256 : MB == 2 ? 512 : 2048 / W;   // workgroups resident at once
            static_assert(W >= 2, "the update's workgroup");
            p.vec.cpb = p.vec.cpb * W >= 4 ? p.vec.cpb * W / 4 : 1;
            const uint32_t blocks = (p.vec.n + p.vec.cpb - 1) / p.vec.cpb, last = tiles % slots;
            if (last && last + blocks <= slots) more = blocks;
            p.vec_blocks = more ? 0 : blocks;
        }
    }
    launch_timed(g, gemm_wave_kernel<T, Epi, AK, BK, REG, MB, MB, W, S, WPE>, dim3(tiles + more, splits),
                 dim3(64 * W), s, sh, reinterpret_cast<const T *>(g.A), reinterpret_cast<const T *>(g.B), p);
    return hipGetLastError();
}

// Waves per tile, on the planner's choice of 64x64 tiles and the one count of the others.
uint32_t gemm_wave_waves(const GemmLaunch &g, uint32_t tile) {
    if (tile == 16) return 16;
    const bool reg = !wave_dword_rows(g);
    if (tile == 32) return g.dtype == 0 || reg ? 8 : 4;
    if (reg) return 4;
    const uint32_t w = wave_share(g.dtype, tiles_of(g, 64));
    return w == 1 && g.op == Op::DwOpt ? 4 : w;   // one wave: too few for the parameter update
}

template <typename T, class Epi, bool AK, bool BK>
static hipError_t run_wave(const GemmLaunch &g, const typename Epi::Params &p, hipStream_t s) {
    const uint32_t waves = g.waves ? g.waves : gemm_wave_waves(g, g.tile);
    if constexpr (sizeof(T) == 2) {
        if (!wave_dword_rows(g)) {
            switch (g.tile * 32 + waves) {
            case 16 * 32 + 16: return run_wave_t<T, Epi, AK, BK, true, 1, 16, 1, 4>(g, p, s);
            case 32 * 32 + 8: return run_wave_t<T, Epi, AK, BK, true, 2, 8, 1, 4>(g, p, s);
            case 64 * 32 + 4: return run_wave_t<T, Epi, AK, BK, true, 4, 4, 1, 2>(g, p, s);
            }
            return hipErrorInvalidValue;
        }
        switch (g.tile * 32 + waves) {
        case 16 * 32 + 16: return run_wave_t<T, Epi, AK, BK, false, 1, 16, 2, 4>(g, p, s);
        case 32 * 32 + 4: return run_wave_t<T, Epi, AK, BK, false, 2, 4, 2, 2>(g, p, s);
        case 64 * 32 + 2: return run_wave_t<T, Epi, AK, BK, false, 4, 2, 1, 2>(g, p, s);
        case 64 * 32 + 4: return run_wave_t<T, Epi, AK, BK, false, 4, 4, 1, 2>(g, p, s);
        }
    } else {
        switch (g.tile * 32 + waves) {
        case 16 * 32 + 16: return run_wave_t<T, Epi, AK, BK, false, 1, 16, 2, 4>(g, p, s);
        case 32 * 32 + 8: return run_wave_t<T, Epi, AK, BK, false, 2, 8, 1, 4>(g, p, s);
        case 64 * 32 + 8: return run_wave_t<T, Epi, AK, BK, false, 4, 8, 1, 2>(g, p, s);
        case 64 * 32 + 4: return run_wave_t<T, Epi, AK, BK, false, 4, 4, 1, 2>(g, p, s);
        case 64 * 32 + 2: return run_wave_t<T, Epi, AK, BK, false, 4, 2, 1, 2>(g, p, s);
        case 64 * 32 + 1:
            if constexpr (!std::is_same<typename Epi::Params, OptEpi>::value)
                return run_wave_t<T, Epi, AK, BK, false, 4, 1, 1, 2>(g, p, s);
        }
    }
    return hipErrorInvalidValue;
}

template <typename T> static hipError_t run_wave_op(const GemmLaunch &g, hipStream_t s) {
    switch (g.op) {
    case Op::Fwd: return run_wave<T, EpiFwdK<T>, true, false>(g, g.fwd, s);
    case Op::InputGrad: return run_wave<T, EpiStoreK, true, true>(g, g.st, s);
    case Op::DwOpt: return run_wave<T, EpiOptK<T>, false, false>(g, g.opt, s);
    case Op::DwPartial: return run_wave<T, EpiStoreK, false, false>(g, g.st, s);
    case Op::HiddenErr:
        return hidden_err_wave_ok(g.err, g.N) ? run_wave<T, EpiErrK<T>, true, true>(g, g.err, s) : hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
    }
}

// Every row of both operands starts on a 4-byte boundary: direct-to-LDS loads.
bool wave_dword_rows(const GemmLaunch &g) {
    if (g.dtype == 0) return true;
    auto ok = [](const void *p, uint32_t ld) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0 && ld % 2 == 0; };
    return ok(g.A, g.lda) && ok(g.B, g.ldb);
}

// k of a slice when a dW's batch is split `splits` ways (whole k-tiles).
uint32_t gemm_wave_slice(uint32_t K, uint32_t splits) {
    return ((K + (splits ? splits : 1u) - 1u) / (splits ? splits : 1u) + 63u) / 64u * 64u;
}

// The layouts the kernel is instantiated for, and 32-bit byte offsets below 2 GiB within a
// tile's rows (k-contiguous) or within a slice of the operand (m/n-contiguous).
bool gemm_wave_ok(const GemmLaunch &g, uint32_t splits) {
    const uint64_t esz = g.dtype == 1 ? 2 : 4;
    if (!g.M || !g.N || !g.K) return false;
    const bool layout = g.op == Op::Fwd ? g.a_kcontig && !g.b_kcontig
                        : g.op == Op::InputGrad || g.op == Op::HiddenErr ? g.a_kcontig && g.b_kcontig
                        : g.op == Op::DwOpt || g.op == Op::DwPartial ? !g.a_kcontig && !g.b_kcontig : false;
    const uint64_t k = gemm_wave_slice(g.K, splits);
    auto span = [&](bool kc, uint32_t ld) { return ((kc ? 64ull : k + 64ull) * ld + g.K) * esz; };
    return layout && span(g.a_kcontig, g.lda) < (1ull << 31) && span(g.b_kcontig, g.ldb) < (1ull << 31);
}

// The choice among the three tiles (gemm_cost.h weighs the chosen one against other kernels):
// the least of their estimated times (us), the larger of two lines fitted to measurements of
// 100 shapes between 16 x 16 x 64 and 16384 x 4096 x 4096 (each within ~20%): what one
// workgroup takes (the latency of its k-tiles, kt of 128 bytes), and the GPU's rate over
// units of 256 workgroups (one per CU; a CU with one more of the first few than others
// sets the time).
//   f16: 16x16 is ahead below ~256 of its tiles, 64x64 from ~128 of its own on, 32x32
//        between (512 x 2048, K 2048: 74 / 19 / 12 us; 128 x 2048: 21 / 7.4 / 12)
//   f32: 64x64 is bound by its MFMAs (0.5 us per k-tile and unit)
// 64x64 grids that fill one round with fewer waves per tile (wave_share) have a line of
// their own.  A dW costs more per k-tile on the small tiles (both operands transposed in
// LDS) and with odd rows, and its optimiser's bytes on top.
//
// *splits (a dW that may be split): batch slices that give every CU a workgroup, of at
// least 8 k-tiles, when the partial planes' traffic and the reduction's launch cost less
// than they save: 1216 x 256 over 9952 rows 34-54 us in one piece, 20 in 3 slices; 512 x 512
// over 8192 rows 22 -> 12; 2048 x 10 over 16384 rows 31 -> 14.
uint32_t gemm_wave_tile(const GemmLaunch &g, uint32_t *splits, double *us) {
    struct Line { double l0, l1, r0, c, d, dw; };
    static const Line f16[3] = {{2.6, 0.14, 1.0, 0.085, 1.9, 1.5},
                                {2.2, 0.155, 3.0, 0.108, 0.4, 1.25},
                                {5.5, 0.17, 2.0, 0.195, 1.9, 1.0}};
    static const Line reg[3] = {{2.6, 0.15, 1.0, 0.090, 1.9, 1.5},
                                {3.0, 0.18, 3.0, 0.130, 0.6, 1.45},
                                {6.0, 0.36, 2.0, 0.230, 2.8, 1.45}};
    static const Line f32[3] = {{2.2, 0.11, 1.0, 0.060, 2.0, 1.0},
                                {3.6, 0.14, 2.0, 0.122, 1.7, 1.0},
                                {5.0, 0.51, 4.0, 0.497, 2.7, 1.0}};
    const bool dword = wave_dword_rows(g), dw = g.op == Op::DwOpt;
    const Line *l = g.dtype == 0 ? f32 : dword ? f16 : reg;
    const double kt = (double)((g.K + (g.dtype == 0 ? 31u : 63u)) / (g.dtype == 0 ? 32u : 64u));
    const double elems = (double)g.M * g.N, state = g.dtype == 0 ? 16.0 : 26.0;   // optimiser bytes per element
    const uint32_t most = *splits;
    uint32_t best = 0;
    for (uint32_t i = 0, t = 16; i < 3; ++i, t *= 2) {
        const uint64_t tiles = tiles_of(g, t);
        uint32_t fill = tiles >= 256 ? 1u : (uint32_t)(256 / tiles);   // slices that fill the CUs
        if (fill > most) fill = most;
        while (fill > 1 && kt / fill < 8.0) --fill;
        for (const uint32_t sp : {1u, fill}) {
            if (!gemm_wave_ok(g, sp)) continue;
            double units = (double)tiles * sp / 256.0;
            if (units > 1.0 && units < 3.0) units = std::ceil(units);
            const double k = kt / sp, f = dw ? l[i].dw : 1.0;
            const double lat = l[i].l0 + l[i].l1 * f * k, rate = l[i].r0 + units * (l[i].c * f * k + l[i].d);
            double e = lat > rate ? lat : rate;
            if (t == 64 && dword && sp == 1) {
                const uint32_t w = wave_share(g.dtype, tiles);
                if (w == 2) e = g.dtype == 0 ? 8.0 + 1.98 * kt : 6.5 + 0.83 * kt;
                if (w == 1 && !dw) e = 12.0 + 3.9 * kt;
            }
            if (dw) e += sp == 1 ? elems * state / 7.0e6 : 3.0 + elems * (state + 8.0 * sp) / 4.5e6;
            if (!best || e < *us) {
                best = t;
                *us = e;
                *splits = sp;
            }
        }
    }
    return best;
}

hipError_t launch_gemm_wave(const GemmLaunch &g, hipStream_t s) {
    if (!gemm_wave_ok(g, g.splits)) return hipErrorInvalidValue;
    return g.dtype == 1 ? run_wave_op<half_t>(g, s) : run_wave_op<float>(g, s);
}

}  // namespace skl
