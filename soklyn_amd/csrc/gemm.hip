// gemm.hip — launchers of the GEMM kernels for the three DenseBlock
// contractions (forward, dX, dW) on gfx950.
#include <stdlib.h>

#include "epilogue.h"
#include "gemm.h"
#include "gemm_dma.h"
#include "launch.h"

namespace skl {

// ---- tile configurations ----------------------------------------------------------
template <typename T, int BM, int BN, int BK, int WM, int WN> struct Cfg {
    typedef T type;
    static constexpr int bm = BM, bn = BN, bk = BK, wm = WM, wn = WN, nt = WM * WN * 64;
};
typedef Cfg<half_t, 256, 256, 64, 2, 4> CfgH256w8;   // 8 waves, 128x64 per wave, 2 waves / SIMD
typedef Cfg<half_t, 128, 128, 64, 2, 2> CfgH128;
// fp32: 8 waves of 64x32 on a 128x128 tile (two per SIMD hide each other's LDS and
// barrier waits; C2 on 256 tiles, one workgroup per CU: dX 75.6 -> 72.0 us, step +2.3%
// against 4 waves of 64x64)
typedef Cfg<float, 128, 128, 32, 2, 4> CfgF128;
typedef Cfg<float, 64, 64, 32, 2, 2> CfgF64;

template <class C, bool AK, bool BK_, bool VOK, class Epi>
static hipError_t run(const GemmLaunch &g, const typename Epi::Params &p, hipStream_t s) {
    typedef typename C::type T;
    GemmShape sh;
    sh.M = g.M;
    sh.N = g.N;
    sh.K = g.K;
    sh.lda = g.lda;
    sh.ldb = g.ldb;
    sh.tiles_m = (g.M + C::bm - 1) / C::bm;
    sh.tiles_n = (g.N + C::bn - 1) / C::bn;
    const uint32_t splits = g.splits ? g.splits : 1;
    const uint32_t kps_raw = (g.K + splits - 1) / splits;
    sh.k_per_split = ((kps_raw + C::bk - 1) / C::bk) * C::bk;
    dim3 grid(sh.tiles_m * sh.tiles_n, 1, splits);
    launch_timed(g, gemm_kernel<T, C::bm, C::bn, C::bk, C::wm, C::wn, AK, BK_, VOK, Epi>, grid, dim3(C::nt), s, sh,
                 reinterpret_cast<const T *>(g.A), reinterpret_cast<const T *>(g.B), p);
    return hipGetLastError();
}

static bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Decide whether both operands can be staged in 16-byte chunks.
static bool vec_ok(const GemmLaunch &g, int vec) {
    // contiguous extent of A: K if k-contig else M; of B: K if k-contig else N
    const uint32_t a_ext = g.a_kcontig ? g.K : g.M;
    const uint32_t b_ext = g.b_kcontig ? g.K : g.N;
    return (g.lda % vec) == 0 && (g.ldb % vec) == 0 && (a_ext % vec) == 0 && (b_ext % vec) == 0 &&
           aligned16(g.A) && aligned16(g.B);
}

template <class C, bool AK, bool BK_, class Epi>
static hipError_t dispatch_vec(const GemmLaunch &g, const typename Epi::Params &p, hipStream_t s) {
    constexpr int VEC = Mfma<typename C::type>::VEC;
    if (g.a_kcontig != AK || g.b_kcontig != BK_) return hipErrorInvalidValue;
    return vec_ok(g, VEC) ? run<C, AK, BK_, true, Epi>(g, p, s) : run<C, AK, BK_, false, Epi>(g, p, s);
}

// Only the (layout, epilogue) pairs the DenseBlock path uses are instantiated:
//   forward  : A k-contig, B n-contig
//   dX       : A k-contig, B k-contig
//   dW       : A m-contig, B n-contig
template <class C> static hipError_t dispatch_op(const GemmLaunch &g, hipStream_t s) {
    typedef typename C::type T;
    switch (g.op) {
    // forward on W or on a transposed copy of W
    case Op::Fwd:
        return g.b_kcontig ? dispatch_vec<C, true, true, EpiFwdK<T>>(g, g.fwd, s)
                           : dispatch_vec<C, true, false, EpiFwdK<T>>(g, g.fwd, s);
    case Op::InputGrad: return dispatch_vec<C, true, true, EpiStoreK>(g, g.st, s);
    // dW also runs on transposed copies of X and dP (both k-contiguous)
    case Op::DwPartial:
        return g.a_kcontig ? dispatch_vec<C, true, true, EpiStoreK>(g, g.st, s)
                           : dispatch_vec<C, false, false, EpiStoreK>(g, g.st, s);
    case Op::DwOpt:
        return g.a_kcontig ? dispatch_vec<C, true, true, EpiOptK<T>>(g, g.opt, s)
                           : dispatch_vec<C, false, false, EpiOptK<T>>(g, g.opt, s);
    case Op::HiddenErr: break;   // the 256x256 kernel only
    }
    return hipErrorInvalidValue;
}

// The 256x256 tile only runs the all-k-contiguous layout (large fp16
// problems are given transposed operands by the caller).
template <class C> static hipError_t dispatch_kk(const GemmLaunch &g, hipStream_t s) {
    typedef typename C::type T;
    switch (g.op) {
    case Op::Fwd: return dispatch_vec<C, true, true, EpiFwdK<T>>(g, g.fwd, s);
    case Op::InputGrad:
    case Op::DwPartial: return dispatch_vec<C, true, true, EpiStoreK>(g, g.st, s);
    case Op::DwOpt: return dispatch_vec<C, true, true, EpiOptK<T>>(g, g.opt, s);
    case Op::HiddenErr: break;   // the 256x256 kernel only
    }
    return hipErrorInvalidValue;
}

bool gemm_large_tile(uint32_t dtype, uint32_t M, uint32_t N) {
    return dtype == 1 && ((M + 255) / 256) * ((N + 255) / 256) >= 192;
}

// Output tiles of the general (non-256) configuration; drives split-K.
uint32_t gemm_tiles(uint32_t dtype, uint32_t M, uint32_t N) {
    if (dtype == 1) return ((M + 127) / 128) * ((N + 127) / 128);
    const uint32_t t128 = ((M + 127) / 128) * ((N + 127) / 128);
    if (t128 >= 192) return t128;
    return ((M + 63) / 64) * ((N + 63) / 64);
}

uint32_t gemm_bk(uint32_t dtype) { return dtype == 1 ? 64 : 32; }

// The direct-to-LDS kernel (gemm_dma.h).  SOKLYN_GEMM_DMA=0 leaves it out of the
// planner's choice (A/B comparisons).
bool gemm_dma_enabled() {
    static bool on = [] {
        const char *e = getenv("SOKLYN_GEMM_DMA");
        return !(e && atoi(e) == 0);
    }();
    return on;
}

uint32_t gemm_dma_tile_forced() {
    static uint32_t t = [] {
        const char *e = getenv("SOKLYN_GEMM_TILE");
        const int v = e ? atoi(e) : 0;
        return v == 128 || v == 256 ? (uint32_t)v : 0u;
    }();
    return t;
}

// Operand layouts the direct-to-LDS kernel is instantiated for: every op with
// both operands k-contiguous, the forward on W as stored (n-contiguous), and dW
// on X and dP as stored (m- and n-contiguous).
static bool dma_layout_ok(const GemmLaunch &g) {
    if (g.a_kcontig && g.b_kcontig) return true;
    if (g.op == Op::Fwd) return g.a_kcontig && !g.b_kcontig;
    if (g.op == Op::DwOpt || g.op == Op::DwPartial) return !g.a_kcontig && !g.b_kcontig;
    return false;
}

static uint32_t epi_ldc(const GemmLaunch &g) {
    switch (g.op) {
    case Op::Fwd: return g.fwd.ldc;
    case Op::InputGrad:
    case Op::DwPartial: return g.st.ldc;
    case Op::DwOpt: return g.opt.ldc;
    case Op::HiddenErr: return g.err.ldc;
    }
    return 0;
}

// The operands as given fit the 256x256 kernel: fp16, whole tiles, K a multiple
// of 128 (two k-tiles), 16-byte rows, 32-bit byte offsets within each operand.
bool gemm_dma_shape_ok(const GemmLaunch &g) {
    if (!gemm_dma_enabled() || g.dtype != 1 || !dma_layout_ok(g)) return false;
    if ((g.M % 256) || (g.N % 256) || (g.K % 128) || g.K == 0) return false;
    if (!vec_ok(g, 8)) return false;
    const uint64_t a_rows = g.a_kcontig ? g.M : g.K, b_rows = g.b_kcontig ? g.N : g.K;
    return a_rows * g.lda * 2 < (1ull << 32) && b_rows * g.ldb * 2 < (1ull << 32);
}

// The fused error epilogue's 4-column accesses need every per-element buffer
// 16-byte aligned (fp32) / 8-byte aligned (fp16 at a multiple of 4 elements).
static bool err_epi_aligned(const ErrEpi &e) {
    const void *p[] = {e.predrop, e.preact, e.mask, e.grad, e.d_prenorm, e.d_prenorm_h,
                       e.norm ? e.d_norm_w : nullptr, e.norm ? e.d_norm_b : nullptr,
                       e.norm == 1 ? e.prenorm : nullptr, e.norm >= 2 ? e.centered : nullptr,
                       e.norm ? e.nw : nullptr, e.norm == 3 ? e.norm_rstd : nullptr};
    for (const void *q : p)
        if (q && !aligned16(q)) return false;
    return true;
}

// The hidden error of an M x N output can be fused into the 256x256 kernel:
// whole tiles (no padded output), 4-aligned rows, aligned buffers.  Ragged
// outputs keep the GEMM + error kernel pair: an element-by-element form of the
// fused epilogue was measured 1.3x slower than that pair on config 5's shapes.
bool hidden_err_fusable(const ErrEpi &e, uint32_t M, uint32_t N) {
    return M % 256 == 0 && N % 256 == 0 && e.ldc % 4 == 0 && err_epi_aligned(e);
}

// ... or into the K-splitting kernel: whole 4-column groups, any number of rows.
bool hidden_err_wave_ok(const ErrEpi &e, uint32_t N) { return N % 4 == 0 && e.ldc % 4 == 0 && err_epi_aligned(e); }

// Whole output tiles with a 4-aligned leading dimension: the batched epilogue.
static bool dma_full_epilogue(const GemmLaunch &g) {
    const uint32_t mv = g.mv ? g.mv : g.M, nv = g.nv ? g.nv : g.N;
    if (g.op == Op::HiddenErr && !err_epi_aligned(g.err)) return false;
    return mv == g.M && nv == g.N && epi_ldc(g) % 4 == 0;
}

bool gemm_direct_ok(const GemmLaunch &g) {
    return gemm_large_tile(g.dtype, g.M, g.N) && gemm_dma_shape_ok(g) && dma_full_epilogue(g) &&
           (g.splits == 0 || g.splits == 1);
}

// 256x256: 4 waves (one per SIMD, 16x16x32 MFMAs on AGPR accumulators) for the
// epilogues DmaOneWave selects on whole tiles; otherwise 8 waves (two per SIMD: one
// issues MFMAs while the other waits on LDS; see gemm_dma.h) with
// v_mfma_f32_16x16x32_f16 when A is k-contiguous (C3 shapes: dX 2% faster back to
// back, 5% with a cold last-level cache; forward 2-3%) and 32x32x16 when both
// operands are transposed, whose 16x16 fragments at 8 waves overflow the register
// budget even with A single-buffered.  128x128: 4 waves of 64x64, two workgroups per
// CU, 16x16x32 for every layout.
template <class Epi, bool AK, bool BK_, int NW, int MI, int BT>
static hipError_t run_dma_t(const GemmLaunch &g, const typename Epi::Params &p, uint32_t splits, uint32_t kps,
                            hipStream_t s) {
    GemmShape sh{};
    sh.M = g.M;
    sh.N = g.N;
    sh.K = g.K;
    sh.lda = g.lda;
    sh.ldb = g.ldb;
    sh.k_per_split = kps;
    sh.tiles_m = (g.m_rows ? g.m_rows : g.M) / BT;
    sh.tiles_n = g.N / BT;
    sh.m_base = g.m_begin;
    sh.mv = g.mv ? g.mv : g.M;
    sh.nv = g.nv ? g.nv : g.N;
    const dim3 grid(sh.tiles_m * sh.tiles_n, splits);
    const half_t *A = reinterpret_cast<const half_t *>(g.A);
    const half_t *B = reinterpret_cast<const half_t *>(g.B);
    if (dma_full_epilogue(g))
        launch_timed(g, gemm_dma_kernel<Epi, AK, BK_, NW, false, MI, BT>, grid, dim3(64 * NW), s, sh, A, B, p);
    else if constexpr (EpiSums<Epi>::value || (NW == 4 && BT == 256))
        return hipErrorInvalidValue;   // whole tiles only (hidden_err_fusable; the one-wave-per-SIMD tile)
    else
        launch_timed(g, gemm_dma_kernel<Epi, AK, BK_, NW, true, MI, BT>, grid, dim3(64 * NW), s, sh, A, B, p);
    return hipGetLastError();
}

// Epilogues that run the 256x256 tile with one wave per SIMD (4 waves, 16x16x32 MFMAs
// on AGPR accumulators, a third fewer LDS fragment bytes per flop than 8 waves): the
// fp32 store (dX, split-K dW partials) and the fused optimiser.  Measured on the C3
// shapes against 8 waves on one box: main loop 4% faster per k for dX and dW; dX
// 213.1 -> 207.7 us, dW + Adam 281.3 -> 267.8 us.  The forward and the fused hidden
// error keep 8 waves: their store-heavy epilogues run slower with half the threads
// (forward 225.0 -> 241.3 us).
template <class Epi> struct DmaOneWave { static constexpr bool value = false; };
template <> struct DmaOneWave<EpiStoreK> { static constexpr bool value = true; };
template <> struct DmaOneWave<EpiOptK<half_t>> { static constexpr bool value = true; };

template <class Epi, bool AK, bool BK_>
static hipError_t run_dma(const GemmLaunch &g, const typename Epi::Params &p, uint32_t splits, uint32_t kps,
                          hipStream_t s) {
    if (g.tile == 128) return run_dma_t<Epi, AK, BK_, 4, 16, 128>(g, p, splits, kps, s);
    if constexpr (DmaOneWave<Epi>::value)
        if (dma_full_epilogue(g)) return run_dma_t<Epi, AK, BK_, 4, 16, 256>(g, p, splits, kps, s);
    return run_dma_t<Epi, AK, BK_, 8, AK ? 16 : 32, 256>(g, p, splits, kps, s);
}

// The 128x128 kernel on operands as stored: fp16 forward and input gradient, K whole
// 16-byte chunks (it is contiguous in A), rows and bases on 4-byte boundaries, byte offsets
// below 2 GiB with the tiles and k-tiles past the ends.
bool gemm_dma_rag_ok(const GemmLaunch &g) {
    if (!gemm_dma_enabled() || g.dtype != 1 || (g.op != Op::Fwd && g.op != Op::InputGrad) || !dma_layout_ok(g))
        return false;
    auto dword = [](const void *p, uint32_t ld) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0 && ld % 2 == 0; };
    const uint64_t a_rows = g.M + 256ull, b_rows = g.b_kcontig ? g.N + 256ull : g.K + 512ull;
    return g.M && g.N && g.K && g.K % 8 == 0 && dword(g.A, g.lda) && dword(g.B, g.ldb) &&
           a_rows * g.lda * 2 < (1ull << 31) && b_rows * g.ldb * 2 < (1ull << 31);
}

template <class Epi, bool B_KC> static hipError_t run_dma_rag(const GemmLaunch &g, const typename Epi::Params &p,
                                                             bool whole, hipStream_t s) {
    GemmShape sh{};
    sh.M = g.M;
    sh.N = g.N;
    sh.K = g.K;
    sh.lda = g.lda;
    sh.ldb = g.ldb;
    sh.k_per_split = (g.K + 127) / 128 * 128;
    sh.tiles_m = (g.M + 127) / 128;
    sh.tiles_n = (g.N + 127) / 128;
    sh.mv = g.M;
    sh.nv = g.N;
    sh.whole = whole;
    launch_timed(g, gemm_dma_kernel<Epi, true, B_KC, 4, true, 16, 128, true>, dim3(sh.tiles_m * sh.tiles_n), dim3(256), s,
                 sh, reinterpret_cast<const half_t *>(g.A), reinterpret_cast<const half_t *>(g.B), p);
    return hipGetLastError();
}

static hipError_t launch_dma_rag(const GemmLaunch &g, hipStream_t s) {
    if (!gemm_dma_rag_ok(g)) return hipErrorInvalidValue;
    if (g.op == Op::Fwd) {
        // 8-column, 16-byte stores of the caches
        const FwdEpi &e = g.fwd;
        const bool whole = e.ldc % 8 == 0 && aligned16(e.bias) && aligned16(e.z_out) &&
                           (!e.fuse_act || (aligned16(e.predrop) && aligned16(e.out) && (!e.use_dropout || aligned16(e.mask))));
        return g.b_kcontig ? hipErrorInvalidValue : run_dma_rag<EpiFwdK<half_t>, false>(g, e, whole, s);
    }
    return run_dma_rag<EpiStoreK, true>(g, g.st, g.st.ldc % 4 == 0 && aligned16(g.st.out), s);
}

hipError_t launch_gemm_dma(const GemmLaunch &g, hipStream_t s) {
    if (g.rag) return launch_dma_rag(g, s);
    if (!gemm_dma_shape_ok(g)) return hipErrorInvalidValue;
    // split-K: slices of k_per_split (a multiple of 128), the last one possibly shorter
    const uint32_t splits_req = g.splits ? g.splits : 1;
    const uint32_t kps = ((g.K / splits_req + 127) / 128) * 128;
    const uint32_t splits = (g.K + kps - 1) / kps;
    if (splits > 1 && g.op != Op::DwPartial) return hipErrorInvalidValue;
    if (g.m_rows || g.m_begin) {
        // a band of output rows: whole tiles inside M, not the column-sum epilogue
        const uint32_t t = g.tile == 128 ? 128u : 256u;
        if (g.op == Op::HiddenErr || g.m_begin % 256 || g.m_rows % t || g.m_rows == 0 ||
            (uint64_t)g.m_begin + g.m_rows > g.M)
            return hipErrorInvalidValue;
    }
    const bool kk = g.a_kcontig && g.b_kcontig;
    switch (g.op) {
    case Op::Fwd:
        return kk ? run_dma<EpiFwdK<half_t>, true, true>(g, g.fwd, splits, kps, s)
                  : run_dma<EpiFwdK<half_t>, true, false>(g, g.fwd, splits, kps, s);
    case Op::InputGrad: return run_dma<EpiStoreK, true, true>(g, g.st, splits, kps, s);
    case Op::DwPartial:
        return kk ? run_dma<EpiStoreK, true, true>(g, g.st, splits, kps, s)
                  : run_dma<EpiStoreK, false, false>(g, g.st, splits, kps, s);
    case Op::DwOpt:
        return kk ? run_dma<EpiOptK<half_t>, true, true>(g, g.opt, splits, kps, s)
                  : run_dma<EpiOptK<half_t>, false, false>(g, g.opt, splits, kps, s);
    case Op::HiddenErr:
        return kk ? run_dma<EpiErrK<half_t>, true, true>(g, g.err, splits, kps, s) : hipErrorInvalidValue;
    }
    return hipErrorInvalidValue;
}

// Split-K slices launch_gemm_dma makes of K for `splits` requested.
uint32_t gemm_dma_splits(uint32_t K, uint32_t splits) {
    const uint32_t kps = ((K / (splits ? splits : 1) + 127) / 128) * 128;
    return (K + kps - 1) / kps;
}

// ---- dW of at most 16 columns ---------------------------------------------------------
// A stream over X, whatever its size and pitch (64-bit offsets): 1024 workgroups of
// 256 columns of X and a batch slice keep the GPU's loads in flight, and their short sums are
// the more precise the longer the batch (f32 142860 x 1603 -> 10: 6.0e-7 against 64 bits, 1.07e-6 on the K-splitting
// kernel).  The planner's skinny_us says where it is taken, with the times of both.
constexpr uint32_t SKINNY_N = 16;

// dW partial sums, thread per W row: thread k of workgroup (x, y) walks the batch rows
// of slice y in order, acc[n] += X[b][k] * dP[b][n], with 64 rows of dP (fp32) at a
// time in LDS (16-byte broadcast reads) and the X loads of 16 rows issued before
// their FMAs; partials[y][k][0..15].
__global__ void __launch_bounds__(256) skinny_dw_kernel(GemmShape sh, const float *__restrict__ X,
                                                        const float *__restrict__ dp, float *__restrict__ partials,
                                                        uint32_t per) {
    __shared__ __attribute__((aligned(16))) float dps[64][SKINNY_N];
    const uint32_t K = sh.M, N = sh.N;          // output [K x N]; reduction over sh.K batch rows
    const uint32_t k = blockIdx.x * 256 + threadIdx.x;
    const uint32_t r0 = blockIdx.y * per;
    const uint32_t r1 = min(sh.K, r0 + per);
    float acc[SKINNY_N];
#pragma unroll
    for (int n = 0; n < (int)SKINNY_N; ++n) acc[n] = 0.0f;
    for (uint32_t rb = r0; rb < r1; rb += 64) {
        const uint32_t nrows = min(64u, r1 - rb);
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < 64 * SKINNY_N; i += 256) {
            const uint32_t r = i / SKINNY_N, n = i % SKINNY_N;
            dps[r][n] = (r < nrows && n < N) ? dp[(uint64_t)(rb + r) * sh.ldb + n] : 0.0f;
        }
        __syncthreads();
        if (k < K) {
            for (uint32_t r0b = 0; r0b < nrows; r0b += 16) {
                float xv[16];
#pragma unroll
                for (uint32_t u = 0; u < 16; ++u)
                    xv[u] = r0b + u < nrows ? X[(uint64_t)(rb + r0b + u) * sh.lda + k] : 0.0f;
#pragma unroll
                for (uint32_t u = 0; u < 16; ++u) {
                    if (r0b + u >= nrows) break;
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const floatx4 d = *reinterpret_cast<const floatx4 *>(&dps[r0b + u][4 * q]);
                        acc[4 * q + 0] = fmaf(xv[u], d[0], acc[4 * q + 0]);
                        acc[4 * q + 1] = fmaf(xv[u], d[1], acc[4 * q + 1]);
                        acc[4 * q + 2] = fmaf(xv[u], d[2], acc[4 * q + 2]);
                        acc[4 * q + 3] = fmaf(xv[u], d[3], acc[4 * q + 3]);
                    }
                }
            }
        }
    }
    if (k >= K) return;
    float *p = partials + ((uint64_t)blockIdx.y * K + k) * SKINNY_N;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<floatx4 *>(p + 4 * q) = floatx4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
}

// The same on MFMA (fp16; dP as its fp16 copy, the dW GEMMs' operand): thread t
// of workgroup (x, y) loads column k = 256 x + t of X for 32 batch rows at a time
// (coalesced 2-byte loads, all 32 issued before use) and writes them to LDS
// transposed (xt[t][0..31], one 64-byte run); the 32 x 16 block of dP goes to
// pt[n][0..31].  Wave w then runs v_mfma_f32_16x16x32_f16 on its 4 tiles of 16 W
// rows: src0 lane l = xt[16 q + l % 16][8 (l / 16) ..] (X^T), src1 lane l =
// pt[l % 16][8 (l / 16) ..] (dP); lane l ends with rows 4 (l / 16) .. + 3 of column
// l % 16 of the tile.  LDS rows of 40 halves (80 bytes) keep the 16-byte reads of
// 16 lanes in distinct banks.  partials[y][k][0..15] as in skinny_dw_kernel.
__global__ void __launch_bounds__(256) skinny_dw_mfma_kernel(GemmShape sh, const half_t *__restrict__ X,
                                                             const half_t *__restrict__ dp16,
                                                             float *__restrict__ partials, uint32_t per) {
    __shared__ __attribute__((aligned(16))) half_t xt[256][40];
    __shared__ __attribute__((aligned(16))) half_t pt[SKINNY_N][40];
    const uint32_t K = sh.M, N = sh.N;          // output [K x N]; reduction over sh.K batch rows
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t k0 = blockIdx.x * 256, k = k0 + tid;
    const uint32_t r0 = blockIdx.y * per;
    const uint32_t r1 = min(sh.K, r0 + per);
    floatx4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) acc[q] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t rb = r0; rb < r1; rb += 32) {
        const uint32_t nrows = min(32u, r1 - rb);
        half_t xv[32];
#pragma unroll
        for (uint32_t u = 0; u < 32; ++u)
            xv[u] = (u < nrows && k < K) ? X[(uint64_t)(rb + u) * sh.lda + k] : (half_t)0;
        half_t pv[2];
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t i = tid + 256 * h, u = i >> 4, n = i & 15u;   // 32 rows x 16 columns
            pv[h] = (u < nrows && n < N) ? dp16[(uint64_t)(rb + u) * sh.ldb + n] : (half_t)0;
        }
        __syncthreads();   // the previous block's fragments are read
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<halfx8 *>(&xt[tid][8 * q]) = *reinterpret_cast<const halfx8 *>(&xv[8 * q]);
#pragma unroll
        for (uint32_t h = 0; h < 2; ++h) {
            const uint32_t i = tid + 256 * h;
            pt[i & 15u][i >> 4] = pv[h];
        }
        __syncthreads();
        const halfx8 b = *reinterpret_cast<const halfx8 *>(&pt[lane & 15u][8 * (lane >> 4)]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const halfx8 a = *reinterpret_cast<const halfx8 *>(&xt[wave * 64 + 16 * q + (lane & 15u)][8 * (lane >> 4)]);
            acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc[q], 0, 0, 0);
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
#pragma unroll
        for (uint32_t r = 0; r < 4; ++r) {
            const uint32_t ko = k0 + wave * 64 + 16 * q + 4 * (lane >> 4) + r;
            if (ko < K) partials[((uint64_t)blockIdx.y * K + ko) * SKINNY_N + (lane & 15u)] = acc[q][r];
        }
    }
}

uint32_t skinny_dw_slices(uint32_t rows, uint32_t K) {
    const uint32_t col_blocks = (K + 255) / 256;
    uint32_t sl = (1024 + col_blocks - 1) / col_blocks;
    const uint32_t cap = (rows + 63) / 64;
    if (sl > cap) sl = cap;
    return sl < 1 ? 1 : sl;
}

hipError_t launch_skinny_dw(const GemmLaunch &g, float *partials, uint32_t slices, hipStream_t s) {
    if (g.N > SKINNY_N || !g.M || !g.K || !slices || g.a_kcontig || g.b_kcontig ||
        (reinterpret_cast<uintptr_t>(partials) & 15u))
        return hipErrorInvalidValue;
    GemmShape sh{};
    sh.M = g.M;          // W rows (inputs)
    sh.N = g.N;          // W cols (outputs)
    sh.K = g.K;          // batch rows
    sh.lda = g.lda;      // X row pitch
    sh.ldb = g.ldb;      // d_prenorm row pitch
    const uint32_t per = (g.K + slices - 1) / slices;
    const dim3 grid((g.M + 255) / 256, slices);
    if (g.dtype == 1)
        launch_timed(g, skinny_dw_mfma_kernel, grid, dim3(256), s, sh, reinterpret_cast<const half_t *>(g.A),
                     reinterpret_cast<const half_t *>(g.B), partials, per);
    else
        launch_timed(g, skinny_dw_kernel, grid, dim3(256), s, sh, reinterpret_cast<const float *>(g.A),
                     reinterpret_cast<const float *>(g.B), partials, per);
    return hipGetLastError();
}

hipError_t launch_gemm(const GemmLaunch &g, hipStream_t s) {
    if (g.M == 0 || g.N == 0) return hipSuccess;
    if (gemm_direct_ok(g)) return launch_gemm_dma(g, s);
    if (g.dtype == 1) {
        if (gemm_large_tile(g.dtype, g.M, g.N) && g.a_kcontig && g.b_kcontig) return dispatch_kk<CfgH256w8>(g, s);
        return dispatch_op<CfgH128>(g, s);
    }
    const uint32_t t128 = ((g.M + 127) / 128) * ((g.N + 127) / 128);
    return t128 >= 192 || g.tile == 128 ? dispatch_op<CfgF128>(g, s) : dispatch_op<CfgF64>(g, s);
}

}  // namespace skl
