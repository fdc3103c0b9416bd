// epilogue.h — what the GEMM kernels do with an output element: the forward (bias,
// activation, dropout, cache stores), the plain fp32 store, the optimiser step on W and
// the hidden-layer error.
#pragma once

#include <hip/hip_ext.h>

#include <type_traits>

#include "gemm.h"
#include "launch.h"
#include "vec_opt.h"

namespace skl {

// Launches a GEMM kernel; with g.time_start / g.time_stop set, the dispatch
// itself carries the timing events.
template <typename K, typename... Args>
static void launch_timed(const GemmLaunch &g, K kernel, dim3 grid, dim3 block, hipStream_t s, Args... args) {
    if (g.time_start || g.time_stop)
        hipExtLaunchKernelGGL(kernel, grid, block, 0, s, g.time_start, g.time_stop, 0, args...);
    else
        hipLaunchKernelGGL(kernel, grid, block, 0, s, args...);
}


template <typename T> __device__ __forceinline__ T ld_t(const void *p, uint64_t i) {
    return reinterpret_cast<const T *>(p)[i];
}
template <typename T> __device__ __forceinline__ void st_t(void *p, uint64_t i, T v) {
    reinterpret_cast<T *>(p)[i] = v;
}

// ---- forward: bias (+ act + dropout) ------------------------------------------
//
// Every epilogue has a whole-vector form in three parts, so a caller can batch
// the global loads of many 4-column groups before computing any of them:
//   column(e, n)        per-column operands of columns n..n+3 (loaded once)
//   load(e, idx, m, p)  per-element operands of row m, columns n..n+3
//   finish(e, idx, m, n, v, col, p)  compute from the fp32 accumulators v, store
// apply() handles one 4-column group, including ragged edges.
template <typename T> struct EpiFwdK {
    typedef FwdEpi Params;
    __device__ __forceinline__ static uint32_t ldc(const FwdEpi &e) { return e.ldc; }
    __device__ __forceinline__ static FwdEpi at_split(const FwdEpi &e, uint32_t) { return e; }
    struct Col { f32x4 bias; };
    struct Pre {};
    __device__ __forceinline__ static Col column(const FwdEpi &e, uint32_t n) {
        Col c;
        c.bias = e.bias ? load4<T>(e.bias, n) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        return c;
    }
    __device__ __forceinline__ static void load(const FwdEpi &, uint64_t, uint32_t, Pre &) {}
    __device__ __forceinline__ static void finish(const FwdEpi &e, uint64_t idx, uint32_t m, uint32_t n, floatx4 v,
                                                  const Col &col, const Pre &) {
        // 4 consecutive columns: one 8-byte (fp16) / 16-byte (fp32) access per tensor
        f32x4 z = v;
        if (e.bias) z = z + col.bias;
        store4_nt<T>(e.z_out, idx, z);
        if (!e.fuse_act) return;
        const f32x4 zt = round4<T>(z);
        f32x4 a;
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] = activation<T>(e.act, zt[j], e.leaky);
        store4_nt<T>(e.predrop, idx, a);
        if (e.use_dropout) {
            const float scale = 1.0f / (1.0f - e.p);
            f32x4 mk, o;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool keep = dropout_u(n + j, m, e.seed + m * 7u) >= e.p;
                mk[j] = keep ? scale : 0.0f;
                o[j] = keep ? a[j] * scale : 0.0f;
            }
            store4_nt<T>(e.mask, idx, mk);
            store4_nt<T>(e.out, idx, o);
        } else {
            store4_nt<T>(e.out, idx, a);
        }
    }
    // 8 consecutive columns (fp16 outputs: 16-byte stores)
    static constexpr int kVec = sizeof(T) == 2 ? 8 : 4;
    struct Col8 { f32x4 lo, hi; };
    __device__ __forceinline__ static Col8 column8(const FwdEpi &e, uint32_t n) {
        Col8 c;
        c.lo = e.bias ? load4<T>(e.bias, n) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        c.hi = e.bias ? load4<T>(e.bias, n + 4) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        return c;
    }
    __device__ __forceinline__ static void st8(void *p, uint64_t idx, f32x4 lo, f32x4 hi) {
        const half_t h[8] = {(half_t)lo[0], (half_t)lo[1], (half_t)lo[2], (half_t)lo[3],
                             (half_t)hi[0], (half_t)hi[1], (half_t)hi[2], (half_t)hi[3]};
        __builtin_nontemporal_store(*reinterpret_cast<const u32x4 *>(h),
                                    reinterpret_cast<u32x4 *>(reinterpret_cast<half_t *>(p) + idx));
    }
    __device__ __forceinline__ static void finish8(const FwdEpi &e, uint64_t idx, uint32_t m, uint32_t n, floatx4 v0,
                                                   floatx4 v1, const Col8 &col) {
        f32x4 z0 = v0, z1 = v1;
        if (e.bias) {
            z0 = z0 + col.lo;
            z1 = z1 + col.hi;
        }
        st8(e.z_out, idx, z0, z1);
        if (!e.fuse_act) return;
        const f32x4 t0 = round4<T>(z0), t1 = round4<T>(z1);
        f32x4 a0, a1;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a0[j] = activation<T>(e.act, t0[j], e.leaky);
            a1[j] = activation<T>(e.act, t1[j], e.leaky);
        }
        st8(e.predrop, idx, a0, a1);
        if (e.use_dropout) {
            const float scale = 1.0f / (1.0f - e.p);
            f32x4 m0, m1, o0, o1;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool k0 = dropout_u(n + j, m, e.seed + m * 7u) >= e.p;
                const bool k1 = dropout_u(n + 4 + j, m, e.seed + m * 7u) >= e.p;
                m0[j] = k0 ? scale : 0.0f;
                o0[j] = k0 ? a0[j] * scale : 0.0f;
                m1[j] = k1 ? scale : 0.0f;
                o1[j] = k1 ? a1[j] * scale : 0.0f;
            }
            st8(e.mask, idx, m0, m1);
            st8(e.out, idx, o0, o1);
        } else {
            st8(e.out, idx, a0, a1);
        }
    }
    // one element (ragged tiles): per-column operands loaded once per column
    struct Col1 { float bias; };
    __device__ __forceinline__ static Col1 column1(const FwdEpi &e, uint32_t n) {
        return Col1{e.bias ? to_f32(ld_t<T>(e.bias, n)) : 0.0f};
    }
    __device__ __forceinline__ static void apply1(const FwdEpi &e, uint32_t m, uint32_t n, float v, const Col1 &col,
                                                  uint32_t) {
        float z = v;
        if (e.bias) z = z + col.bias;   // f32 acc + f32(b), one rounding
        const T zt = from_f32<T>(z);
        const uint64_t idx = (uint64_t)m * e.ldc + n;
        st_t<T>(e.z_out, idx, zt);
        if (!e.fuse_act) return;
        const float a = activation<T>(e.act, to_f32(zt), e.leaky);
        st_t<T>(e.predrop, idx, from_f32<T>(a));
        if (e.use_dropout) {
            if (dropout_u(n, m, e.seed + m * 7u) >= e.p) {
                const float scale = 1.0f / (1.0f - e.p);
                st_t<T>(e.mask, idx, from_f32<T>(scale));
                st_t<T>(e.out, idx, from_f32<T>(a * scale));
            } else {
                st_t<T>(e.mask, idx, (T)0);
                st_t<T>(e.out, idx, (T)0);
            }
        } else {
            st_t<T>(e.out, idx, from_f32<T>(a));
        }
    }
    __device__ __forceinline__ static void apply(const FwdEpi &e, const GemmShape &sh, uint32_t m, uint32_t n,
                                                 floatx4 v, uint32_t) {
        if (m >= sh.M) return;
        if (n + 3 < sh.N && (e.ldc & 3u) == 0) {
            finish(e, (uint64_t)m * e.ldc + n, m, n, v, column(e, n), Pre{});
            return;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t c = n + j;
            if (c >= sh.N) break;
            float z = v[j];
            if (e.bias) z = z + to_f32(ld_t<T>(e.bias, c));   // f32 acc + f32(b), one rounding
            const T zt = from_f32<T>(z);
            const uint64_t idx = (uint64_t)m * e.ldc + c;
            st_t<T>(e.z_out, idx, zt);
            if (e.fuse_act) {
                const float a = activation<T>(e.act, to_f32(zt), e.leaky);
                st_t<T>(e.predrop, idx, from_f32<T>(a));
                if (e.use_dropout) {
                    if (dropout_u(c, m, e.seed + m * 7u) >= e.p) {
                        const float scale = 1.0f / (1.0f - e.p);
                        st_t<T>(e.mask, idx, from_f32<T>(scale));
                        st_t<T>(e.out, idx, from_f32<T>(a * scale));
                    } else {
                        st_t<T>(e.mask, idx, (T)0);
                        st_t<T>(e.out, idx, (T)0);
                    }
                } else {
                    st_t<T>(e.out, idx, from_f32<T>(a));
                }
            }
        }
    }
};

// ---- plain fp32 store (input gradient; split-K partials) -----------------------
struct EpiStoreK {
    static constexpr int kDmaSpacing = 1;   // front-loaded refill (measured fastest for dX)
    static constexpr int kReadsPerMfma = 1; // 32x32 schedule (the split-K dW partial)
    typedef StoreEpi Params;
    __device__ __forceinline__ static uint32_t ldc(const StoreEpi &e) { return e.ldc; }
    // the partial plane of split-K slice `split`
    __device__ __forceinline__ static StoreEpi at_split(const StoreEpi &e, uint32_t split) {
        StoreEpi r = e;
        r.out += (uint64_t)split * e.split_stride;
        return r;
    }
    struct Col {};
    struct Pre {};
    __device__ __forceinline__ static Col column(const StoreEpi &, uint32_t) { return Col{}; }
    __device__ __forceinline__ static void load(const StoreEpi &, uint64_t, uint32_t, Pre &) {}
    __device__ __forceinline__ static void finish(const StoreEpi &e, uint64_t idx, uint32_t, uint32_t, floatx4 v,
                                                  const Col &, const Pre &) {
        __builtin_nontemporal_store(v, reinterpret_cast<floatx4 *>(e.out + idx));
    }
    // one-wave-per-SIMD tiles: from the accumulator registers (half-line row segments,
    // so a plain store the L2 can join)
    static constexpr bool kDirect = true;
    static constexpr int kDirectBatch = 8;
    __device__ __forceinline__ static void direct(const StoreEpi &e, uint64_t idx, uint32_t, uint32_t, floatx4 v,
                                                  const Pre &) {
        *reinterpret_cast<floatx4 *>(e.out + idx) = v;
    }
    struct Col1 {};
    __device__ __forceinline__ static Col1 column1(const StoreEpi &, uint32_t) { return Col1{}; }
    __device__ __forceinline__ static void apply1(const StoreEpi &e, uint32_t m, uint32_t n, float v, const Col1 &,
                                                  uint32_t split) {
        e.out[(uint64_t)split * e.split_stride + (uint64_t)m * e.ldc + n] = v;
    }
    __device__ __forceinline__ static void apply(const StoreEpi &e, const GemmShape &sh, uint32_t m, uint32_t n,
                                                 floatx4 v, uint32_t split) {
        if (m >= sh.M) return;
        float *o = e.out + (uint64_t)split * e.split_stride + (uint64_t)m * e.ldc;
        if (n + 3 < sh.N && (e.ldc & 3u) == 0) {
            *reinterpret_cast<floatx4 *>(o + n) = v;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (n + j < sh.N) o[n + j] = v[j];
        }
    }
};

// ---- dW + optimiser on W (fused) -----------------------------------------------
template <typename T> struct EpiOptK {
    typedef OptEpi Params;
    typedef T elem;
    __device__ __forceinline__ static uint32_t ldc(const OptEpi &e) { return e.ldc; }
    __device__ __forceinline__ static OptEpi at_split(const OptEpi &e, uint32_t) { return e; }
    struct Col {};
    struct Pre { floatx4 p, dv, dm; };
    __device__ __forceinline__ static Col column(const OptEpi &, uint32_t) { return Col{}; }
    __device__ __forceinline__ static void load(const OptEpi &e, uint64_t idx, uint32_t, Pre &q) {
        q.p = *reinterpret_cast<const floatx4 *>(e.master + idx);
        q.dv = *reinterpret_cast<const floatx4 *>(e.dv + idx);
        q.dm = *reinterpret_cast<const floatx4 *>(e.dm + idx);
    }
    __device__ __forceinline__ static void finish(const OptEpi &e, uint64_t idx, uint32_t m, uint32_t n, floatx4 v,
                                                  const Col &, const Pre &q) {
        floatx4 p = q.p, dv = q.dv, dm = q.dm;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float pj = p[j], vj = dv[j], mj = dm[j];
            const float g = dw_checked<T>(e, m, n + j, v[j]);
            optimiser_step<sizeof(T) == 2>(pj, vj, mj, g * kLossScaleInv, e.inv_m, e.lr, e.clamp, e.opt,
                                           e.regularisation, e.regu_coeff, true);
            p[j] = pj; dv[j] = vj; dm[j] = mj;
        }
        *reinterpret_cast<floatx4 *>(e.master + idx) = p;
        *reinterpret_cast<floatx4 *>(e.dv + idx) = dv;
        *reinterpret_cast<floatx4 *>(e.dm + idx) = dm;
        if (e.param) {
            T t[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) t[j] = from_f32<T>(p[j]);
            if constexpr (sizeof(T) == 2) {
                *reinterpret_cast<uint64_t *>(reinterpret_cast<T *>(e.param) + idx) = __builtin_bit_cast(uint64_t, t);
            } else {
                *reinterpret_cast<floatx4 *>(reinterpret_cast<T *>(e.param) + idx) = __builtin_bit_cast(floatx4, t);
            }
        }
    }
    struct Col1 {};
    __device__ __forceinline__ static Col1 column1(const OptEpi &, uint32_t) { return Col1{}; }
    __device__ __forceinline__ static void apply1(const OptEpi &e, uint32_t m, uint32_t n, float v, const Col1 &,
                                                  uint32_t) {
        const uint64_t idx = (uint64_t)m * e.ldc + n;
        float pj = e.master[idx], vj = e.dv[idx], mj = e.dm[idx];
        const float g = dw_checked<T>(e, m, n, v);
        optimiser_step<sizeof(T) == 2>(pj, vj, mj, g * kLossScaleInv, e.inv_m, e.lr, e.clamp, e.opt,
                                       e.regularisation, e.regu_coeff, true);
        e.master[idx] = pj;
        e.dv[idx] = vj;
        e.dm[idx] = mj;
        if (e.param) st_t<T>(e.param, idx, from_f32<T>(pj));
    }
    __device__ __forceinline__ static void apply(const OptEpi &e, const GemmShape &sh, uint32_t m, uint32_t n,
                                                 floatx4 v, uint32_t) {
        if (m >= sh.M) return;
        const uint64_t base = (uint64_t)m * e.ldc;
        if (n + 3 < sh.N && (e.ldc & 3u) == 0) {
            Pre q;
            load(e, base + n, m, q);
            finish(e, base + n, m, n, v, Col{}, q);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c = n + j;
                if (c >= sh.N) break;
                const uint64_t idx = base + c;
                float pj = e.master[idx], vj = e.dv[idx], mj = e.dm[idx];
                const float g = dw_checked<T>(e, m, c, v[j]);
                optimiser_step<sizeof(T) == 2>(pj, vj, mj, g * kLossScaleInv, e.inv_m, e.lr, e.clamp, e.opt,
                                               e.regularisation, e.regu_coeff, true);
                e.master[idx] = pj;
                e.dv[idx] = vj;
                e.dm[idx] = mj;
                if (e.param) st_t<T>(e.param, idx, from_f32<T>(pj));
            }
        }
    }
};

// ---- hidden-layer error from the dX sum (fused) -----------------------------------
// compute_hidden_layer_error_kernel's epilogue (backward.cu:79-100) on the sum in
// the accumulators: e = mask * act'(s, predrop, preact); grad = e; the element-
// local norm gradient (util.cu:175-215, loss scale 1) into d_prenorm, its fp16
// copy and dNorm; and per-thread running column sums of d_prenorm / dNorm_w /
// dNorm_b, which flush() reduces over the 8 waves in a fixed order into the
// tile's row of partials (the inputs of the bias / norm-parameter update).
template <typename T> struct EpiErrK {
    typedef ErrEpi Params;
    static constexpr bool kColSums = true;
    __device__ __forceinline__ static uint32_t ldc(const ErrEpi &e) { return e.ldc; }
    __device__ __forceinline__ static ErrEpi at_split(const ErrEpi &e, uint32_t) { return e; }
    // per-column operands of 4 columns: the norm weight, and BatchNorm's per-column rstd
    struct Col { f32x4 nw, rstd; };
    // per-element operands of one row's 4 columns, as loaded (T)
    typedef typename std::conditional<sizeof(T) == 2, f16x4, f32x4>::type V4;
    struct Pre { V4 pd, pa, mk, pn; float rstd; };
    // running sums of the thread's 4 columns
    struct Acc { f32x4 dp, nw, nb; };
    __device__ __forceinline__ static Col column(const ErrEpi &e, uint32_t n) {
        Col c;
        c.nw = e.norm ? load4<float>(e.nw, n) : f32x4{0, 0, 0, 0};
        c.rstd = e.norm == 3 ? load4<T>(e.norm_rstd, n) : f32x4{0, 0, 0, 0};
        return c;
    }
    // nontemporal: the forward caches are read once here (C4's fused hidden error
    // 0.268 -> 0.262 ms against plain loads)
    __device__ __forceinline__ static V4 ld4(const void *p, uint64_t idx) {
        return __builtin_nontemporal_load(reinterpret_cast<const V4 *>(reinterpret_cast<const T *>(p) + idx));
    }
    __device__ __forceinline__ static void load(const ErrEpi &e, uint64_t idx, uint32_t m, Pre &q) {
        q.pd = ld4(e.predrop, idx);
        q.pa = ld4(e.preact, idx);
        q.mk = ld4(e.mask, idx);
        q.pn = e.norm ? ld4(e.norm == 1 ? e.prenorm : e.centered, idx) : V4{0, 0, 0, 0};
        q.rstd = (e.norm == 1 || e.norm == 2) ? to_f32(reinterpret_cast<const T *>(e.norm_rstd)[m]) : 0.0f;
    }
    __device__ __forceinline__ static void finish(const ErrEpi &e, uint64_t idx, uint32_t, uint32_t, floatx4 v,
                                                  const Col &col, const Pre &q, Acc &acc) {
        f32x4 g, dp, dnw = {0, 0, 0, 0}, dnb = {0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            g[j] = (float)q.mk[j] * activation_derivative<T>(e.act, v[j], (float)q.pd[j], (float)q.pa[j], e.leaky);
            dp[j] = g[j];
            if (e.norm) {
                const float p = (float)q.pn[j];
                const NormGrad ng = norm_grad(e.norm, g[j], p, p, e.norm == 3 ? col.rstd[j] : q.rstd, col.nw[j],
                                              e.inv_n, e.inv_m);
                dp[j] = ng.d_prenorm;
                dnw[j] = ng.dnw;
                dnb[j] = ng.dnb;
            }
        }
        __builtin_nontemporal_store(g, reinterpret_cast<f32x4 *>(e.grad + idx));
        *reinterpret_cast<f32x4 *>(e.d_prenorm + idx) = dp;
        if constexpr (sizeof(T) == 2)
            *reinterpret_cast<f16x4 *>(e.d_prenorm_h + idx) = f16x4{(half_t)dp[0], (half_t)dp[1], (half_t)dp[2],
                                                                    (half_t)dp[3]};
        if (e.norm) {
            __builtin_nontemporal_store(dnw, reinterpret_cast<f32x4 *>(e.d_norm_w + idx));
            __builtin_nontemporal_store(dnb, reinterpret_cast<f32x4 *>(e.d_norm_b + idx));
        }
        acc.dp += dp;
        acc.nw += dnw;
        acc.nb += dnb;
    }
    struct Col1 {};   // no element-by-element form: whole 4-column groups only
    // The tile's column sums from SLOTS threads per 4-column group (slot, group), added in slot
    // order: writes the columns < ncols of partials[tm][k].  Every thread of the NT calls it.
    template <int SLOTS, int BN, int NT>
    __device__ __forceinline__ static void flush_slots(const ErrEpi &e, const Acc &acc, float *lds, uint32_t tid,
                                                       uint32_t slot, uint32_t group, uint32_t tm, uint32_t n0) {
        if (slot < SLOTS) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c = 4u * group + j;
                lds[(slot * 3 + 0) * BN + c] = acc.dp[j];
                lds[(slot * 3 + 1) * BN + c] = acc.nw[j];
                lds[(slot * 3 + 2) * BN + c] = acc.nb[j];
            }
        }
        __syncthreads();
        for (uint32_t t = tid; t < 3 * BN; t += NT) {
            const uint32_t k = t / BN, c = t % BN;
            if ((k > 0 && !e.norm) || n0 + c >= e.ncols) continue;
            float s = 0.0f;
#pragma unroll
            for (uint32_t w = 0; w < SLOTS; ++w) s += lds[(w * 3 + k) * BN + c];
            e.partials[((uint64_t)tm * 3 + k) * e.ncols + n0 + c] = s;
        }
    }
    // The tile's column sums: each of the NW waves leaves its 3 x 256 running sums
    // in LDS (column 4 lane + j of the tile), then the block adds the waves in
    // order 0..NW-1 and writes the columns < ncols of partials[tm][k].  lds:
    // NW x 3 x 256 floats; the caller has made sure no wave still reads it.
    template <int NW, int BN>
    __device__ __forceinline__ static void flush(const ErrEpi &e, const Acc &acc, float *lds, uint32_t tid,
                                                 uint32_t tm, uint32_t n0) {
        // thread (wave, lane) holds the sums of columns 4 (lane % CPL) .. + 3 over
        // its rows; slot wave RPS + lane / CPL of the NW RPS partials per column
        constexpr uint32_t CPL = BN / 4, RPS = 64 / CPL, SLOTS = NW * RPS;
        const uint32_t lane = tid & 63u, wave = tid >> 6;
        flush_slots<SLOTS, BN, 64 * NW>(e, acc, lds, tid, wave * RPS + lane / CPL, lane % CPL, tm, n0);
    }
};

}  // namespace skl
