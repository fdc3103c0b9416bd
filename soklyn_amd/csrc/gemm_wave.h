// gemm_wave.h — GEMM whose waves split K among themselves, for outputs whose 128x128 or
// 256x256 tiles would leave most of the GPU idle (gfx950).
//
// A workgroup owns one (16 MB) x (16 NB) output tile and each of its W waves computes the
// whole tile over its own k-tiles (w, w + W, ...; 128 bytes of k each): it fills a private
// ring of S LDS stages by direct-to-LDS loads, waits for its own loads only, reads the
// fragments into registers, refills the stage and runs the MFMAs (16x16x32 f16, 16x16x4
// f32).  No barrier until the W partial tiles are added in LDS, in wave order, in front of
// the epilogue.  What bounds it: for a few hundred small tiles the latency of the first
// loads (all W S stages of a workgroup are in flight at once: 64-128 KB per CU), then the
// L2 -> LDS rate of a CU (a tile moves (MB + NB) 2 KB per k-tile); in fp32 the MFMAs.
//
// Operands as stored, k-contiguous or m/n-contiguous, rows and base on a 4-byte boundary
// (direct-to-LDS loads move dwords), or, for fp16 with odd row lengths, REG: the same
// tiles through registers by 16-byte loads at 2-byte alignment.  Edges need no padded
// copies: dwords past the operand's end read as zero (the buffer resource's range check),
// columns past a row's end only reach output columns that are not stored, and k past K is
// zeroed on the k-contiguous side (whole 16-byte chunks by an out-of-range offset, the
// last partial chunk by masking its fragments); the other side's rows past K are out of
// range already.
#pragma once

#include <type_traits>

#include "gemm.h"
#include "gemm_dma.h"
#include "vec_opt.h"

namespace skl {

// Byte offset no operand tile reaches (the host checks that spans stay below it).
constexpr uint32_t kWaveOob = 0x80000000u;

// One operand tile of a wave: ROWS rows (m or n) x 128 bytes of k.
// k-contiguous: LDS row = 128 bytes, 16-byte chunk c of row r at slot c ^ ((r >> 1) & 7).
template <typename T, int ROWS> struct WaveOpK {
    static constexpr int NF = ROWS / 16, IPO = ROWS / 8;
    static constexpr uint32_t CE = 16 / sizeof(T);
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t voff, kc, chunks, step, lds;
    uint32_t frag, g;
    __device__ __forceinline__ void init(const T *p, uint32_t ld, uint32_t rows, uint32_t K, uint32_t r0,
                                         uint32_t lane, uint32_t lds_op) {
        // from the tile's first row to its last (rounded to the dword of the last element)
        const uint32_t n = min(rows - r0, (uint32_t)ROWS);
        const uint32_t bytes = (((n - 1u) * ld + K) * (uint32_t)sizeof(T) + 3u) & ~3u;
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(p) + (uint64_t)r0 * ld, (short)0, (int)bytes,
                                                 0x00020000);
        // instruction t fills rows 8 t .. + 7: row 8 t + lane / 8, whose swizzle term is
        // (lane / 16) ^ 4 (t & 1)
        kc = (lane & 7u) ^ (lane >> 4);
        voff = (lane >> 3) * ld * (uint32_t)sizeof(T);
        chunks = (K + CE - 1) / CE;
        step = 8u * ld * (uint32_t)sizeof(T);
        lds = lds_op;
        g = (lane >> 4) ^ ((lane & 15u) >> 1);
        frag = lds_op + (lane & 15u) * 128u;
    }
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t stage) const {
#pragma unroll
        for (int t = 0; t < IPO; ++t) {
            const uint32_t c = kt * 8u + (kc ^ (4u * (t & 1)));
            const uint32_t off = c < chunks ? voff + t * step + c * 16u : kWaveOob;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rsrc, reinterpret_cast<__attribute__((address_space(3))) void *>(lds + stage + t * 1024u), 16, (int)off,
                0, 0, 0);
        }
    }
    // LDS address of fragment 0 of k-step ks (4 chunks); fragment i is 2048 bytes further
    __device__ __forceinline__ uint32_t at(uint32_t stage, int ks) const { return frag + stage + ((4u * ks) ^ g) * 16u; }
};

// m- or n-contiguous fp16: 64 k-rows of P bytes, chunk c of k-row r at slot c ^ swz(r); a
// fragment is two ds_read_b64_tr_b16 (16 lanes read 4 k-rows x 32 bytes, which the
// swizzle spreads over distinct banks).
template <int COLS> struct WaveOpNH {
    static constexpr int NF = COLS / 16;
    static constexpr uint32_t P = 2u * COLS, LPR = P / 16u, RPI = 64u / LPR;
    static constexpr int IPO = 64 / RPI;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t voff, step, kstep, lds, rel;
    __device__ __forceinline__ static uint32_t swz(uint32_t r) {
        return COLS == 64 ? 2u * (r & 3u) : COLS == 32 ? (r & 2u) : 0u;
    }
    __device__ __forceinline__ void init(const half_t *p, uint32_t ld, uint32_t cols, uint32_t K, uint32_t c0,
                                         uint32_t lane, uint32_t lds_op) {
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(p), (short)0,
                                                 (int)((((K - 1u) * ld + cols) * 2u + 3u) & ~3u), 0x00020000);
        const uint32_t r = lane / LPR;
        voff = r * ld * 2u + c0 * 2u + ((lane % LPR) ^ swz(r)) * 16u;
        step = RPI * ld * 2u;
        kstep = 64u * ld * 2u;
        lds = lds_op;
        const uint32_t s = lane & 15u, row = 8u * (lane >> 4) + (s >> 2);
        rel = row * P + ((((s & 3u) >> 1) ^ swz(row)) * 16u) + (s & 1u) * 8u;
    }
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t stage) const {
#pragma unroll
        for (int t = 0; t < IPO; ++t)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rsrc, reinterpret_cast<__attribute__((address_space(3))) void *>(lds + stage + t * 1024u), 16,
                (int)(voff + kt * kstep + t * step), 0, 0, 0);
    }
    // fragment i of the first k-step
    __device__ __forceinline__ uint32_t at(uint32_t stage, int i) const { return (rel ^ (32u * i)) + lds + stage; }
};

// m- or n-contiguous fp32: 32 k-rows of P bytes; k-row r sits at position
// 16 (r / 16) + 4 (r % 4) + (r % 16) / 4, so the four k-rows a ds_read_b32 takes (one per
// 16 lanes) are neighbours, and chunk c of position q at slot c ^ swz(q).
template <int COLS> struct WaveOpNF {
    static constexpr int NF = COLS / 16;
    static constexpr uint32_t P = 4u * COLS, LPR = P / 16u, RPI = 64u / LPR;
    static constexpr int IPO = 32 / RPI;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t voff, row, kstep, lds, rel;
    __device__ __forceinline__ static uint32_t swz(uint32_t q) {
        return COLS == 64 ? 4u * (q & 3u) : COLS == 32 ? 2u * (q & 2u) : 0u;
    }
    __device__ __forceinline__ void init(const float *p, uint32_t ld, uint32_t cols, uint32_t K, uint32_t c0,
                                         uint32_t lane, uint32_t lds_op) {
        rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p), (short)0,
                                                 (int)(((K - 1u) * ld + cols) * 4u), 0x00020000);
        // instruction t fills positions RPI t + q, q = lane / LPR
        const uint32_t q = lane / LPR;
        row = ld * 4u;
        voff = (4u * (q & 3u) + (q >> 2)) * row + c0 * 4u + ((lane % LPR) ^ swz(q)) * 16u;
        kstep = 32u * row;
        lds = lds_op;
        const uint32_t g = lane >> 4, c = lane & 15u;
        rel = g * P + (((c >> 2) ^ swz(g)) * 16u) + (c & 3u) * 4u;
    }
    __device__ __forceinline__ void issue(uint32_t kt, uint32_t stage) const {
#pragma unroll
        for (int t = 0; t < IPO; ++t) {
            const uint32_t q = RPI * t;   // position of the instruction's first row
            const uint32_t r = 16u * (q / 16u) + (q % 16u) / 4u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rsrc, reinterpret_cast<__attribute__((address_space(3))) void *>(lds + stage + t * 1024u), 16,
                (int)(voff + kt * kstep + r * row), 0, 0, 0);
        }
    }
    // fragment i of the first k-step (16 k): the first of the lane's k 4 (lane / 16) .. + 3
    __device__ __forceinline__ uint32_t at(uint32_t stage, int i) const { return (rel ^ (64u * i)) + lds + stage; }
};

// The same LDS tiles filled through registers, for fp16 rows at any 2-byte alignment: load
// takes a k-tile into registers (16 bytes per lane and instruction), put writes it to LDS.
// A chunk that would pass the operand's last element is read element by element.
__device__ __forceinline__ u32x4 wave_load16(const half_t *__restrict__ p, uint32_t e, uint32_t total) {
    u32x4 v = {0, 0, 0, 0};
    if (e + 8u <= total) {
        __builtin_memcpy(&v, p + e, 16);
    } else {
        half_t h[8];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) h[i] = e + i < total ? p[e + i] : (half_t)0;
        v = __builtin_bit_cast(u32x4, h);
    }
    return v;
}
__device__ __forceinline__ void wave_put16(uint32_t lds, u32x4 v) {
    *reinterpret_cast<__attribute__((address_space(3))) u32x4 *>(lds) = v;
}
template <int ROWS> struct WaveRegK : WaveOpK<half_t, ROWS> {
    typedef WaveOpK<half_t, ROWS> B;
    const half_t *p;
    uint32_t base, ldr, left, total;
    __device__ __forceinline__ void init(const half_t *p_, uint32_t ld, uint32_t rows, uint32_t K, uint32_t r0,
                                         uint32_t lane, uint32_t lds_op) {
        B::init(p_, ld, rows, K, r0, lane, lds_op);
        p = p_ + (uint64_t)r0 * ld;
        const uint32_t row = lane >> 3, n = min(rows - r0, (uint32_t)ROWS);
        base = row * ld;
        ldr = 8u * ld;
        left = row < n ? (n - row + 7u) / 8u : 0u;   // instructions whose row exists
        total = (n - 1u) * ld + K;
    }
    __device__ __forceinline__ void load(uint32_t kt, u32x4 (&r)[B::IPO]) const {
#pragma unroll
        for (int t = 0; t < B::IPO; ++t) {
            const uint32_t c = kt * 8u + (B::kc ^ (4u * (t & 1)));
            r[t] = (uint32_t)t < left && c < B::chunks ? wave_load16(p, base + t * ldr + c * 8u, total)
                                                       : u32x4{0, 0, 0, 0};
        }
    }
    __device__ __forceinline__ void put(const u32x4 (&r)[B::IPO], uint32_t lane) const {
#pragma unroll
        for (int t = 0; t < B::IPO; ++t) wave_put16(B::lds + t * 1024u + lane * 16u, r[t]);
    }
};
template <int COLS> struct WaveRegN : WaveOpNH<COLS> {
    typedef WaveOpNH<COLS> B;
    const half_t *p;
    uint32_t base, ldr, ktr, row, kmax, total;
    bool in;
    __device__ __forceinline__ void init(const half_t *p_, uint32_t ld, uint32_t cols, uint32_t K, uint32_t c0,
                                         uint32_t lane, uint32_t lds_op) {
        B::init(p_, ld, cols, K, c0, lane, lds_op);
        p = p_;
        row = lane / B::LPR;
        const uint32_t col = c0 + ((lane % B::LPR) ^ B::swz(row)) * 8u;
        in = col < cols;
        base = row * ld + col;
        ldr = B::RPI * ld;
        ktr = 64u * ld;
        kmax = K;
        total = (K - 1u) * ld + cols;
    }
    __device__ __forceinline__ void load(uint32_t kt, u32x4 (&r)[B::IPO]) const {
#pragma unroll
        for (int t = 0; t < B::IPO; ++t)
            r[t] = in && kt * 64u + row + B::RPI * t < kmax ? wave_load16(p, base + kt * ktr + t * ldr, total)
                                                            : u32x4{0, 0, 0, 0};
    }
    __device__ __forceinline__ void put(const u32x4 (&r)[B::IPO], uint32_t lane) const {
#pragma unroll
        for (int t = 0; t < B::IPO; ++t) wave_put16(B::lds + t * 1024u + lane * 16u, r[t]);
    }
};

template <typename T, bool KC, int ROWS, bool REG> struct WaveOpSel { typedef WaveOpK<T, ROWS> type; };
template <int ROWS> struct WaveOpSel<half_t, false, ROWS, false> { typedef WaveOpNH<ROWS> type; };
template <int ROWS> struct WaveOpSel<float, false, ROWS, false> { typedef WaveOpNF<ROWS> type; };
template <int ROWS> struct WaveOpSel<half_t, true, ROWS, true> { typedef WaveRegK<ROWS> type; };
template <int ROWS> struct WaveOpSel<half_t, false, ROWS, true> { typedef WaveRegN<ROWS> type; };

// The fragments of one operand for the two k-steps of a k-tile: LDS reads and the wait for
// them in one asm statement (the compiler would wait for every direct-to-LDS load in
// flight before an LDS read of its own).
template <typename T, bool KC, int NF> struct WaveFrags;
template <typename T, int NF> struct WaveFrags<T, true, NF> {
    static_assert(NF == 1 || NF == 2 || NF == 4, "fragments of a tile");
    u32x4 v[2][NF];
    template <class Op> __device__ __forceinline__ void read(const Op &op, uint32_t stage) {
        const uint32_t a0 = op.at(stage, 0), a1 = op.at(stage, 1);
        if constexpr (NF == 1)
            asm volatile(
            "ds_read_b128 %0, %2\n\t"
            "ds_read_b128 %1, %3\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0]), "=&v"(v[1][0])
            : "v"(a0), "v"(a1) : "memory");
        else if constexpr (NF == 2)
            asm volatile(
            "ds_read_b128 %0, %4\n\t"
            "ds_read_b128 %1, %4 offset:2048\n\t"
            "ds_read_b128 %2, %5\n\t"
            "ds_read_b128 %3, %5 offset:2048\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[1][0]), "=&v"(v[1][1])
            : "v"(a0), "v"(a1) : "memory");
        else if constexpr (NF == 4)
            asm volatile(
            "ds_read_b128 %0, %8\n\t"
            "ds_read_b128 %1, %8 offset:2048\n\t"
            "ds_read_b128 %2, %8 offset:4096\n\t"
            "ds_read_b128 %3, %8 offset:6144\n\t"
            "ds_read_b128 %4, %9\n\t"
            "ds_read_b128 %5, %9 offset:2048\n\t"
            "ds_read_b128 %6, %9 offset:4096\n\t"
            "ds_read_b128 %7, %9 offset:6144\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0]), "=&v"(v[0][1]), "=&v"(v[0][2]), "=&v"(v[0][3]), "=&v"(v[1][0]), "=&v"(v[1][1]),
              "=&v"(v[1][2]), "=&v"(v[1][3])
            : "v"(a0), "v"(a1) : "memory");
    }
    __device__ __forceinline__ u32x4 get(int ks, int i) const { return v[ks][i]; }
    // zero the elements of k-tile kt at k >= K
    __device__ __forceinline__ void cut(uint32_t kt, uint32_t K, uint32_t lane) {
        constexpr int CE = 16 / sizeof(T), PD = 4 / sizeof(T);   // elements per chunk, per dword
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int n = (int)K - (int)((kt * 8u + 4u * ks + (lane >> 4)) * CE);   // valid elements (may be < 0)
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const uint32_t m = n >= (d + 1) * PD ? ~0u : (PD == 2 && n == d * PD + 1) ? 0xffffu : 0u;
#pragma unroll
                for (int i = 0; i < NF; ++i) v[ks][i][d] &= m;
            }
        }
    }
};
template <int NF> struct WaveFrags<half_t, false, NF> {
    static_assert(NF == 1 || NF == 2 || NF == 4, "fragments of a tile");
    u32x2 v[2][NF][2];
    template <class Op> __device__ __forceinline__ void read(const Op &op, uint32_t stage) {
        uint32_t a[NF];
#pragma unroll
        for (int i = 0; i < NF; ++i) a[i] = op.at(stage, i);
        // k 0..3 of the lane's 8, k 4..7 four k-rows (4 P bytes) on; the second k-step 32 P on
        if constexpr (NF == 1)
            asm volatile(
            "ds_read_b64_tr_b16 %0, %4\n\t"
            "ds_read_b64_tr_b16 %1, %4 offset:128\n\t"
            "ds_read_b64_tr_b16 %2, %4 offset:1024\n\t"
            "ds_read_b64_tr_b16 %3, %4 offset:1152\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[1][0][0]), "=&v"(v[1][0][1])
            : "v"(a[0]) : "memory");
        else if constexpr (NF == 2)
            asm volatile(
            "ds_read_b64_tr_b16 %0, %8\n\t"
            "ds_read_b64_tr_b16 %1, %8 offset:256\n\t"
            "ds_read_b64_tr_b16 %2, %9\n\t"
            "ds_read_b64_tr_b16 %3, %9 offset:256\n\t"
            "ds_read_b64_tr_b16 %4, %8 offset:2048\n\t"
            "ds_read_b64_tr_b16 %5, %8 offset:2304\n\t"
            "ds_read_b64_tr_b16 %6, %9 offset:2048\n\t"
            "ds_read_b64_tr_b16 %7, %9 offset:2304\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[0][1][0]), "=&v"(v[0][1][1]), "=&v"(v[1][0][0]),
              "=&v"(v[1][0][1]), "=&v"(v[1][1][0]), "=&v"(v[1][1][1])
            : "v"(a[0]), "v"(a[1]) : "memory");
        else if constexpr (NF == 4)
            asm volatile(
            "ds_read_b64_tr_b16 %0, %16\n\t"
            "ds_read_b64_tr_b16 %1, %16 offset:512\n\t"
            "ds_read_b64_tr_b16 %2, %17\n\t"
            "ds_read_b64_tr_b16 %3, %17 offset:512\n\t"
            "ds_read_b64_tr_b16 %4, %18\n\t"
            "ds_read_b64_tr_b16 %5, %18 offset:512\n\t"
            "ds_read_b64_tr_b16 %6, %19\n\t"
            "ds_read_b64_tr_b16 %7, %19 offset:512\n\t"
            "ds_read_b64_tr_b16 %8, %16 offset:4096\n\t"
            "ds_read_b64_tr_b16 %9, %16 offset:4608\n\t"
            "ds_read_b64_tr_b16 %10, %17 offset:4096\n\t"
            "ds_read_b64_tr_b16 %11, %17 offset:4608\n\t"
            "ds_read_b64_tr_b16 %12, %18 offset:4096\n\t"
            "ds_read_b64_tr_b16 %13, %18 offset:4608\n\t"
            "ds_read_b64_tr_b16 %14, %19 offset:4096\n\t"
            "ds_read_b64_tr_b16 %15, %19 offset:4608\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[0][1][0]), "=&v"(v[0][1][1]), "=&v"(v[0][2][0]),
              "=&v"(v[0][2][1]), "=&v"(v[0][3][0]), "=&v"(v[0][3][1]), "=&v"(v[1][0][0]), "=&v"(v[1][0][1]),
              "=&v"(v[1][1][0]), "=&v"(v[1][1][1]), "=&v"(v[1][2][0]), "=&v"(v[1][2][1]), "=&v"(v[1][3][0]),
              "=&v"(v[1][3][1])
            : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]) : "memory");
    }
    __device__ __forceinline__ u32x4 get(int ks, int i) const {
        return u32x4{v[ks][i][0].x, v[ks][i][0].y, v[ks][i][1].x, v[ks][i][1].y};
    }
};
template <int NF> struct WaveFrags<float, false, NF> {
    static_assert(NF == 1 || NF == 2 || NF == 4, "fragments of a tile");
    u32x2 v[2][NF][2];
    template <class Op> __device__ __forceinline__ void read(const Op &op, uint32_t stage) {
        uint32_t a[NF];
#pragma unroll
        for (int i = 0; i < NF; ++i) a[i] = op.at(stage, i);
        // the lane's 4 k are 4 P bytes apart (offsets in units of 256 bytes); the second k-step 16 P on
        if constexpr (NF == 1)
            asm volatile(
            "ds_read2st64_b32 %0, %4 offset0:0 offset1:1\n\t"
            "ds_read2st64_b32 %1, %4 offset0:2 offset1:3\n\t"
            "ds_read2st64_b32 %2, %4 offset0:4 offset1:5\n\t"
            "ds_read2st64_b32 %3, %4 offset0:6 offset1:7\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[1][0][0]), "=&v"(v[1][0][1])
            : "v"(a[0]) : "memory");
        else if constexpr (NF == 2)
            asm volatile(
            "ds_read2st64_b32 %0, %8 offset0:0 offset1:2\n\t"
            "ds_read2st64_b32 %1, %8 offset0:4 offset1:6\n\t"
            "ds_read2st64_b32 %2, %9 offset0:0 offset1:2\n\t"
            "ds_read2st64_b32 %3, %9 offset0:4 offset1:6\n\t"
            "ds_read2st64_b32 %4, %8 offset0:8 offset1:10\n\t"
            "ds_read2st64_b32 %5, %8 offset0:12 offset1:14\n\t"
            "ds_read2st64_b32 %6, %9 offset0:8 offset1:10\n\t"
            "ds_read2st64_b32 %7, %9 offset0:12 offset1:14\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[0][1][0]), "=&v"(v[0][1][1]), "=&v"(v[1][0][0]),
              "=&v"(v[1][0][1]), "=&v"(v[1][1][0]), "=&v"(v[1][1][1])
            : "v"(a[0]), "v"(a[1]) : "memory");
        else if constexpr (NF == 4)
            asm volatile(
            "ds_read2st64_b32 %0, %16 offset0:0 offset1:4\n\t"
            "ds_read2st64_b32 %1, %16 offset0:8 offset1:12\n\t"
            "ds_read2st64_b32 %2, %17 offset0:0 offset1:4\n\t"
            "ds_read2st64_b32 %3, %17 offset0:8 offset1:12\n\t"
            "ds_read2st64_b32 %4, %18 offset0:0 offset1:4\n\t"
            "ds_read2st64_b32 %5, %18 offset0:8 offset1:12\n\t"
            "ds_read2st64_b32 %6, %19 offset0:0 offset1:4\n\t"
            "ds_read2st64_b32 %7, %19 offset0:8 offset1:12\n\t"
            "ds_read2st64_b32 %8, %16 offset0:16 offset1:20\n\t"
            "ds_read2st64_b32 %9, %16 offset0:24 offset1:28\n\t"
            "ds_read2st64_b32 %10, %17 offset0:16 offset1:20\n\t"
            "ds_read2st64_b32 %11, %17 offset0:24 offset1:28\n\t"
            "ds_read2st64_b32 %12, %18 offset0:16 offset1:20\n\t"
            "ds_read2st64_b32 %13, %18 offset0:24 offset1:28\n\t"
            "ds_read2st64_b32 %14, %19 offset0:16 offset1:20\n\t"
            "ds_read2st64_b32 %15, %19 offset0:24 offset1:28\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0][0][0]), "=&v"(v[0][0][1]), "=&v"(v[0][1][0]), "=&v"(v[0][1][1]), "=&v"(v[0][2][0]),
              "=&v"(v[0][2][1]), "=&v"(v[0][3][0]), "=&v"(v[0][3][1]), "=&v"(v[1][0][0]), "=&v"(v[1][0][1]),
              "=&v"(v[1][1][0]), "=&v"(v[1][1][1]), "=&v"(v[1][2][0]), "=&v"(v[1][2][1]), "=&v"(v[1][3][0]),
              "=&v"(v[1][3][1])
            : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]) : "memory");
    }
    __device__ __forceinline__ u32x4 get(int ks, int i) const {
        return u32x4{v[ks][i][0].x, v[ks][i][0].y, v[ks][i][1].x, v[ks][i][1].y};
    }
};

// The MFMAs of a k-tile.  fp32: k-slice j of every block before slice j + 1 (an MFMA on the
// accumulator of the one just issued would wait for it).
template <int MB, int NB, class FA, class FB>
__device__ __forceinline__ void wave_mfma(floatx4 (&acc)[MB][NB], const FA &fa, const FB &fb, half_t) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, fb.get(ks, j)),
                                                                   __builtin_bit_cast(halfx8, fa.get(ks, i)), acc[i][j],
                                                                   0, 0, 0);
}
template <int MB, int NB, class FA, class FB>
__device__ __forceinline__ void wave_mfma(floatx4 (&acc)[MB][NB], const FA &fa, const FB &fb, float) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        floatx4 a[MB], b[NB];
#pragma unroll
        for (int i = 0; i < MB; ++i) a[i] = __builtin_bit_cast(floatx4, fa.get(ks, i));
#pragma unroll
        for (int j = 0; j < NB; ++j) b[j] = __builtin_bit_cast(floatx4, fb.get(ks, j));
#define SKL_K_SLICE(C)                                                                              \
    _Pragma("unroll") for (int i = 0; i < MB; ++i) _Pragma("unroll") for (int j = 0; j < NB; ++j)   \
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j].C, a[i].C, acc[i][j], 0, 0, 0);
        SKL_K_SLICE(x)
        SKL_K_SLICE(y)
        SKL_K_SLICE(z)
        SKL_K_SLICE(w)
#undef SKL_K_SLICE
    }
}

// Grid: (tiles, splits); split y reduces k in [y k_per_split, (y + 1) k_per_split)
// (k_per_split whole k-tiles).  WPE: waves per SIMD the registers are budgeted for.
template <typename T, class Epi, bool A_KC, bool B_KC, bool REG, int MB, int NB, int W, int S, int WPE>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
    gemm_wave_kernel(GemmShape sh, const T *__restrict__ A, const T *__restrict__ B, typename Epi::Params ep) {
    typedef typename WaveOpSel<T, A_KC, 16 * MB, REG>::type OA;
    typedef typename WaveOpSel<T, B_KC, 16 * NB, REG>::type OB;
    static_assert(!REG || S == 1, "the register form keeps its next k-tile in registers");
    constexpr uint32_t BM = 16 * MB, BN = 16 * NB, BKE = 128 / sizeof(T), NT = 64 * W;
    constexpr uint32_t STAGE = (BM + BN) * 128;      // bytes per k-tile
    constexpr int IPT = OA::IPO + OB::IPO;           // loads per k-tile
    constexpr uint32_t EP = BN + 4;                  // floats per staged row
    constexpr uint32_t RING = W * S * STAGE, EPI = W * BM * EP * 4;
    __shared__ __attribute__((aligned(1024))) char smem[RING > EPI ? RING : EPI];
    lds_char *lsm = (lds_char *)(smem);

    const uint32_t tid = threadIdx.x, lane = tid & 63u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // workgroups past the tiles' run the bias / norm-parameter update
    if constexpr (std::is_same<typename Epi::Params, OptEpi>::value) {
        const uint32_t tiles = sh.tiles_m * sh.tiles_n;
        if (blockIdx.x >= tiles) {
            vec_opt_block<T, NT>(ep.vec, blockIdx.x - tiles);
            return;
        }
    }
    uint32_t tm, tn;
    tile_coords(blockIdx.x, sh.tiles_m, sh.tiles_n, tm, tn);
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t kbeg = blockIdx.y * sh.k_per_split;
    const uint32_t kend = min(sh.K, kbeg + sh.k_per_split);
    const uint32_t kt0 = wave, kt1 = (kend - kbeg + BKE - 1) / BKE;   // k-tiles of the slice

    const uint32_t lds0 = (uint32_t)(uintptr_t)lsm + wave * (S * STAGE);
    OA oa;
    OB ob;
    // m/n-contiguous operands start at the slice's first k-row (only dW, with both, is split)
    oa.init(A_KC ? A : A + (uint64_t)kbeg * sh.lda, sh.lda, sh.M, A_KC ? sh.K : kend - kbeg, m0, lane, lds0);
    ob.init(B_KC ? B : B + (uint64_t)kbeg * sh.ldb, sh.ldb, sh.N, B_KC ? sh.K : kend - kbeg, n0, lane, lds0 + BM * 128);

    floatx4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // fragments of the k-tile in the stage, k past K zeroed where it is not by range
    auto frags = [&](auto &fa, auto &fb, uint32_t kt, uint32_t stage) {
        fa.read(oa, stage);
        fb.read(ob, stage);
        if constexpr (A_KC) {
            if (sh.K % OA::CE != 0 && kt == sh.K / BKE) {
                fa.cut(kt, sh.K, lane);
                if constexpr (B_KC) fb.cut(kt, sh.K, lane);
            }
        }
    };
    if constexpr (REG) {
        u32x4 ra[OA::IPO], rb[OB::IPO];
        if (kt0 < kt1) {
            oa.load(kt0, ra);
            ob.load(kt0, rb);
        }
        for (uint32_t kt = kt0; kt < kt1; kt += W) {
            oa.put(ra, lane);
            ob.put(rb, lane);
            if (kt + W < kt1) {
                oa.load(kt + W, ra);
                ob.load(kt + W, rb);
            }
            WaveFrags<T, A_KC, MB> fa;
            WaveFrags<T, B_KC, NB> fb;
            frags(fa, fb, kt, 0);   // a wave's LDS accesses complete in order
            wave_mfma<MB, NB>(acc, fa, fb, T());
        }
    } else {
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (kt0 + s * W < kt1) {
                oa.issue(kt0 + s * W, s * STAGE);
                ob.issue(kt0 + s * W, s * STAGE);
            }
        for (uint32_t kb = kt0; kb < kt1; kb += S * W) {
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const uint32_t kt = kb + s * W;
                if (kt >= kt1) break;
                // this stage's loads have landed (in order: only those of later stages may pend)
                if (kt + (S - 1) * W < kt1)
                    wait_vmcnt<(S - 1) * IPT>();
                else
                    wait_vmcnt<0>();
                asm volatile("" ::: "memory");
                WaveFrags<T, A_KC, MB> fa;
                WaveFrags<T, B_KC, NB> fb;
                frags(fa, fb, kt, s * STAGE);
                __builtin_amdgcn_sched_barrier(0);
                if (kt + S * W < kt1) {   // the stage is read: refill it
                    oa.issue(kt + S * W, s * STAGE);
                    ob.issue(kt + S * W, s * STAGE);
                }
                wave_mfma<MB, NB>(acc, fa, fb, T());
            }
        }
        wait_vmcnt<0>();
    }
    lds_barrier();   // every wave is done with its ring: the partial tiles go over it

    // lane l of block (i, j): columns 4 (l / 16) .. + 3 of row l % 16
    float *E = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
            *reinterpret_cast<floatx4 *>(E + (wave * BM + 16 * i + (lane & 15u)) * EP + 16 * j + 4 * (lane >> 4)) =
                acc[i][j];
    lds_barrier();
    if constexpr (EpiSums<Epi>::value) {
        // the hidden error: 4 columns per lane (the launcher has checked their alignment), a
        // thread's group of columns fixed; the operands of up to 4 rows loaded before any use
        constexpr uint32_t QN = BM * BN / 4, GR = BN / 4, ACT = QN < NT ? QN : NT, ROWS = QN / ACT;
        constexpr uint32_t UB = ROWS < 4 ? ROWS : 4;
        static_assert(NT % GR == 0 && ROWS % UB == 0, "one column group per thread");
        static_assert((ACT / GR) * 3 * BN * 4 <= sizeof(smem), "column sums fit the ring");
        const uint32_t group = tid % GR, n = n0 + 4 * group;
        const bool live = tid < ACT && n + 3 < sh.N;
        typename EpiSums<Epi>::Acc csum{};
        if (live) {
            const typename Epi::Col col = Epi::column(ep, n);
#pragma unroll 1
            for (uint32_t u0 = 0; u0 < ROWS; u0 += UB) {
                typename Epi::Pre pre[UB];
#pragma unroll
                for (uint32_t u = 0; u < UB; ++u) {
                    const uint32_t m = m0 + (tid + (u0 + u) * ACT) / GR;
                    if (m < sh.M) Epi::load(ep, (uint64_t)m * Epi::ldc(ep) + n, m, pre[u]);
                }
#pragma unroll
                for (uint32_t u = 0; u < UB; ++u) {
                    const uint32_t r = (tid + (u0 + u) * ACT) / GR, m = m0 + r;
                    if (m >= sh.M) continue;
                    floatx4 v = *reinterpret_cast<const floatx4 *>(E + r * EP + 4 * group);
#pragma unroll
                    for (int w = 1; w < W; ++w)
                        v += *reinterpret_cast<const floatx4 *>(E + (w * BM + r) * EP + 4 * group);
                    Epi::finish(ep, (uint64_t)m * Epi::ldc(ep) + n, m, n, v, col, pre[u], csum);
                }
            }
        }
        lds_barrier();   // every wave is done reading E
        Epi::template flush_slots<ACT / GR, BN, NT>(ep, csum, E, tid, tid / GR, group, tm, n0);
    } else {
    if (sh.nv) {   // output rows on 4-element boundaries: 4 columns per lane
        // (the optimiser's state loaded ahead of this sum made a 2048 x 1000 dW 3 us slower)
        for (uint32_t q = tid; q < BM * BN / 4; q += NT) {
            const uint32_t r = q / (BN / 4), c = (q % (BN / 4)) * 4;
            floatx4 v = *reinterpret_cast<const floatx4 *>(E + r * EP + c);
#pragma unroll
            for (int w = 1; w < W; ++w) v += *reinterpret_cast<const floatx4 *>(E + (w * BM + r) * EP + c);
            Epi::apply(ep, sh, m0 + r, n0 + c, v, blockIdx.y);
        }
    } else {
        // otherwise an element per lane, consecutive lanes consecutive columns (NT is a multiple of BN: a thread keeps its column)
        static_assert(NT % BN == 0, "one column per thread");
        const uint32_t c = tid % BN, n = n0 + c;
        if (n < sh.N) {
            const typename Epi::Col1 col = Epi::column1(ep, n);
            for (uint32_t r = tid / BN; r < BM && m0 + r < sh.M; r += NT / BN) {
                float v = E[r * EP + c];
#pragma unroll
                for (int w = 1; w < W; ++w) v += E[(w * BM + r) * EP + c];
                Epi::apply1(ep, m0 + r, n, v, col, blockIdx.y);
            }
        }
    }
    }
    // or it rides behind the tiles (the launcher's choice)
    if constexpr (std::is_same<typename Epi::Params, OptEpi>::value) {
        for (uint32_t blk = blockIdx.x; blk < ep.vec_blocks; blk += gridDim.x) vec_opt_block<T, NT>(ep.vec, blk);
    }
}

}  // namespace skl
