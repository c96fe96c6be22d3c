// gemm_tile.hpp — device-side building blocks of the gfx950 GEMM.
//
// BLIS computes C := beta*C + alpha*A*B with five loops around a register
// microkernel: jc/pc/ic blocking with packm copies of A and B into cache-
// resident micro-panels (frame/3/gemm/bli_gemm_blk_var{1,2,3}.c,
// frame/1m/packm/bli_packm_blk_var1.c), a macro-kernel over MR x NR tiles
// (frame/3/gemm/bli_gemm_ker_var2.c:37-284) and the microkernel itself
// (ref_kernels/3/bli_gemm_ref.c:163-317).
//
// On gfx950 the same blocking is expressed as:
//   jc/ic loops   -> the workgroup grid (one BM x BN tile of C per workgroup),
//                    rasterised in groups and remapped so that neighbouring
//                    tiles share an XCD's L2;
//   pc loop       -> the in-kernel k loop over BK-deep slabs;
//   packm         -> coalesced 16-byte global loads of a BM x BK slab of A and
//                    a BK x BN slab of B into double-buffered LDS, stored
//                    k-major ("packed panels") regardless of the source layout;
//   jr/ir + ukr   -> each wave owns a WM x WN sub-tile built from 16x16x4
//                    MFMA blocks whose accumulators stay in registers for the
//                    whole k loop.
// Inside a wave tile, MFMA block i, row r maps to wave row TM*r + i (and block
// j, column c to wave column TN*c + j). With that interleave a lane's TM A
// fragments (and TN B fragments) are contiguous in LDS, so they are fetched
// as 16-byte vectors, and each accumulator register of a lane covers TM
// consecutive rows of C, which are written back as 16-byte vectors.
//
// Semantics kept from the reference microkernel: beta == 0 overwrites C
// without reading it (bli_gemm_ref.c:257-310); edges m < BM, n < BN and a
// partial last k slab are handled in-kernel by zero-filled loads and masked
// stores.
#pragma once

#include <type_traits>

#include <hip/hip_runtime.h>
#include <cstdint>

namespace blis_amd {
namespace dev {

typedef double d2_t __attribute__((ext_vector_type(2)));
typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float  f4_t __attribute__((ext_vector_type(4)));
// 16-byte vectors at element alignment, for C: gfx950 takes vector accesses
// at any dword address, so a column of C needs no 16-byte alignment.
typedef d2_t d2u_t __attribute__((aligned(8)));
typedef f4_t f4u_t __attribute__((aligned(4)));

template <typename T> struct Mma;
// Operand layout (both types, measured on gfx950): lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16]. Accumulator layout differs:
//   f32 16x16x4: lane l, register r holds D[4*(l/16) + r][l % 16];
//   f64 16x16x4: lane l, register r holds D[4*r + l/16][l % 16].
// acc_row(r, g) gives the D row of register r in lane group g = l / 16.
template <> struct Mma<double> {
    using acc_t = d4_t;
    using vec_t = d2_t;             // 16-byte vector
    using uvec_t = d2u_t;           // the same at element alignment
    static constexpr int V = 2;     // elements per 16-byte vector
    __device__ static inline acc_t mma(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static constexpr int acc_row(int r, int g) { return 4 * r + g; }
};
template <> struct Mma<float> {
    using acc_t = f4_t;
    using vec_t = f4_t;
    using uvec_t = f4u_t;
    static constexpr int V = 4;
    __device__ static inline acc_t mma(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __device__ static constexpr int acc_row(int r, int g) { return 4 * g + r; }
};

// Workgroup barrier that orders LDS accesses only. __syncthreads() also waits
// for every global load in flight, which undoes prefetching across it.
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Workgroup tile BM x BN, k slab BK, wave tile WM x WN.
template <typename T, int BM_, int BN_, int BK_, int WM_, int WN_>
struct TileCfg {
    using M = Mma<T>;
    static constexpr int BM = BM_, BN = BN_, BK = BK_, WM = WM_, WN = WN_;
    static constexpr int WGM = BM / WM, WGN = BN / WN;
    static constexpr int NW = WGM * WGN;          // waves per workgroup
    static constexpr int NT = 64 * NW;            // threads per workgroup
    static constexpr int TM = WM / 16, TN = WN / 16;
    static constexpr int V = M::V;
    // LDS row pitch: rows are padded by one 16-byte vector (a one-element
    // pad for FP64 was measured to raise bank conflicts: it costs the 16-byte
    // alignment of the fragment reads).
    static constexpr int PAD = V;
    static constexpr int LDA = BM + PAD;
    static constexpr int LDB = BN + PAD;
    static constexpr int A_ELEMS = BK * LDA;
    static constexpr int B_ELEMS = BK * LDB;
    static constexpr int STAGE = A_ELEMS + B_ELEMS;
    static constexpr int NVA = (BM * BK / V) / NT;  // 16-byte vectors per thread
    static constexpr int NVB = (BN * BK / V) / NT;
    // Waves per SIMD a kernel of this tile is compiled for: whole workgroups,
    // as many as the LDS holds, while the registers of a wave (accumulators,
    // staged vectors, two sets of fragments and about 20 more) fit. The
    // unrolled k loop would take what it likes otherwise: 166 registers and
    // one workgroup per CU for the 128 x 128 FP64 tile, 17.8 ms at 8192^3
    // against 15.0 ms with two. Loads without a descriptor keep 64-bit addresses
    // and bounds besides, so their kernels give up a workgroup for registers (the
    // 128 x 64 FP64 tile spilled up to 15).
    static constexpr int waves_per_eu(bool buf) {
        const int es = (int)sizeof(T) / 4, per = NW >= 4 ? NW / 4 : 1;
        const int regs = TM * TN * 4 * es + (NVA + NVB) * 4 + 2 * (TM + TN) * es + 20;
        int w = 163840 / (2 * STAGE * (int)sizeof(T)) * NW / 4;
        if (w > 8) w = 8;
        while (w > per && 512 / w / 8 * 8 < regs) w -= per;
        if (!buf && w > per) w -= per;
        return w < 1 ? 1 : w;
    }
    static_assert(WM % 16 == 0 && WN % 16 == 0, "wave tile must be 16-aligned");
    static_assert(BK % 4 == 0 && BK % V == 0, "BK must cover MFMA k and vectors");
    static_assert((BM * BK / V) % NT == 0 && NVA >= 1, "A slab must split evenly");
    static_assert((BN * BK / V) % NT == 0 && NVB >= 1, "B slab must split evenly");
    static_assert(BM % V == 0 && BN % V == 0, "tile must hold whole vectors");
};

// Parameters of one GEMM problem as seen by a tile routine. Layout flags are
// template parameters of the routine: A_K means A is contiguous along k
// (A_eff(i,p) = a[p + i*lda]), otherwise along m (a[i + p*lda]); B_K means B
// is contiguous along k (B_eff(p,j) = b[p + j*ldb]), otherwise along n
// (b[j + p*ldb]). C(i,j) = c[i*c_si + j*c_sj].
template <typename T>
struct TileProblem {
    const T* a;
    const T* b;
    T*       c;
    int64_t  m, n, k;
    int64_t  lda, ldb;
    int64_t  c_si, c_sj;
    T        alpha, beta;
    int      vec_a, vec_b;   // 16-byte alignment of A and B (loads without a descriptor)
    int      vec_c;          // c_si == 1: C is stored in vectors
    int      a_k, b_k;       // layouts, where they are not template parameters
};

// One operand of a tile, read a k slab at a time. The operand is X_eff,
// rows x K, with X_eff(r, p) = x[p + r*ld] when K_CONTIG, else x[r + p*ld];
// the tile covers rows [row0, row0 + ROWS). Each thread owns NV 16-byte
// vectors of a slab, between their load and their LDS store.
//
// BUF: the slab is read through a buffer descriptor whose base moves with
// the slab (scalar arithmetic) and whose extent ends at the operand's last
// element, so every lane of every tile issues the same 16-byte loads at the
// same offsets, with no branch, no clamp and no 64-bit vector address: the
// hardware returns zero past the end. What else an edge tile reads between
// the operand's first and last element (the next column's rows, a row's
// padding) lands in tile rows outside the matrix, which feed only outputs
// that are never stored; the k positions past K of a K_CONTIG operand, which
// every output sums over, are zeroed on the way to LDS. Buffer loads need
// 4-byte alignment only, so odd leading dimensions take the same path. It
// needs lines along k that neither overlap nor run backwards (those along the
// rows may overlap) and slab offsets below 2^32 bytes (buf_ok in
// gemm_plan.hpp). Against 64-bit addresses with element loads on edge and
// unaligned tiles (device time): 1999 x 1501 x 1003 T/N on odd
// leading dimensions 150 against 170 us, 512^3 12.2 against 13.5 us, the
// 10,000-problem FP64 batch 1546 against 1739 us (its 64 x 64 kernels no
// longer spill); 8192^3, all interior, is unchanged.
// Not BUF (the other strides): 16-byte loads for slabs wholly inside an
// aligned operand, element loads behind bounds checks otherwise.
template <typename T, class TL, int ROWS, bool K_CONTIG, int NV, bool BUF>
struct SlabLoader {
    using vec_t = typename Mma<T>::vec_t;
    static constexpr int V = TL::V;
    static constexpr int LD = ROWS + TL::PAD;   // LDS row pitch
    // Vectors along the contiguous direction, and slab lines between a
    // thread's consecutive vectors.
    static constexpr int CV = K_CONTIG ? TL::BK / V : ROWS / V;
    static constexpr int LINES = TL::NT / CV;
    static_assert(TL::NT % CV == 0, "a thread's vectors must be whole lines apart");
    vec_t r[NV];
    const T* x;
    int64_t ld, K, rows, row0;
    int vec;
    // BUF: start of the next slab to load, bytes from there to the operand's
    // end, and the thread's first offset.
    const char* base;
    int64_t left;
    uint32_t off0;

    __device__ inline void init(const T* x_, int64_t rows_, int64_t K_, int64_t ld_, int vec_,
                                int64_t row0_, int tid) {
        x = x_; ld = ld_; K = K_; rows = rows_; row0 = row0_; vec = vec_;
        if constexpr (BUF) {
            constexpr int ES = (int)sizeof(T);
            const int c = tid % CV, l = tid / CV;
            off0 = (uint32_t)l * ((uint32_t)ld * ES) + (uint32_t)(c * 16);
            base = (const char*)(x + (K_CONTIG ? row0 * ld : row0));
            left = (K_CONTIG ? (rows - 1 - row0) * ld + K : (K - 1) * ld + (rows - row0)) * ES;
        }
    }

    // Load slab s; BUF loaders are called for consecutive slabs.
    __device__ inline void load(int s, int tid) {
        if constexpr (BUF) {
            const uint32_t n = (uint32_t)(left >> 32) != 0 ? 0xFFFFFFFFu : (uint32_t)left;
            auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)n, 0x00020000);
            const uint32_t step = (uint32_t)LINES * ((uint32_t)ld * (uint32_t)sizeof(T));
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                auto t = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off0 + q * step), 0, 0);
                r[q] = __builtin_bit_cast(vec_t, t);
            }
            const int64_t adv = (K_CONTIG ? (int64_t)TL::BK : TL::BK * ld) * (int64_t)sizeof(T);
            base += adv;
            left -= adv;
        } else {
            const int64_t k0 = (int64_t)s * TL::BK;
            const bool whole = vec && row0 + ROWS <= rows && k0 + TL::BK <= K;   // uniform
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                const int v = tid + q * TL::NT;
                const int c = v % CV, l = v / CV;
                const int64_t row = row0 + (K_CONTIG ? l : c * V), pk = k0 + (K_CONTIG ? c * V : l);
                const T* src = K_CONTIG ? x + pk + row * ld : x + row + pk * ld;
                if (whole) {
                    r[q] = *reinterpret_cast<const vec_t*>(src);
                    continue;
                }
                const int64_t run = K_CONTIG ? K - pk : rows - row;   // elements left along it
                const bool line = K_CONTIG ? row < rows : pk < K;
                if (vec && line && run >= V) {
                    r[q] = *reinterpret_cast<const vec_t*>(src);
                } else {
#pragma unroll
                    for (int e = 0; e < V; ++e) {
                        T val = T(0);
                        if (line && e < run) val = src[e];
                        r[q][e] = val;
                    }
                }
            }
        }
    }

    // Store the loaded slab into an LDS stage, k-major; kext: its k extent
    // (BK but for a partial last slab). The mask is applied to every slab: a
    // branch around it would end the loop's basic block, and with it the
    // compiler's freedom to move loads, LDS traffic and MFMAs past each other
    // (8192^3 FP64 16.0 ms with the branch, 15.0 without).
    __device__ inline void store(T* S, int kext, int tid) {
        if constexpr (BUF && K_CONTIG) {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                const bool out = (tid % CV) * V + e >= kext;
#pragma unroll
                for (int q = 0; q < NV; ++q) r[q][e] = out ? T(0) : r[q][e];
            }
        }
#pragma unroll
        for (int q = 0; q < NV; ++q) {
            const int v = tid + q * TL::NT;
            const int c = v % CV, l = v / CV;
            if constexpr (!K_CONTIG) {
                *reinterpret_cast<vec_t*>(S + l * LD + c * V) = r[q];
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) S[(c * V + e) * LD + l] = r[q][e];
            }
        }
    }
};

// The same with the layout decided at run time, for kernels that walk problems
// of every layout (the batch): the layout only enters a thread's offsets, the
// slab stride and the LDS store, so it costs a uniform branch around the stores
// and no registers. Not BUF: element loads behind bounds checks, for strides
// that a descriptor does not take.
template <typename T, class TL, int ROWS, int NV, bool BUF>
struct SlabLoaderRt {
    using vec_t = typename Mma<T>::vec_t;
    static constexpr int V = TL::V;
    static constexpr int LD = ROWS + TL::PAD;
    static constexpr int CVK = TL::BK / V, CVR = ROWS / V;   // vectors along k, along rows
    static_assert(TL::NT % CVK == 0 && TL::NT % CVR == 0, "whole lines apart");
    vec_t r[NV];
    bool k_contig;
    const char* base;
    int64_t left, adv;      // BUF: as SlabLoader's; else lines and length of a line left
    uint32_t off0, step;
    int64_t ld;             // not BUF

    __device__ inline void init(const T* x, int64_t rows, int64_t K, int64_t ld_, int k_contig_,
                                int64_t row0, int tid) {
        constexpr int ES = (int)sizeof(T);
        k_contig = k_contig_ != 0;
        const int c = k_contig ? tid % CVK : tid % CVR, l = k_contig ? tid / CVK : tid / CVR;
        if constexpr (BUF) {
            const uint32_t line = (uint32_t)ld_ * ES;
            off0 = (uint32_t)l * line + (uint32_t)(c * 16);
            step = (uint32_t)(k_contig ? TL::NT / CVK : TL::NT / CVR) * line;
            adv = (k_contig ? (int64_t)TL::BK : TL::BK * ld_) * ES;
            base = (const char*)(x + (k_contig ? row0 * ld_ : row0));
            left = (k_contig ? (rows - 1 - row0) * ld_ + K : (K - 1) * ld_ + (rows - row0)) * ES;
        } else {
            ld = ld_;
            // This thread's first element, and what is left of lines and of a line
            // from there; a slab moves along the line or to later lines.
            base = (const char*)(x + (k_contig ? (row0 + l) * ld : row0 + l * ld) + c * V);
            left = (k_contig ? rows - row0 : K) - l;
            adv = (k_contig ? K : rows - row0) - c * V;
        }
    }

    __device__ inline void load(int, int) {
        if constexpr (BUF) {
            const uint32_t n = (uint32_t)(left >> 32) != 0 ? 0xFFFFFFFFu : (uint32_t)left;
            auto rs = __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)n, 0x00020000);
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                auto t = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(off0 + q * step), 0, 0);
                r[q] = __builtin_bit_cast(vec_t, t);
            }
            base += adv;
            left -= adv;
        } else {
            const int lines = k_contig ? TL::NT / CVK : TL::NT / CVR;
#pragma unroll
            for (int q = 0; q < NV; ++q) {
                const T* src = (const T*)base + q * lines * ld;
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    T val = T(0);
                    if (q * lines < left && e < adv) val = src[e];
                    r[q][e] = val;
                }
            }
            base += (k_contig ? (int64_t)TL::BK : TL::BK * ld) * (int64_t)sizeof(T);
            if (k_contig) adv -= TL::BK;
            else left -= TL::BK;
        }
    }

    __device__ inline void store(T* S, int kext, int tid) {
        if (k_contig) {
            const int c = tid % CVK, l = tid / CVK;
#pragma unroll
            for (int q = 0; q < NV; ++q)
#pragma unroll
                for (int e = 0; e < V; ++e)
                    S[(c * V + e) * LD + l + q * (TL::NT / CVK)] = c * V + e < kext ? r[q][e] : T(0);
        } else {
            const int c = tid % CVR, l = tid / CVR;
#pragma unroll
            for (int q = 0; q < NV; ++q)
                *reinterpret_cast<vec_t*>(S + (l + q * (TL::NT / CVR)) * LD + c * V) = r[q];
        }
    }
};

// Rank-BK update of the wave's accumulators from one LDS stage.
template <typename T, class TL>
__device__ inline void mma_slab(const T* As, const T* Bs,
                                typename Mma<T>::acc_t (&acc)[TL::TM][TL::TN],
                                int wm0, int wn0, int lane) {
    using vec_t = typename Mma<T>::vec_t;
    constexpr int V = TL::V;
    const int lr = lane & 15, lk = lane >> 4;
    auto fragments = [&](int ks, T (&af)[TL::TM], T (&bf)[TL::TN]) {
        const T* ap = As + (ks + lk) * TL::LDA + wm0 + TL::TM * lr;
        const T* bp = Bs + (ks + lk) * TL::LDB + wn0 + TL::TN * lr;
        if constexpr (TL::TM % V == 0) {
#pragma unroll
            for (int q = 0; q < TL::TM / V; ++q) {
                vec_t t = *reinterpret_cast<const vec_t*>(ap + q * V);
#pragma unroll
                for (int e = 0; e < V; ++e) af[q * V + e] = t[e];
            }
        } else {
#pragma unroll
            for (int i = 0; i < TL::TM; ++i) af[i] = ap[i];
        }
        if constexpr (TL::TN % V == 0) {
#pragma unroll
            for (int q = 0; q < TL::TN / V; ++q) {
                vec_t t = *reinterpret_cast<const vec_t*>(bp + q * V);
#pragma unroll
                for (int e = 0; e < V; ++e) bf[q * V + e] = t[e];
            }
        } else {
#pragma unroll
            for (int j = 0; j < TL::TN; ++j) bf[j] = bp[j];
        }
    };
    auto multiply = [&](const T (&af)[TL::TM], const T (&bf)[TL::TN]) {
#pragma unroll
        for (int i = 0; i < TL::TM; ++i)
#pragma unroll
            for (int j = 0; j < TL::TN; ++j)
                acc[i][j] = Mma<T>::mma(af[i], bf[j], acc[i][j]);
    };
    if constexpr (sizeof(T) == 8) {
        // The next k step's fragments are read ahead of this one's MFMAs:
        // 1% on the FP64 tiles (128 x 128 14.68 against 14.80 ms at 8192^3
        // N/T, 64 x 128 249 against 257 us at 2000^3); the FP32 tiles gain
        // nothing (256 x 128 at 8192^3 N/N 7.95 against 7.66 ms).
        T af[2][TL::TM], bf[2][TL::TN];
        fragments(0, af[0], bf[0]);
#pragma unroll
        for (int i = 0; i < TL::BK / 4; ++i) {
            if (i + 1 < TL::BK / 4) fragments(4 * (i + 1), af[(i + 1) & 1], bf[(i + 1) & 1]);
            multiply(af[i & 1], bf[i & 1]);
        }
    } else {
#pragma unroll
        for (int ks = 0; ks < TL::BK; ks += 4) {
            T af[TL::TM], bf[TL::TN];
            fragments(ks, af, bf);
            multiply(af, bf);
        }
    }
}

// alpha*acc + beta*c as one fixed operation sequence (a product, then a
// fused multiply-add), used by every store path. Each output element then
// has the same arithmetic whatever the tile shape or store path, so every
// tile configuration gives bit-identical results.
template <typename T>
__device__ inline T epilogue(T alpha, T acc, T beta, T old) {
    return fma(beta, old, alpha * acc);
}

// Write the wave's accumulators: C := alpha*acc + beta*C (beta == 0 does not
// read C). For accumulator register r, a lane in group g = lane/16 owns the
// TM consecutive wave rows TM*acc_row(r, g) + [0, TM) of wave column
// TN*(lane%16) + j, written as 16-byte vectors when they fit.
template <typename T, class TL, bool INTERIOR>
__device__ inline void store_tile(const TileProblem<T>& p,
                                  const typename Mma<T>::acc_t (&acc)[TL::TM][TL::TN],
                                  int64_t row0, int64_t col0, int lane) {
    using vec_t = typename Mma<T>::vec_t;
    using uvec_t = typename Mma<T>::uvec_t;
    constexpr int V = TL::V;
    constexpr int TM = TL::TM;
    const int g = lane >> 4, lc = lane & 15;
    const T alpha = p.alpha, beta = p.beta;
#pragma unroll
    for (int j = 0; j < TL::TN; ++j) {
        const int64_t col = col0 + TL::TN * lc + j;
        if (!INTERIOR && col >= p.n) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t rb = row0 + (int64_t)TM * Mma<T>::acc_row(r, g);
            if constexpr (TM % V == 0) {
                if (INTERIOR || (p.vec_c && rb + TM <= p.m)) {
                    T* dst = p.c + rb + col * p.c_sj;
#pragma unroll
                    for (int q = 0; q < TM / V; ++q) {
                        vec_t o;
                        if (beta == T(0)) {
#pragma unroll
                            for (int e = 0; e < V; ++e) o[e] = alpha * acc[q * V + e][j][r];
                        } else {
                            const vec_t old = *reinterpret_cast<const uvec_t*>(dst + q * V);
#pragma unroll
                            for (int e = 0; e < V; ++e)
                                o[e] = epilogue(alpha, acc[q * V + e][j][r], beta, old[e]);
                        }
                        *reinterpret_cast<uvec_t*>(dst + q * V) = o;
                    }
                    continue;
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int64_t row = rb + i;
                if (row < p.m) {
                    T* dst = p.c + row * p.c_si + col * p.c_sj;
                    *dst = (beta == T(0)) ? alpha * acc[i][j][r]
                                          : epilogue(alpha, acc[i][j][r], beta, *dst);
                }
            }
        }
    }
}

// Stored region of a structured C (gemmt, syrk, syr2k): element (i, j) is
// written only when it lies on the stored side of the diagonal j - i == doff
// (lower: j - i <= doff; upper: j - i >= doff), BLIS's convention for
// diagonal offsets (frame/include/bli_param_macro_defs.h:638-673).
// uplo: 0 = every element, 1 = lower, 2 = upper.
struct CMask {
    int     uplo = 0;
    int64_t doff = 0;
};

// store_tile restricted to the stored region of C: a TM-row vector is
// written whole when all its rows are stored, otherwise element by element.
// The per-element arithmetic is the same epilogue() as store_tile.
template <typename T, class TL>
__device__ inline void store_tile_masked(const TileProblem<T>& p,
                                         const typename Mma<T>::acc_t (&acc)[TL::TM][TL::TN],
                                         int64_t row0, int64_t col0, int lane, CMask cm) {
    using vec_t = typename Mma<T>::vec_t;
    using uvec_t = typename Mma<T>::uvec_t;
    constexpr int V = TL::V;
    constexpr int TM = TL::TM;
    const int g = lane >> 4, lc = lane & 15;
    const T alpha = p.alpha, beta = p.beta;
    const bool lower = cm.uplo == 1;
#pragma unroll
    for (int j = 0; j < TL::TN; ++j) {
        const int64_t col = col0 + TL::TN * lc + j;
        if (col >= p.n) continue;
        // lower: rows i >= lim are stored; upper: rows i <= lim.
        const int64_t lim = col - cm.doff;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t rb = row0 + (int64_t)TM * Mma<T>::acc_row(r, g);
            if constexpr (TM % V == 0) {
                const bool all_in = lower ? rb >= lim : rb + TM - 1 <= lim;
                if (all_in && p.vec_c && rb + TM <= p.m) {
                    T* dst = p.c + rb + col * p.c_sj;
#pragma unroll
                    for (int q = 0; q < TM / V; ++q) {
                        vec_t o;
                        if (beta == T(0)) {
#pragma unroll
                            for (int e = 0; e < V; ++e) o[e] = alpha * acc[q * V + e][j][r];
                        } else {
                            const vec_t old = *reinterpret_cast<const uvec_t*>(dst + q * V);
#pragma unroll
                            for (int e = 0; e < V; ++e)
                                o[e] = epilogue(alpha, acc[q * V + e][j][r], beta, old[e]);
                        }
                        *reinterpret_cast<uvec_t*>(dst + q * V) = o;
                    }
                    continue;
                }
            }
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int64_t row = rb + i;
                const bool in = lower ? row >= lim : row <= lim;
                if (row < p.m && in) {
                    T* dst = p.c + row * p.c_si + col * p.c_sj;
                    *dst = (beta == T(0)) ? alpha * acc[i][j][r]
                                          : epilogue(alpha, acc[i][j][r], beta, *dst);
                }
            }
        }
    }
}

// Epilogue through LDS, for tiles whose wave rows per lane are too few for
// full-width vector access to C: the accumulators are written to LDS as a
// column-major BM x BN tile (column pitch BM + V), then each thread updates
// whole 16-byte chunks of C columns, so a wave reads and writes entire
// cache lines. The arithmetic per element is the same epilogue() as
// store_tile. smem must hold BN * (BM + V) elements; the caller has
// synchronised after the last use of smem by the k loop.
template <typename T, class TL>
__device__ inline void store_tile_lds(const TileProblem<T>& p,
                                      const typename Mma<T>::acc_t (&acc)[TL::TM][TL::TN],
                                      int64_t m0, int64_t n0, int wm0, int wn0, T* smem) {
    using vec_t = typename Mma<T>::vec_t;
    using uvec_t = typename Mma<T>::uvec_t;
    constexpr int V = TL::V;
    constexpr int TM = TL::TM;
    constexpr int LDC = TL::BM + V;
    static_assert(TL::BN * LDC <= 2 * TL::STAGE, "epilogue tile must fit the LDS stages");
    const int tid = threadIdx.x;
    const int lane = tid & 63, g = lane >> 4, lc = lane & 15;
#pragma unroll
    for (int j = 0; j < TL::TN; ++j) {
        const int col = wn0 + TL::TN * lc + j;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = wm0 + TM * Mma<T>::acc_row(r, g);
#pragma unroll
            for (int i = 0; i < TM; ++i) smem[col * LDC + row + i] = acc[i][j][r];
        }
    }
    __syncthreads();
    constexpr int CH = TL::BM / V;                 // 16-byte chunks per column
    const T alpha = p.alpha, beta = p.beta;
#pragma unroll
    for (int q0 = 0; q0 < CH * TL::BN; q0 += TL::NT) {
        const int q = q0 + tid;
        if ((CH * TL::BN) % TL::NT != 0 && q >= CH * TL::BN) break;
        const int col = q / CH, ch = q % CH;
        const int64_t gc = n0 + col, gr = m0 + (int64_t)ch * V;
        if (gc >= p.n || gr >= p.m) continue;
        const T* src = smem + col * LDC + ch * V;
        T* dst = p.c + gr * p.c_si + gc * p.c_sj;
        if (p.vec_c && gr + V <= p.m) {
            const vec_t a = *reinterpret_cast<const vec_t*>(src);
            vec_t o;
            if (beta == T(0)) {
#pragma unroll
                for (int e = 0; e < V; ++e) o[e] = alpha * a[e];
            } else {
                const vec_t old = *reinterpret_cast<const uvec_t*>(dst);
#pragma unroll
                for (int e = 0; e < V; ++e) o[e] = epilogue(alpha, a[e], beta, old[e]);
            }
            *reinterpret_cast<uvec_t*>(dst) = o;
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                if (gr + e >= p.m) break;
                T* d = dst + e * p.c_si;
                *d = (beta == T(0)) ? alpha * src[e] : epilogue(alpha, src[e], beta, *d);
            }
        }
    }
}

// Compute one BM x BN tile (tile coordinates tm, tn) of one problem. smem
// must hold 2*TL::STAGE elements. The caller synchronises before reusing smem.
// LOADS: how the operands are read.
// PF: k slabs whose global loads are in flight while a slab is multiplied
// (1: one register buffer; 2: two, for tiles that stream their operands
// from HBM, such as the small problems of a batch).
// The loaded values, and so the arithmetic, are the same in every variant.
// Pull the C tile's cache lines into L2 ahead of the epilogue (beta != 0):
// one 4-byte global->LDS load per 128-byte line of each tile column, into a
// scratch LDS area of NT words that nothing reads. Addresses are clamped
// into the matrix. C must be column-stored (c_si == 1).
typedef __attribute__((address_space(3))) void* lds_ptr_t;
template <typename T, class TL>
__device__ inline void prefetch_c(const TileProblem<T>& p, int64_t m0, int64_t n0, int* sink) {
    constexpr int LPC = (TL::BM * (int)sizeof(T) + 127) / 128;   // lines per column
    constexpr int ROWS_PER_LINE = 128 / (int)sizeof(T);
    const int tid = threadIdx.x;
    if (p.beta == T(0) || p.c_si != 1) return;
    const int col = tid / LPC, line = tid % LPC;
    if (col >= TL::BN) return;
    const int64_t r = min(m0 + (int64_t)line * ROWS_PER_LINE, p.m - 1);
    const int64_t c = min(n0 + (int64_t)col, p.n - 1);
    int* dst = sink + (tid & ~63);
    __builtin_amdgcn_global_load_lds((const void*)(p.c + r + c * p.c_sj), (lds_ptr_t)dst, 4, 0, 0);
}

// How a tile routine reads its operands: Guarded and Buffer are SlabLoader,
// RuntimeLayout and RuntimeGuarded SlabLoaderRt (A_K and B_K are not used then).
enum class Loads { Guarded, Buffer, RuntimeLayout, RuntimeGuarded };

template <typename T, class TL, bool A_K, bool B_K, Loads LOADS, int PF, bool LDS_EPI,
          bool C_PF = false, bool MASK = false>
__device__ inline void gemm_tile_impl(const TileProblem<T>& p, int64_t m0, int64_t n0, T* smem,
                                      int* sink = nullptr, CMask cm = CMask{}) {
    static_assert(PF == 1 || PF == 2, "prefetch depth");
    using acc_t = typename Mma<T>::acc_t;
    constexpr bool RT = LOADS == Loads::RuntimeLayout || LOADS == Loads::RuntimeGuarded;
    constexpr bool BUF = LOADS == Loads::Buffer || LOADS == Loads::RuntimeLayout;
    using Loader_A = typename std::conditional<RT, SlabLoaderRt<T, TL, TL::BM, TL::NVA, BUF>,
                                               SlabLoader<T, TL, TL::BM, A_K, TL::NVA, BUF>>::type;
    using Loader_B = typename std::conditional<RT, SlabLoaderRt<T, TL, TL::BN, TL::NVB, BUF>,
                                               SlabLoader<T, TL, TL::BN, B_K, TL::NVB, BUF>>::type;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave % TL::WGM, wn = wave / TL::WGM;
    const int wm0 = wm * TL::WM, wn0 = wn * TL::WN;

    acc_t acc[TL::TM][TL::TN];
#pragma unroll
    for (int i = 0; i < TL::TM; ++i)
#pragma unroll
        for (int j = 0; j < TL::TN; ++j) acc[i][j] = acc_t{};

    const int nk = (int)((p.k + TL::BK - 1) / TL::BK);
    const int klast = (int)(p.k - (int64_t)(nk - 1) * TL::BK);   // the last slab's extent
    auto kext = [&](int s) { return s + 1 == nk ? klast : TL::BK; };
    Loader_A al;
    Loader_B bl;
    al.init(p.a, p.m, p.k, p.lda, RT ? p.a_k : p.vec_a, m0, tid);
    bl.init(p.b, p.n, p.k, p.ldb, RT ? p.b_k : p.vec_b, n0, tid);

    // k == 0 (a batch problem with k == 0 or alpha == 0) touches neither A
    // nor B.
    if constexpr (PF == 1) {
        // One slab in flight. The loop runs over pairs of slabs, one per LDS
        // stage, each step one basic block: load the next slab, multiply this
        // one, store the next, barrier. The last slab is multiplied after it.
        auto step = [&](auto stage, int s) {
            constexpr int B = decltype(stage)::value;
            T* cur = smem + B * TL::STAGE;
            T* nxt = smem + (1 - B) * TL::STAGE;
            al.load(s + 1, tid);
            bl.load(s + 1, tid);
            mma_slab<T, TL>(cur, cur + TL::A_ELEMS, acc, wm0, wn0, lane);
            al.store(nxt, kext(s + 1), tid);
            bl.store(nxt + TL::A_ELEMS, kext(s + 1), tid);
            __syncthreads();
        };
        using Even = std::integral_constant<int, 0>;
        using Odd = std::integral_constant<int, 1>;
        if (nk > 0) {
            al.load(0, tid);
            bl.load(0, tid);
            al.store(smem, kext(0), tid);
            bl.store(smem + TL::A_ELEMS, kext(0), tid);
        }
        __syncthreads();
        int s = 0;
        for (; s + 2 < nk; s += 2) {
            step(Even{}, s);
            step(Odd{}, s + 1);
        }
        if (s + 1 < nk) {
            step(Even{}, s);
            ++s;
        }
        if constexpr (C_PF) prefetch_c<T, TL>(p, m0, n0, sink);
        if (nk > 0) {
            const T* cur = smem + (s & 1) * TL::STAGE;
            mma_slab<T, TL>(cur, cur + TL::A_ELEMS, acc, wm0, wn0, lane);
        }
        if constexpr (LDS_EPI) __syncthreads();   // the epilogue reuses the stages
    } else {
        // Two register buffers. At step s, buffer (s & 1) has already been
        // written to LDS and now receives slab s + 2; buffer ((s + 1) & 1)
        // holds slab s + 1 and is written to the other LDS stage after the
        // multiply. The loop runs over pairs of slabs so that each buffer is a
        // fixed set of registers; one loader walks the slabs and its loaded
        // registers change places with the second buffer's.
        typename Mma<T>::vec_t ra[TL::NVA], rb[TL::NVB];   // odd slabs
        auto swap_in = [&](auto& l, auto& other, auto&& f) {
            constexpr int N = sizeof(other) / sizeof(other[0]);
#pragma unroll
            for (int q = 0; q < N; ++q) { auto t = l.r[q]; l.r[q] = other[q]; other[q] = t; }
            f();
#pragma unroll
            for (int q = 0; q < N; ++q) { auto t = l.r[q]; l.r[q] = other[q]; other[q] = t; }
        };
        auto load = [&](auto buf, int s) {
            if constexpr (decltype(buf)::value == 0) { al.load(s, tid); bl.load(s, tid); }
            else {
                swap_in(al, ra, [&] { al.load(s, tid); });
                swap_in(bl, rb, [&] { bl.load(s, tid); });
            }
        };
        auto store = [&](auto buf, T* S, int s) {
            if constexpr (decltype(buf)::value == 0) {
                al.store(S, kext(s), tid);
                bl.store(S + TL::A_ELEMS, kext(s), tid);
            } else {
                swap_in(al, ra, [&] { al.store(S, kext(s), tid); });
                swap_in(bl, rb, [&] { bl.store(S + TL::A_ELEMS, kext(s), tid); });
            }
        };
        using Even = std::integral_constant<int, 0>;
        using Odd = std::integral_constant<int, 1>;
        if (nk > 0) {
            load(Even{}, 0);
            if (nk > 1) load(Odd{}, 1);
            store(Even{}, smem, 0);
        }
        __syncthreads();
        auto multiply = [&](auto stage) {
            const T* cur = smem + decltype(stage)::value * TL::STAGE;
            mma_slab<T, TL>(cur, cur + TL::A_ELEMS, acc, wm0, wn0, lane);
        };
        auto stage_next = [&](auto buf, int s) {   // slab s + 1 to the other stage
            constexpr int B = decltype(buf)::value;
            store(std::integral_constant<int, 1 - B>{}, smem + (1 - B) * TL::STAGE, s + 1);
            __syncthreads();
        };
        auto step = [&](auto buf, int s) {         // slab s, with s + 2 < nk
            load(buf, s + 2);
            multiply(buf);
            stage_next(buf, s);
        };
        int s = 0;
        for (; s + 3 < nk; s += 2) {
            step(Even{}, s);
            step(Odd{}, s + 1);
        }
        if (nk - s == 3) {
            step(Even{}, s);
            multiply(Odd{});
            stage_next(Odd{}, s + 1);
            multiply(Even{});
        } else if (nk - s == 2) {
            multiply(Even{});
            stage_next(Even{}, s);
            multiply(Odd{});
        } else if (nk - s == 1) {
            multiply(Even{});
        }
        if constexpr (LDS_EPI) __syncthreads();
    }

    if constexpr (MASK)
        store_tile_masked<T, TL>(p, acc, m0 + wm0, n0 + wn0, lane, cm);
    else if constexpr (LDS_EPI)
        store_tile_lds<T, TL>(p, acc, m0, n0, wm0, wn0, smem);
    else if (p.vec_c && m0 + TL::BM <= p.m && n0 + TL::BN <= p.n)
        store_tile<T, TL, true>(p, acc, m0 + wm0, n0 + wn0, lane);
    else
        store_tile<T, TL, false>(p, acc, m0 + wm0, n0 + wn0, lane);
}

// Whether a tile of the plain kernels writes C through LDS: when a lane's TM
// rows are not whole 16-byte vectors (FP32 waves of 32 rows), so that writing
// from the accumulators would go element by element, and the C tile fits the
// stages. FP32 8192 x 8192 x 256 on the 64 x 64 tile takes 298 us in place of
// 376, on 128 x 64 with eight waves 294 in place of 391; 3001 x 2999 x 333 on
// 64 x 64 64 in place of 81. Vectors from the accumulators are as fast as
// through LDS (128 x 64 with four waves: 308 and 311 us), and so are the
// one-row waves of the 32 x 32 tile (389 and 390 us), which keep the shorter
// path.
template <class TL> constexpr bool lds_epilogue() {
    return TL::TM > 1 && TL::TM % TL::V != 0 && TL::BN * (TL::BM + TL::V) <= 2 * TL::STAGE;
}

// LDS_EPI: write C through store_tile_lds instead of straight from the
// accumulators. C_PF: prefetch the C tile into L2 one slab before the epilogue
// (one-slab prefetch depth only), through `sink` (NT ints of LDS nobody reads). MASK: write only the stored region `cm` of
// a structured C (store_tile_masked).
template <typename T, class TL, bool A_K, bool B_K, Loads LOADS, int PF = 1, bool LDS_EPI = false,
          bool C_PF = false, bool MASK = false>
__device__ inline void gemm_tile(const TileProblem<T>& p, int64_t tm, int64_t tn, T* smem,
                                 int* sink = nullptr, CMask cm = CMask{}) {
    static_assert(!C_PF || PF == 1, "C prefetch is placed for one slab in flight");
    static_assert(!MASK || !LDS_EPI, "masked stores go straight from the accumulators");
    const int64_t m0 = tm * TL::BM, n0 = tn * TL::BN;
    gemm_tile_impl<T, TL, A_K, B_K, LOADS, PF, LDS_EPI, C_PF, MASK>(p, m0, n0, smem, sink, cm);
}

} // namespace dev
} // namespace blis_amd
