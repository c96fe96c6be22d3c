// gemm.hip — gfx950 GEMM launch planner and kernels.
//
// Host side of the BLIS five-loop GEMM (frame/3/gemm/bli_gemm_cntl.c:75-565,
// sandbox/gemmlike/bls_gemm_bp_var1.c:37-318): it normalises operand
// storage, picks a tile configuration (the analogue of BLIS's MC/NC/KC/MR/NR
// blocksizes, config/zen3/bli_cntx_init_zen3.c:204-220) and launches one
// workgroup per output tile. The device side lives in gemm_tile.hpp.
//
// Storage normalisation follows bli_gemm_cntl_init's operation transpose
// (bli_gemm_cntl.c:104-161): when C is row-stored the problem is recast as
// C^T := B^T A^T so that the kernel always writes column-stored C. Operands
// with neither unit row nor unit column stride are first packed into a
// contiguous column-major copy, as packm does for general-stride inputs
// (ref_kernels/1m/bli_packm_cxk_ref.c:78-147).
#include "gemm_plan.hpp"

#include <algorithm>

namespace blis_amd {

using namespace dev;

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// One tile per workgroup. With gridDim.y > 1 each blockIdx.y is a k partition
// of a split-k product: partition z covers k in [z*kchunk, min(k,
// (z+1)*kchunk)) and stores alpha * A_z * B_z, without reading anything
// there first, into its own m x n column-major slice of `parts` (ld = m).
// splitk_reduce_kernel then forms C.
template <typename T, class TL, bool A_K, bool B_K, bool BUF>
__global__ __launch_bounds__(TL::NT)
__attribute__((amdgpu_waves_per_eu(TL::waves_per_eu(BUF)))) void gemm_kernel(TileProblem<T> p, GridInfo g,
                                                      int64_t kchunk, T* parts) {
    __shared__ T smem[2 * TL::STAGE];
    if (gridDim.y > 1) {
        const int64_t z = blockIdx.y, k0 = z * kchunk;
        p.a += A_K ? k0 : k0 * p.lda;
        p.b += B_K ? k0 : k0 * p.ldb;
        p.k = min(kchunk, p.k - k0);
        p.c = parts + z * p.m * p.n;
        p.c_si = 1;
        p.c_sj = p.m;
        p.vec_c = 1;
        p.beta = T(0);
    }
    int tm, tn;
    tile_coords(blockIdx.x, gridDim.x, g, tm, tn);
    gemm_tile<T, TL, A_K, B_K, BUF ? Loads::Buffer : Loads::Guarded, 1, lds_epilogue<TL>()>(
        p, tm, tn, smem);
}

// count products at fixed element strides, one per blockIdx.y:
// C_z := beta*C_z + alpha*A_z*B_z with A_z = A + z*sa, B_z = B + z*sb,
// C_z = C + z*sc.
template <typename T, class TL, bool A_K, bool B_K, bool BUF>
__global__ __launch_bounds__(TL::NT)
__attribute__((amdgpu_waves_per_eu(TL::waves_per_eu(BUF)))) void gemm_strided_kernel(TileProblem<T> p, GridInfo g,
                                                              int64_t sa, int64_t sb, int64_t sc) {
    __shared__ T smem[2 * TL::STAGE];
    const int64_t z = blockIdx.y;
    p.a += z * sa;
    p.b += z * sb;
    p.c += z * sc;
    int tm, tn;
    tile_coords(blockIdx.x, gridDim.x, g, tm, tn);
    gemm_tile<T, TL, A_K, B_K, BUF ? Loads::Buffer : Loads::Guarded, 1, lds_epilogue<TL>()>(
        p, tm, tn, smem);
}

// C := beta*C + sum_z parts_z, partitions added in ascending z (a fixed
// order, so the result does not depend on scheduling). beta == 0 does not
// read C. Only the stored region `cm` of C is written. A thread takes one
// 16-byte vector of rows and keeps eight partitions' loads in flight: the sum
// is one pass over s*m*n partials, bound by the latency of its loads while
// the output is small.
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const T* __restrict__ parts, int s,
                                                            int64_t m, int64_t n, T* c,
                                                            int64_t c_si, int64_t c_sj, T beta,
                                                            CMask cm) {
    using vec_t = typename Mma<T>::vec_t;
    using uvec_t = typename Mma<T>::uvec_t;
    constexpr int V = Mma<T>::V;
    const uint32_t mv = (uint32_t)((m + V - 1) / V);
    const int64_t total = (int64_t)mv * n, slice = m * n;
    for (int64_t t = blockIdx.x * (int64_t)256 + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * 256) {
        const int64_t j = total >> 32 ? t / mv : (uint32_t)t / mv;
        const int64_t i = (t - j * mv) * V;
        // Rows [lo, hi) of the vector are stored.
        int64_t lo = i, hi = min(i + V, m);
        if (cm.uplo == 1) lo = max(lo, j - cm.doff);
        if (cm.uplo == 2) hi = min(hi, j - cm.doff + 1);
        if (lo >= hi) continue;
        const T* p = parts + i + j * m;
        vec_t acc;
        if (i + V <= m) {
            acc = *reinterpret_cast<const uvec_t*>(p);
            int z = 1;
            for (; z + 8 <= s; z += 8) {
                vec_t v[8];
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    v[u] = *reinterpret_cast<const uvec_t*>(p + (z + u) * slice);
#pragma unroll
                for (int u = 0; u < 8; ++u) acc += v[u];
            }
            for (; z < s; ++z) acc += *reinterpret_cast<const uvec_t*>(p + z * slice);
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e) {
                acc[e] = T(0);
                if (i + e < m) {
                    T x = p[e];
                    for (int z = 1; z < s; ++z) x += p[e + z * slice];
                    acc[e] = x;
                }
            }
        }
        T* dst = c + i * c_si + j * c_sj;
        if (c_si == 1 && lo == i && hi == i + V) {
            if (beta != T(0)) acc = beta * *reinterpret_cast<const uvec_t*>(dst) + acc;
            *reinterpret_cast<uvec_t*>(dst) = acc;
        } else {
#pragma unroll
            for (int e = 0; e < V; ++e)
                if (i + e >= lo && i + e < hi)
                    dst[e * c_si] = (beta == T(0)) ? acc[e] : beta * dst[e * c_si] + acc[e];
        }
    }
}

// C := beta*C for alpha == 0 or k == 0 (bli_l3_return_early_if_trivial,
// frame/3/bli_l3_util.c:41-65). beta == 0 stores zeros without reading C.
template <typename T>
__global__ void scalm_kernel(T* c, int64_t m, int64_t n, int64_t rs, int64_t cs, T beta) {
    const int64_t total = m * n;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = t % m, j = t / m;
        T* dst = c + i * rs + j * cs;
        *dst = (beta == T(0)) ? T(0) : beta * *dst;
    }
}

// dst (column-major m x n, ld = m) := src with arbitrary strides.
template <typename T>
__global__ void pack_kernel(const T* src, int64_t m, int64_t n, int64_t rs, int64_t cs, T* dst) {
    const int64_t total = m * n;
    for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
         t += (int64_t)gridDim.x * blockDim.x) {
        const int64_t i = t % m, j = t / m;
        dst[t] = src[i * rs + j * cs];
    }
}

// dst(r, c) = src(r, c) for an operand stored rows-contiguous along c,
// src(r, c) = src[c + r*lds], written column-wise: dst[r + c*ldd]. 64 x 64
// tiles through LDS, coalesced on both sides.
template <typename T>
__global__ __launch_bounds__(256) void transpose_kernel(const T* __restrict__ src, int64_t rows,
                                                        int64_t cols, int64_t lds,
                                                        T* __restrict__ dst, int64_t ldd) {
    __shared__ T tile[64][65];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t trows = (rows + 63) / 64, tcols = (cols + 63) / 64;
    for (int64_t t = blockIdx.x; t < trows * tcols; t += gridDim.x) {
        const int64_t r0 = (t % trows) * 64, c0 = (t / trows) * 64;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t r = r0 + ty + 4 * q, c = c0 + tx;
            if (r < rows && c < cols) tile[ty + 4 * q][tx] = src[c + r * lds];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t r = r0 + tx, c = c0 + ty + 4 * q;
            if (r < rows && c < cols) dst[r + c * ldd] = tile[tx][ty + 4 * q];
        }
        __syncthreads();
    }
}

static int grid_for(int64_t total) {
    int64_t g = (total + 255) / 256;
    if (g < 1) g = 1;
    if (g > 8192) g = 8192;
    return (int)g;
}

void scalm_run(Dt dt, int64_t m, int64_t n, double beta, View c, hipStream_t st) {
    if (m <= 0 || n <= 0) return;
    const int g = grid_for(m * n);
    if (dt == Dt::F64)
        hipLaunchKernelGGL(scalm_kernel<double>, dim3(g), dim3(256), 0, st,
                           (double*)c.ptr, m, n, c.rs, c.cs, beta);
    else
        hipLaunchKernelGGL(scalm_kernel<float>, dim3(g), dim3(256), 0, st,
                           (float*)c.ptr, m, n, c.rs, c.cs, (float)beta);
    HIP_CHECK(hipGetLastError());
}

void pack_run(Dt dt, const void* src, int64_t m, int64_t n, int64_t rs, int64_t cs,
              void* dst, hipStream_t st) {
    const int g = grid_for(m * n);
    if (dt == Dt::F64)
        hipLaunchKernelGGL(pack_kernel<double>, dim3(g), dim3(256), 0, st,
                           (const double*)src, m, n, rs, cs, (double*)dst);
    else
        hipLaunchKernelGGL(pack_kernel<float>, dim3(g), dim3(256), 0, st,
                           (const float*)src, m, n, rs, cs, (float*)dst);
    HIP_CHECK(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Launch plumbing
// ---------------------------------------------------------------------------

void splitk_reduce_run(Dt dt, const SplitK& sk, const Plan& pl, double beta, const CMask& cm,
                       hipStream_t st) {
    const int64_t V = dt == Dt::F64 ? Mma<double>::V : Mma<float>::V;
    const int g = grid_for((pl.m + V - 1) / V * pl.n);
    if (dt == Dt::F64)
        hipLaunchKernelGGL(splitk_reduce_kernel<double>, dim3(g), dim3(256), 0, st,
                           (const double*)sk.ws, sk.parts, pl.m, pl.n, (double*)pl.c, pl.c_si,
                           pl.c_sj, beta, cm);
    else
        hipLaunchKernelGGL(splitk_reduce_kernel<float>, dim3(g), dim3(256), 0, st,
                           (const float*)sk.ws, sk.parts, pl.m, pl.n, (float*)pl.c, pl.c_si,
                           pl.c_sj, (float)beta, cm);
    HIP_CHECK(hipGetLastError());
}

template <typename T, class TL, bool BUF>
static void launch_tl(const TileProblem<T>& p, bool a_k, bool b_k, GridInfo g, const SplitK& sk,
                      hipStream_t st) {
    g.grid_m = (int)((p.m + TL::BM - 1) / TL::BM);
    g.grid_n = (int)((p.n + TL::BN - 1) / TL::BN);
    if (g.group_m < 1) g.group_m = 1;
    const dim3 grid(g.grid_m * g.grid_n, sk.parts), block(TL::NT);
    T* ws = (T*)sk.ws;
    if (!a_k && !b_k)
        hipLaunchKernelGGL((gemm_kernel<T, TL, false, false, BUF>), grid, block, 0, st, p, g,
                           sk.kchunk, ws);
    else if (!a_k && b_k)
        hipLaunchKernelGGL((gemm_kernel<T, TL, false, true, BUF>), grid, block, 0, st, p, g,
                           sk.kchunk, ws);
    else if (a_k && !b_k)
        hipLaunchKernelGGL((gemm_kernel<T, TL, true, false, BUF>), grid, block, 0, st, p, g,
                           sk.kchunk, ws);
    else
        hipLaunchKernelGGL((gemm_kernel<T, TL, true, true, BUF>), grid, block, 0, st, p, g,
                           sk.kchunk, ws);
    HIP_CHECK(hipGetLastError());
}

// Every tile of the table reads its operands through buffer descriptors. A
// problem whose strides do not allow that runs on one of three tiles built
// without them, the one nearest in size: the tile never changes the result.
template <typename T>
static void launch_tile(int tile, const TileProblem<T>& p, bool a_k, bool b_k,
                        const GridInfo& g, const SplitK& sk, hipStream_t st) {
    const TileShape& ts = tile_shape(dt_of<T>(), tile);
    if (!buf_problem(p, a_k, b_k, ts.bm, ts.bn, ts.bk)) {
        constexpr int BK = std::is_same<T, double>::value ? 16 : 32;
        if (ts.bm * ts.bn > 64 * 64)
            launch_tl<T, TileCfg<T, 128, 64, BK, 32, 32>, false>(p, a_k, b_k, g, sk, st);
        else if (ts.bm == 64)
            launch_tl<T, TileCfg<T, 64, 64, BK, 32, 32>, false>(p, a_k, b_k, g, sk, st);
        else
            launch_tl<T, TileCfg<T, 32, 32, BK, 16, 16>, false>(p, a_k, b_k, g, sk, st);
        return;
    }
#define BLIS_AMD_CASE(idx, BM, BN, BK, WM, WN) \
    case idx: launch_tl<T, TileCfg<T, BM, BN, BK, WM, WN>, true>(p, a_k, b_k, g, sk, st); return;
    if constexpr (std::is_same<T, double>::value) {
        switch (tile) { BLIS_AMD_TILES_F64(BLIS_AMD_CASE) }
    } else {
        switch (tile) { BLIS_AMD_TILES_F32(BLIS_AMD_CASE) }
    }
#undef BLIS_AMD_CASE
    abort_with(BLIS_INVALID_UKR_ID, "gemm: tile index out of range");
}

static void transpose_run(Dt dt, const void* src, int64_t rows, int64_t cols, int64_t lds,
                          void* dst, int64_t ldd, hipStream_t st) {
    const int64_t tiles = ((rows + 63) / 64) * ((cols + 63) / 64);
    const unsigned g = (unsigned)std::max<int64_t>(1, std::min<int64_t>(tiles, 16384));
    if (dt == Dt::F64)
        hipLaunchKernelGGL(transpose_kernel<double>, dim3(g), dim3(256), 0, st, (const double*)src,
                           rows, cols, lds, (double*)dst, ldd);
    else
        hipLaunchKernelGGL(transpose_kernel<float>, dim3(g), dim3(256), 0, st, (const float*)src,
                           rows, cols, lds, (float*)dst, ldd);
    HIP_CHECK(hipGetLastError());
}

// The FP64 128x128 tile of sixteen 32x32 waves (tile 13) stages a
// k-contiguous operand into LDS by transposing scalar stores, which costs
// about 2% of a large product. On that tile it pays to transpose the operand
// once (rows x k, reused `reuse` times) and take the faster path; the
// arithmetic is the same either way. us as is and transposed: A and B
// k-contiguous at 8192^3 16192 / 16003 and 15770 / 15718, at 8192 x 8192 x
// 1024 2193 / 2149 and 2148 / 2115; at 4096^3, where the rule says no, 2056 /
// 2079 and 2002 / 2009. The default large FP64 tile (6, eight 64x32 waves)
// loses at most 1.8% by it, about what the transpose costs, and takes the
// operand as it comes.
static bool transpose_pays(Dt dt, int64_t reuse, int64_t rows, int64_t k) {
    const double es = (double)dt_size(dt);
    const double gemm_s = 2.0 * (double)reuse * rows * k / (dt == Dt::F64 ? 60e12 : 120e12);
    const double tr_s = 2.0 * rows * k * es / 4e12 + 8e-6;
    return 0.02 * gemm_s > tr_s;
}

// k-contiguous operands of a large product to the rows-contiguous path, one
// transpose each into workspace (operands already packed are left alone).
static void transpose_k_operands(Plan& p, Dt dt, Scratch& sc, hipStream_t st) {
    const size_t es = dt_size(dt);
    if (p.a_k && !p.a_packed && transpose_pays(dt, p.n, p.m, p.k)) {
        const int64_t ldw = (p.m + 3) / 4 * 4;
        void* w = sc.take((size_t)ldw * p.k * es, 0);
        transpose_run(dt, p.a, p.m, p.k, p.lda, w, ldw, st);
        p.a = w; p.lda = ldw; p.a_k = false;
    }
    if (p.b_k && !p.b_packed && transpose_pays(dt, p.m, p.n, p.k)) {
        const int64_t ldw = (p.n + 3) / 4 * 4;
        void* w = sc.take((size_t)ldw * p.k * es, 1);
        transpose_run(dt, p.b, p.n, p.k, p.ldb, w, ldw, st);
        p.b = w; p.ldb = ldw; p.b_k = false;
    }
}

int gemm_default_tile(Dt dt, int64_t m, int64_t n, int64_t k) {
    // Size heuristic from a sweep of the tile table on MI355X: the best
    // large-problem tiles are the ones with high wave occupancy (several
    // waves per SIMD hide LDS and barrier latency); small problems use small
    // tiles so that enough workgroups exist to fill the 256 CUs.
    // Large shapes re-measured with exhaustive autotuning at m, n in
    // 4096..16384 and k in 128..8192: FP64 128x128 tiles of eight 64x32
    // waves beat sixteen 32x32 waves by 4-8% (8192^3 NN 14.90 vs 15.72 ms);
    // FP32 short-k products prefer 128x64 tiles. Mid-size bands (256 to
    // 1023 tiles of 128x128) take the tile with the least total time over
    // the tuning database's shapes in that band.
    auto tiles = [&](int bm, int bn) { return ((m + bm - 1) / bm) * ((n + bn - 1) / bn); };
    if (dt == Dt::F64) {
        if (tiles(128, 128) >= 1024) return 6;   // 128x128 (BK 16), 8 waves of 64x32
        if (tiles(128, 128) >= 256) return 10;   // 64x128 (BK 16), 8 waves of 32x32
        if (tiles(64, 64) >= 512) return 3;      // 64x64 (BK 16), 4 waves of 32x32
        return 4;                                // 32x32 (BK 16), 4 waves of 16x16
    }
    if (k <= 256 && tiles(128, 64) >= 512) return 1;   // 128x64 (BK 32), 4 waves of 64x32
    if (tiles(256, 128) >= 512) return 12;       // 256x128 (BK 16), 8 waves of 64x64
    if (tiles(128, 128) >= 512) return 9;        // 128x64 (BK 32), 8 waves of 32x32
    if (tiles(128, 128) >= 256) return 10;       // 64x128 (BK 32), 8 waves of 32x32
    if (tiles(64, 64) >= 512) return 3;
    return 4;
}

// gemm_choose_split for a call on stream st. A captured product takes one pass
// unless that is many times slower (m, n <= k/4 and k >= 2048): the graph would
// keep its partitions for as long as the process lives.
SplitChoice split_on_stream(Dt dt, int64_t m, int64_t n, int64_t k, bool masked, hipStream_t st) {
    const SplitChoice c = gemm_choose_split(dt, m, n, k, masked);
    if (c.split <= 1 || (!masked && k >= 2048 && 4 * std::max(m, n) <= k)) return c;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    HIP_CHECK(hipStreamIsCapturing(st, &cap));
    return cap == hipStreamCaptureStatusNone ? c : gemm_choose_split(dt, m, n, k, masked, 1);
}

// Process-wide override used when a caller passes no configuration
// (set through bli_amd_gemm_set_config; tile -1 restores the heuristic).
static GemmConfig g_override;

// Split-k launch parameters for `split` requested partitions of whole
// 64-deep k blocks (every tile's BK divides 64, so the partition, and with
// it the rounding, is the same for every tile).
SplitK split_params(int64_t k, int split) {
    SplitK sk;
    if (split > 1) {
        const int64_t blocks = (k + 63) / 64;
        const int64_t want = std::min(split, 64);
        sk.kchunk = (blocks + want - 1) / want * 64;
        sk.parts = (int)((k + sk.kchunk - 1) / sk.kchunk);
    }
    return sk;
}

// Launch a normalised, packed plan with configuration cfg: the tile kernel,
// and for split-k the partition products into scratch and one reduction.
static void launch_plan(Dt dt, Plan& pl, const GemmConfig& cfg, double alpha, double beta,
                        Scratch& sc, hipStream_t st) {
    GridInfo g{};
    g.group_m = cfg.group_m;
    g.xcd_remap = cfg.xcd_remap;
    int tile = cfg.tile >= 0 ? cfg.tile : gemm_default_tile(dt, pl.m, pl.n, pl.k);
    if (tile < 0 || tile >= tile_count(dt)) abort_with(BLIS_INVALID_UKR_ID, "gemm: bad tile");
    // Split-k: each partition a full product into its own m x n slice of
    // scratch, then one reduction into C.
    SplitK sk = split_params(pl.k, cfg.split_k);
    if (sk.parts > 1) {
        const size_t bytes = (size_t)sk.parts * pl.m * pl.n * dt_size(dt);
        sk.ws = sc.base ? sc.take(bytes, 17) : stream_scratch(bytes, st);
        if (sk.ws == nullptr) {     // no memory for the slices
            sk = SplitK{};
            tile = gemm_default_tile(dt, pl.m, pl.n, pl.k);
        }
    }
    if (dt == Dt::F64 && tile == 13) transpose_k_operands(pl, dt, sc, st);
    if (gemm_sup_deep_k(tile, sk.parts, pl.k) && gemm_sup_run(dt, pl, alpha, beta, st)) return;
    if (dt == Dt::F64) {
        launch_tile<double>(tile, make_problem<double>(pl, alpha, beta), pl.a_k, pl.b_k, g, sk, st);
    } else {
        launch_tile<float>(tile, make_problem<float>(pl, alpha, beta), pl.a_k, pl.b_k, g, sk, st);
    }
    if (sk.parts > 1) splitk_reduce_run(dt, sk, pl, beta, CMask{}, st);
}

void gemm_run(const GemmDesc& d, const GemmConfig* cfg, hipStream_t st) {
    if (d.m <= 0 || d.n <= 0) return;
    if (cfg == nullptr) cfg = &g_override;
    if (d.k <= 0 || d.alpha == 0.0) {
        scalm_run(d.dt, d.m, d.n, d.beta, d.c, st);
        return;
    }
    Plan pl = layout(d);
    // Small problems with no configuration given take the sup path, ahead
    // of the heuristic and the learned selector (exhaustive selection times
    // the table's tiles instead).
    if (cfg == &g_override && g_override.tile < 0 && g_override.split_k <= 1 &&
        !pl.a_packed && !pl.b_packed && gemm_sup_applies(pl.m, pl.n, pl.k) &&
        selector_mode() != SELECT_EXHAUSTIVE && gemm_sup_run(d.dt, pl, d.alpha, d.beta, st))
        return;
    GemmConfig picked;
    if (cfg == &g_override && g_override.tile < 0) {
        // No configuration given: the selector (heuristic, learned or
        // exhaustive) picks one from the normalised shape, before anything
        // is packed into scratch.
        const bool va = vec_ok(pl.a, pl.a_packed, pl.lda, d.dt);
        const bool vb = vec_ok(pl.b, pl.b_packed, pl.ldb, d.dt);
        const bool vc = aligned16(pl.c) && pl.c_si == 1 && pl.c_sj % (d.dt == Dt::F64 ? 2 : 4) == 0;
        picked = config_of(selector_pick(d.dt, pl.m, pl.n, pl.k, pl.a_k, pl.b_k, va, vb, vc));
        // Nor has the network seen C without a unit stride, which every tile
        // writes element by element. While that is most of the time, 32 x 32
        // tiles are the fastest: within 0.4% of the best over 80 shapes of
        // k <= 128, the network's picks 4.1% off and at worst 1.63 times. (129 to
        // 512: 2.3%, the network's 1.3%.)
        if (pl.c_si != 1 && pl.k <= 128 && selector_mode() == SELECT_LEARNED) picked.tile = 4;
        if (g_override.split_k > 1) {
            picked.split_k = g_override.split_k;
        } else {
            // A product split by the shape rule takes the rule's tile, unless
            // the selector timed every configuration itself.
            const SplitChoice sc = split_on_stream(d.dt, pl.m, pl.n, pl.k, false, st);
            picked.split_k = sc.split;
            if (sc.split > 1 && selector_mode() != SELECT_EXHAUSTIVE) picked.tile = sc.tile;
        }
        cfg = &picked;
    }
    Scratch sc;
    pack_operands(pl, d.dt, sc, st);
    launch_plan(d.dt, pl, *cfg, d.alpha, d.beta, sc, st);
}

template <typename T, class TL, bool BUF>
static void launch_strided_tl(const TileProblem<T>& p, bool a_k, bool b_k, const GridInfo& g,
                              int count, int64_t sa, int64_t sb, int64_t sc, hipStream_t st) {
    const dim3 grid(g.grid_m * g.grid_n, count), block(TL::NT);
    if (!a_k && !b_k)
        hipLaunchKernelGGL((gemm_strided_kernel<T, TL, false, false, BUF>), grid, block, 0, st, p,
                           g, sa, sb, sc);
    else if (!a_k && b_k)
        hipLaunchKernelGGL((gemm_strided_kernel<T, TL, false, true, BUF>), grid, block, 0, st, p,
                           g, sa, sb, sc);
    else if (a_k && !b_k)
        hipLaunchKernelGGL((gemm_strided_kernel<T, TL, true, false, BUF>), grid, block, 0, st, p,
                           g, sa, sb, sc);
    else
        hipLaunchKernelGGL((gemm_strided_kernel<T, TL, true, true, BUF>), grid, block, 0, st, p, g,
                           sa, sb, sc);
    HIP_CHECK(hipGetLastError());
}

// The 32x32 tile (tile 4 of both tables): these batches are of small
// products, several hundred tiles in all.
template <typename T>
static void launch_strided(const Plan& pl, double alpha, double beta, int count, int64_t sa,
                           int64_t sb, int64_t sc, hipStream_t st) {
    constexpr int V = Mma<T>::V;
    using TL = TileCfg<T, 32, 32, std::is_same<T, double>::value ? 16 : 32, 16, 16>;
    GridInfo g{};
    g.group_m = 8;
    g.xcd_remap = 1;
    g.grid_m = (int)((pl.m + TL::BM - 1) / TL::BM);
    g.grid_n = (int)((pl.n + TL::BN - 1) / TL::BN);
    TileProblem<T> p = make_problem<T>(pl, alpha, beta);
    p.vec_a = p.vec_a && sa % V == 0;
    p.vec_b = p.vec_b && sb % V == 0;
    if (buf_problem(p, pl.a_k, pl.b_k, TL::BM, TL::BN, TL::BK))
        launch_strided_tl<T, TL, true>(p, pl.a_k, pl.b_k, g, count, sa, sb, sc, st);
    else
        launch_strided_tl<T, TL, false>(p, pl.a_k, pl.b_k, g, count, sa, sb, sc, st);
}

void gemm_strided_run(const GemmDesc& d, int count, int64_t sa, int64_t sb, int64_t sc,
                      hipStream_t st) {
    if (d.m <= 0 || d.n <= 0 || count <= 0) return;
    if (d.c.rs != 1 || d.k <= 0 || d.alpha == 0.0)
        abort_with(BLIS_INVALID_UKR_ID, "gemm strided: C must be column-stored, k > 0, alpha != 0");
    Plan pl = layout(d);
    if (pl.a_packed || pl.b_packed)
        abort_with(BLIS_INVALID_UKR_ID, "gemm strided: operands need a unit stride");
    if (d.dt == Dt::F64) launch_strided<double>(pl, d.alpha, d.beta, count, sa, sb, sc, st);
    else launch_strided<float>(pl, d.alpha, d.beta, count, sa, sb, sc, st);
}

// ---------------------------------------------------------------------------
// GEMM without allocation (bli_amd_gemm_noalloc)
// ---------------------------------------------------------------------------
//
// The device memory a GEMM may take beyond its operands (packed copies of
// general-stride operands, split-k partitions) comes from one fixed array
// per GPU instead of the workspace arena. In host code `scratch` only
// names the array; its device address on the current GPU comes from
// hipGetSymbolAddress, taken once per device and kept in g_scratch_ptr.

constexpr size_t NOALLOC_SCRATCH_BYTES = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int NOALLOC_MAX_DEVICES = 64;
static void* g_scratch_ptr[NOALLOC_MAX_DEVICES] = {};
static std::mutex g_scratch_mutex;

// Device address of `scratch` on the current GPU (nullptr on failure).
static void* scratch_address(int dev) {
    if (dev < 0 || dev >= NOALLOC_MAX_DEVICES) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess) {
            (void)hipGetLastError();
            return nullptr;
        }
        g_scratch_ptr[dev] = p;
    }
    return g_scratch_ptr[dev];
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

} // namespace blis_amd

extern "C" __attribute__((visibility("default")))
void bli_amd_gemm_set_config(int tile, int group_m, int xcd_remap, int split_k) {
    blis_amd::init_once();
    std::lock_guard<std::mutex> lock(blis_amd::api_mutex());
    blis_amd::g_override.tile = tile;
    blis_amd::g_override.group_m = group_m > 0 ? group_m : 8;
    blis_amd::g_override.xcd_remap = xcd_remap;
    blis_amd::g_override.split_k = split_k > 0 ? split_k : 1;
}

extern "C" __attribute__((visibility("default")))
int bli_amd_gemm_tile_count(int is_double) {
    return blis_amd::tile_count(is_double ? blis_amd::Dt::F64 : blis_amd::Dt::F32);
}

extern "C" __attribute__((visibility("default")))
int bli_amd_gemm_default_tile(int is_double, long long m, long long n, long long k) {
    return blis_amd::gemm_default_tile(is_double ? blis_amd::Dt::F64 : blis_amd::Dt::F32, m, n, k);
}

// C := beta*C + alpha*op(A)*op(B) for FP32/FP64 device operands, with no
// device allocation: scratch comes from the library's fixed per-GPU array
// (64 MiB). The kernels and their configuration are those of bli_?gemm with
// the default (heuristic) selector, so the results are the same bits.
extern "C" __attribute__((visibility("default")))
int bli_amd_gemm_noalloc(num_t dt, trans_t transa, trans_t transb, dim_t m, dim_t n, dim_t k,
                         const void* alpha, const void* a, inc_t rs_a, inc_t cs_a,
                         const void* b, inc_t rs_b, inc_t cs_b, const void* beta, void* c,
                         inc_t rs_c, inc_t cs_c, void* stream) {
    using namespace blis_amd;
    if (dt != BLIS_FLOAT && dt != BLIS_DOUBLE) return BLIS_INVALID_DATATYPE;
    auto valid = [](trans_t t) {
        return t == BLIS_NO_TRANSPOSE || t == BLIS_TRANSPOSE || t == BLIS_CONJ_NO_TRANSPOSE ||
               t == BLIS_CONJ_TRANSPOSE;
    };
    if (!valid(transa) || !valid(transb)) return BLIS_INVALID_TRANS;
    if (m < 0 || n < 0 || k < 0) return BLIS_NEGATIVE_DIMENSION;
    if (alpha == nullptr || beta == nullptr) return BLIS_NULL_POINTER;
    if (m == 0 || n == 0) return BLIS_SUCCESS;
    const Dt d = dt == BLIS_DOUBLE ? Dt::F64 : Dt::F32;
    const double al = d == Dt::F64 ? *(const double*)alpha : (double)*(const float*)alpha;
    const double be = d == Dt::F64 ? *(const double*)beta : (double)*(const float*)beta;
    const bool touch_ab = k > 0 && al != 0.0;
    // Operands must already be in device memory (host staging allocates).
    if (c == nullptr || !is_device_pointer(c)) return BLIS_FAILURE;
    if (touch_ab && (a == nullptr || b == nullptr || !is_device_pointer(a) ||
                     !is_device_pointer(b)))
        return BLIS_FAILURE;
    const bool ta = (unsigned)transa & BLIS_TRANS_BIT, tb = (unsigned)transb & BLIS_TRANS_BIT;
    GemmDesc g;
    g.dt = d; g.m = m; g.n = n; g.k = k;
    g.a = { const_cast<void*>(a), ta ? cs_a : rs_a, ta ? rs_a : cs_a };
    g.b = { const_cast<void*>(b), tb ? cs_b : rs_b, tb ? rs_b : cs_b };
    g.c = { c, rs_c, cs_c };
    g.alpha = al; g.beta = be;
    hipStream_t st = (hipStream_t)stream;
    if (!touch_ab) {
        scalm_run(d, m, n, be, g.c, st);
        return BLIS_SUCCESS;
    }
    Plan pl = layout(g);
    GemmConfig cfg;
    const SplitChoice choice = gemm_choose_split(d, pl.m, pl.n, pl.k, false);
    cfg.split_k = choice.split;
    cfg.tile = choice.split > 1 ? choice.tile : gemm_default_tile(d, pl.m, pl.n, pl.k);
    // Scratch this call needs, carved as Scratch::take does (256-byte
    // aligned pieces): packed general-stride operands and split-k slices.
    const size_t es = dt_size(d);
    size_t need = 0;
    if (pl.a_packed) need += align256((size_t)pl.m * pl.k * es);
    if (pl.b_packed) need += align256((size_t)pl.k * pl.n * es);
    const SplitK sk = split_params(pl.k, cfg.split_k);
    if (sk.parts > 1) {
        const size_t slices = align256((size_t)sk.parts * pl.m * pl.n * es);
        if (need + slices > NOALLOC_SCRATCH_BYTES) {
            // No room for the partitions beside the packed operands: one pass.
            cfg.split_k = 1;
            cfg.tile = gemm_default_tile(d, pl.m, pl.n, pl.k);
        } else {
            need += slices;
        }
    }
    if (need > NOALLOC_SCRATCH_BYTES) return BLIS_INSUFFICIENT_STACK_BUF_SIZE;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return BLIS_FAILURE;
    Scratch sc;
    sc.base = (char*)scratch_address(dev);
    sc.cap = NOALLOC_SCRATCH_BYTES;
    if (sc.base == nullptr) return BLIS_FAILURE;
    pack_operands(pl, d, sc, st);
    launch_plan(d, pl, cfg, al, be, sc, st);
    return BLIS_SUCCESS;
}
