// trsm.hip — triangular solve B := alpha * inv(op(A)) * B (left) or
// B := alpha * B * inv(op(A)) (right) on gfx950.
//
// Reference structure (paths relative to the BLIS tree):
//   * right side is solved as a left-side problem on transposed operands
//     (frame/3/bli_l3_oapi_ex.c:753-758);
//   * blocked algorithm: diagonal blocks are solved by a triangular kernel and
//     the rest of B is updated by GEMM (frame/3/trsm/bli_trsm_blk_var1.c:37-189,
//     frame/3/trsm/bli_trsm_ll_ker_var2.c:240-335);
//   * the diagonal kernel multiplies by the reciprocal of each diagonal
//     element, which packing stores in place of the element
//     (BLIS_ENABLE_TRSM_PREINVERSION; ref_kernels/1m/bli_packm_cxc_diag_ref.c:
//     99-107, ref_kernels/3/bli_trsm_ref.c:42-231).
//
// GPU formulation. Every case is first reduced to a left-side solve
// L_eff * X = alpha * B' with L_eff lower or upper, by folding op(A) and the
// side into strides. The solve recurses on halves: solve the leading half,
// update the trailing half with one GEMM (the bulk of the m^2 n flops, on the
// MFMA GEMM path), solve the trailing half. Leaves of at most 512 rows are
// solved by substitution in one launch (trsm_slab_kernel); when the triangle
// is diagonally dominant and large, whole 512-row blocks are solved by a
// product with their inverse instead.
#include "internal.hpp"
#include "gemm_tile.hpp"

namespace blis_amd {

namespace detail_trsm {

constexpr int64_t LB = 64;      // rows of the blocks inverted by substitution
constexpr int WPB = 4;          // waves per workgroup of that kernel
constexpr int NB = 256;         // rows of a block of the dominance check
constexpr int64_t PB = 512;     // rows of a block solved by product
constexpr int64_t SLAB = 512;   // most rows of a leaf solved by substitution
// Right-hand sides and rows from which the inverted-diagonal path pays: it
// spends about 75 us on checking and inverting, lost when a block fails the
// check. FP64, n = 1024, by substitution and by product (us): 1024 rows 149
// and 120, 2048 rows 330 and 222, 4096 rows 834 and 559.
constexpr int64_t TRSM_INV_MIN_N = 512;
constexpr int64_t TRSM_INV_MIN_ROWS = 3 * PB;
// Columns per wave when inverting the 64-row blocks: each wave reads the
// triangle's rows once for all of its columns.
constexpr int INV_CPW = 2;

__device__ inline double lane_bcast(double v, int l) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffll), l);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ inline float lane_bcast(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Inverses of 64-row diagonal blocks, one per blockIdx.y: block y is the
// triangle at a + y*a_step (only the stored part is read), its inverse goes
// to b + y*b_step with columns bcs apart. A wave owns CPW columns, row l of
// them in lane l, and substitutes into columns of the identity: the solved
// row i, scaled by the reciprocal of the diagonal, is read from lane i and
// every other lane subtracts its L element times it. The block also zeroes
// its columns of the 512-row block on the far side of the diagonal.
template <typename T, bool LOWER, int CPW>
__global__ __launch_bounds__(64 * WPB) void trsm_inverse_kernel(const T* __restrict__ a,
                                                                int64_t ars, int64_t acs,
                                                                T* __restrict__ b, int64_t bcs,
                                                                int unit_diag, int64_t a_step,
                                                                int64_t b_step) {
    a += (int64_t)blockIdx.y * a_step;
    b += (int64_t)blockIdx.y * b_step;
    const int lane = threadIdx.x & 63;
    const int col0 = (blockIdx.x * WPB + (threadIdx.x >> 6)) * CPW;
    T x[CPW], l[LB];
#pragma unroll
    for (int c = 0; c < CPW; ++c) x[c] = lane == col0 + c ? T(1) : T(0);
#pragma unroll
    for (int i = 0; i < (int)LB; ++i) {
        const bool stored = LOWER ? i < lane : i > lane;
        l[i] = stored ? a[lane * ars + i * acs] : T(0);
    }
    const T inv = unit_diag ? T(1) : T(1) / a[lane * (ars + acs)];
#pragma unroll
    for (int s = 0; s < (int)LB; ++s) {
        const int i = LOWER ? s : (int)LB - 1 - s;
        const T inv_i = lane_bcast(inv, i);
#pragma unroll
        for (int c = 0; c < CPW; ++c) {
            const T xi = lane_bcast(x[c], i) * inv_i;
            // Rows solved earlier are left as they are (an Inf in xi must
            // not turn them into NaN through a zero of L).
            if (lane == i) x[c] = xi;
            else if (LOWER ? lane > i : lane < i) x[c] -= l[i] * xi;
        }
    }
#pragma unroll
    for (int c = 0; c < CPW; ++c) b[lane + (col0 + c) * bcs] = x[c];
    constexpr int GROUP = (int)(PB / LB);
    const int d = (int)(blockIdx.y % GROUP);
    const int z0 = LOWER ? -d * (int)LB : (int)LB;
    const int zn = LOWER ? d * (int)LB : (GROUP - 1 - d) * (int)LB;
    for (int r = lane; r < zn; r += 64)
#pragma unroll
        for (int c = 0; c < CPW; ++c) b[(z0 + r) + (col0 + c) * bcs] = T(0);
}

// Solve L X = alpha B for m <= 128 * SLOTS rows and the 16 columns of B that a
// workgroup of eight waves owns, by substitution. L(i, j) = a[i*ars + j*acs]
// is lower triangular (an upper one comes with reversed rows and columns,
// that is negative strides) and only its stored triangle is read;
// B(i, j) = b[i*brs + j*bcs], X(i, j) = x[i*xrs + j*xcs], which may be B.
//
// The rows are tiles of 16; wave w keeps the sums -L X of tiles w, w + 8, ... of
// its columns in MFMA accumulators for the whole solve, row 4g + r of a tile in
// register r of lane group g. (The FP64 accumulator holds D row 4r + g there,
// so its L operand carries the tile's rows in the order 0, 4, 8, 12, 1, ...)
// The sums start from zero and B joins a row's when the row is solved: it is
// often much larger than the products, and would set the size of every
// rounding (FP32 error of X against FP64 at 512 rows, dominant triangle:
// 3.6e-7 from B, 2.6e-7 from B in two leaves, 3.7e-8 so; 450 rows of a factor
// that is not dominant: 3.7e-7, 2.8e-7, 1.0e-7). A solved tile's registers then
// are, as they stand, the four k steps of an MFMA's B operand over columns
// 4g + r of L. Step q: every wave subtracts L(:, q-1)
// X(q-1) from its tiles below, four MFMAs each, the owner of tile q first,
// which then solves it while the others go on. The 16 x 16 diagonal block is
// solved four rows at a time, which one lane holds for its column: plain
// substitution inside the lane, each row scaled by the reciprocal of its
// diagonal element, then four MFMAs subtract those rows from the ones below.
// The chain of steps is the bound (1.8 us each in FP64, 1.3 in FP32, half of it
// the diagonal block), so what a step needs is fetched ahead: L two steps, the
// diagonal blocks before the first. 512 rows take 60 us (FP32 42) for 1024
// columns and 68 (45) for 4096, 256 rows 26 to 28 (18 to 19); a kernel that substitutes 64 rows at a time across
// a wave took 83 us (68) for 256 rows. Also measured: one column of the tile
// per lane with the block's elements as LDS broadcasts, 121 us for 512 rows;
// rows broadcast across lane groups, 81 us; tiles for 1024 rows in one launch,
// no faster than two leaves and an update.
template <typename T, int SLOTS>
__global__ __launch_bounds__(512) void trsm_slab_kernel(const T* __restrict__ a, int64_t ars,
                                                        int64_t acs, const T* b, int64_t brs,
                                                        int64_t bcs, T* xo, int64_t xrs,
                                                        int64_t xcs, int m, int64_t n, T alpha,
                                                        int unit_diag) {
    using acc_t = typename dev::Mma<T>::acc_t;
    __shared__ T xb[2][256];             // -X of the last two tiles, [register][lane]
    __shared__ T diag[8 * SLOTS][256];   // diagonal blocks, [column][row], reciprocal diagonal
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
    const int lr = sizeof(T) == 8 ? 4 * (c & 3) + (c >> 2) : c;   // L operand row of this lane
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int P = (m + 15) / 16;
    const int64_t col0 = (int64_t)blockIdx.x * 16;
    const int64_t colc = (col0 + c < n ? col0 + c : n - 1) * bcs;

    // Rows and columns past the edge are clamped on load and not stored; in
    // the last diagonal block they are rows of the identity.
    acc_t acc[SLOTS];
    const T* lp[SLOTS];
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
        const int t = 8 * j + w;
        acc[j] = acc_t{};
        lp[j] = a + min(t * 16 + lr, m - 1) * ars + 4 * g * acs;
    }
    T bt[4];                                       // B of the wave's next tile to solve
    auto load_b = [&](int t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) bt[r] = b[min(t * 16 + 4 * g + r, m - 1) * brs + colc];
    };
    load_b(w);
    T l[2][SLOTS][4];
    auto load_l = [&](auto buf, int p) {           // L(t, p) of the wave's tiles t > p
        const int64_t off = (int64_t)p * 16 * acs;
#pragma unroll
        for (int j = 0; j < SLOTS; ++j)
            if (8 * j + w > p && 8 * j + w < P)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    l[decltype(buf)::value][j][k] = lp[j][off + k * acs];
    };
    // The diagonal blocks, one wave each at a time: row c, columns 4e + g.
#pragma unroll 4
    for (int q = w; q < P; q += 8) {
        T v[4], own = T(1);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int dj = 4 * e + g, i = q * 16 + c;
            v[e] = T(0);
            if (i < m && (c > dj || (c == dj && !unit_diag)))
                v[e] = a[i * ars + (int64_t)(q * 16 + dj) * acs];
            own = c == dj && i < m && !unit_diag ? v[e] : own;
        }
        const T inv = T(1) / own;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            diag[q][(4 * e + g) * 16 + c] = c == 4 * e + g ? inv : v[e];
    }
    auto store_x = [&](int q) {                    // tile q of X, by one wave
        const T* src = xb[q & 1];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            // Lanes along X's unit stride.
            const int u = 4 * e + g, i = xcs == 1 ? u : c, j = xcs == 1 ? c : u;
            if (q * 16 + i < m && col0 + j < n)
                xo[(q * 16 + i) * xrs + (col0 + j) * xcs] = -src[(i & 3) * 64 + (i >> 2) * 16 + j];
        }
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    load_l(B0{}, 0);
    load_l(B1{}, 1);
    __syncthreads();

    auto step = [&](auto buf, int q) {
        constexpr int B = decltype(buf)::value;    // == q & 1
        T xf[4] = {};
        auto subtract = [&](acc_t& d, const T (&lt)[4]) {
#pragma unroll
            for (int k = 0; k < 4; ++k) d = dev::Mma<T>::mma(lt[k], xf[k], d);
        };
        if (q > 0) {
#pragma unroll
            for (int k = 0; k < 4; ++k) xf[k] = xb[1 - B][k * 64 + lane];
        }
        if (w == (q & 7)) {
            // The lane group's own 4 x 4 diagonal block, and the columns of
            // L below it as an A operand.
            const T* D = diag[q] + 4 * g * 17;
            const T i0 = D[0], i1 = D[17], i2 = D[34], i3 = D[51];
            const T l10 = D[1], l20 = D[2], l30 = D[3], l21 = D[18], l31 = D[19], l32 = D[35];
            T low[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) low[k] = lr >= 4 * g + 4 ? diag[q][(4 * g + k) * 16 + lr] : T(0);
            acc_t v = acc_t{};
#pragma unroll
            for (int j = 0; j < SLOTS; ++j)
                if (8 * j + w == q) {
                    if (q > 0) subtract(acc[j], l[1 - B][j]);
                    v = acc[j];
                }
            T x[4] = {};                           // -X, rows 4g + r
            auto rows = [&](auto sub) {            // rows 4s .. 4s + 3, held by lane group s
                constexpr int s = decltype(sub)::value;
                const T x0 = fma(alpha, bt[0], v[0]) * i0;
                const T x1 = fma(alpha, bt[1], v[1] - l10 * x0) * i1;
                const T x2 = fma(alpha, bt[2], v[2] - l20 * x0 - l21 * x1) * i2;
                const T x3 = fma(alpha, bt[3], v[3] - l30 * x0 - l31 * x1 - l32 * x2) * i3;
                // Zeros everywhere else, in both operands and in what is kept:
                // an Inf of these rows or of L must not reach a row through a
                // product that substitution does not form.
                const bool own = g == s;
                const T y[4] = { -x0, -x1, -x2, -x3 };
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    x[k] = own ? y[k] : x[k];
                    if constexpr (s < 3)
                        v = dev::Mma<T>::mma(own ? low[k] : T(0), own ? y[k] : T(0), v);
                }
            };
            rows(std::integral_constant<int, 0>{});
            rows(std::integral_constant<int, 1>{});
            rows(std::integral_constant<int, 2>{});
            rows(std::integral_constant<int, 3>{});
#pragma unroll
            for (int k = 0; k < 4; ++k) xb[B][k * 64 + lane] = x[k];
            if (q + 8 < P) load_b(q + 8);
        }
        if (q > 0) {
#pragma unroll
            for (int j = 0; j < SLOTS; ++j)
                if (8 * j + w > q && 8 * j + w < P) subtract(acc[j], l[1 - B][j]);
            if (w == ((q + 4) & 7)) store_x(q - 1);
        }
        if (q + 1 < P) {
            load_l(std::integral_constant<int, 1 - B>{}, q + 1);
        }
        dev::lds_barrier();
    };
#pragma unroll 1
    for (int q = 0; q < P; q += 2) {
        step(B0{}, q);
        if (q + 1 < P) step(B1{}, q + 1);
    }
    if (w == 0) store_x(P - 1);
}

// Which diagonal blocks may be solved by multiplying with their inverse.
// Block q (rows q*NB .. q*NB + nb - 1, one workgroup of NB threads, thread
// t on row q*NB + t) passes when every row is diagonally dominant by a
// factor of two within the block, |l_ii| > 2 * sum_{j != i} |l_ij|, and
// the diagonal magnitudes stay within a factor of 16 of each other. Then
// L = D (I + D^-1 N) with ||D^-1 N||_inf < 1/2, so ||inv(L)||_inf <=
// 2 / min|l_ii| and cond_inf(L) <= 3 * max|l_ii| / min|l_ii| <= 48: the
// product with the FP64 (FP32) inverse keeps the residual of substitution
// to within that factor.
template <typename T, bool LOWER>
__global__ __launch_bounds__(NB) void trsm_diag_check_kernel(const T* __restrict__ a, int64_t ars,
                                                            int64_t acs, int64_t m,
                                                            int unit_diag, int* __restrict__ ok) {
    __shared__ int bad;
    // Largest and smallest |l_ii| as IEEE bit patterns: for non-negative
    // doubles the unsigned order of the patterns is the numeric order, so
    // the extremes are exact whatever the diagonal's range.
    __shared__ unsigned long long dmax, dmin;
    const int t = threadIdx.x;
    const int64_t q0 = (int64_t)blockIdx.x * NB;
    const int64_t nb = (m - q0 < NB) ? m - q0 : NB;
    if (t == 0) { bad = 0; dmax = 0ull; dmin = ~0ull; }
    __syncthreads();
    if (t < nb) {
        const int64_t r = q0 + t;
        // Eight independent partial sums keep eight loads in flight.
        double part[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        const int64_t j0 = LOWER ? q0 : r + 1, j1 = LOWER ? r : q0 + nb;
        int64_t j = j0;
        for (; j + 8 <= j1; j += 8) {
#pragma unroll
            for (int u = 0; u < 8; ++u) part[u] += fabs((double)a[r * ars + (j + u) * acs]);
        }
        for (; j < j1; ++j) part[0] += fabs((double)a[r * ars + j * acs]);
        const double off = ((part[0] + part[1]) + (part[2] + part[3])) +
                           ((part[4] + part[5]) + (part[6] + part[7]));
        const double d = unit_diag ? 1.0 : fabs((double)a[r * ars + r * acs]);
        if (!(d > 2.0 * off) || !(d < 1.0e300)) atomicOr(&bad, 1);
        const unsigned long long bits = (unsigned long long)__double_as_longlong(d);
        atomicMax(&dmax, bits);
        atomicMin(&dmin, bits);
    }
    __syncthreads();
    if (t == 0) {
        const double hi = __longlong_as_double((long long)dmax);
        const double lo = __longlong_as_double((long long)dmin);
        ok[blockIdx.x] = (!bad && hi <= 16.0 * lo) ? 1 : 0;
    }
}

// dst(i, j) = src(i, j) for i < rows, j < cols, both general-strided, through
// 64 x 64 LDS tiles: reads run along i and writes along j, so a copy between
// column-major and row-major storage is coalesced on both sides.
template <typename T>
__global__ __launch_bounds__(256) void trsm_copy_kernel(const T* __restrict__ src, int64_t srs,
                                                        int64_t scs, T* __restrict__ dst,
                                                        int64_t drs, int64_t dcs, int64_t rows,
                                                        int64_t cols) {
    __shared__ T tile[64][65];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t ti = (rows + 63) / 64, tj = (cols + 63) / 64;
    for (int64_t t = blockIdx.x; t < ti * tj; t += gridDim.x) {
        const int64_t i0 = (t % ti) * 64, j0 = (t / ti) * 64;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t i = i0 + tx, j = j0 + ty + 4 * q;
            if (i < rows && j < cols) tile[tx][ty + 4 * q] = src[i * srs + j * scs];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t i = i0 + ty + 4 * q, j = j0 + tx;
            if (i < rows && j < cols) dst[i * drs + j * dcs] = tile[ty + 4 * q][tx];
        }
        __syncthreads();
    }
}

// The parts of a triangle's 512-row diagonal blocks off their 64-row diagonal
// blocks, into a column-major copy: element (i, j) goes to dst[i + j * PB], so
// the blocks along the diagonal are a constant stride apart. Only the stored side
// is read, lanes along the smaller stride.
template <typename T>
__global__ __launch_bounds__(256) void trsm_gather_kernel(const T* __restrict__ a, int64_t ars,
                                                          int64_t acs, T* __restrict__ dst,
                                                          int lower) {
    __shared__ T tile[64][65];
    int tj = blockIdx.x, ti = 1;          // tile (ti, tj) below the diagonal of 8 x 8
    while (tj >= ti) tj -= ti++;
    const int64_t b0 = (int64_t)blockIdx.y * PB;
    const int64_t r0 = b0 + (lower ? ti : tj) * 64, c0 = b0 + (lower ? tj : ti) * 64;
    const bool along = (ars < 0 ? -ars : ars) <= (acs < 0 ? -acs : acs);
    const int u = threadIdx.x & 63;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int v = (threadIdx.x >> 6) + 4 * q, i = along ? u : v, j = along ? v : u;
        tile[j][i] = a[(r0 + i) * ars + (c0 + j) * acs];
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const int v = (threadIdx.x >> 6) + 4 * q;
        dst[(r0 + u) + (c0 + v) * PB] = tile[v][u];
    }
}

struct Solve {
    Dt dt;
    bool lower;
    bool unit;
    View a;          // L_eff(i,j) = a.ptr[i*a.rs + j*a.cs]
    int64_t n;
    hipStream_t st;
    // Where the updates modify the right-hand side and where the solved rows
    // live: B' for both, or separate buffers when blocks are solved by product
    // (B is then written once at the end).
    View rhs;
    View x;
    // Band store of the inverses of the whole 512-row diagonal blocks, when
    // those are solved by product: element (i, j) of the block diagonal
    // inverse at band[(i - j + BAND_KL) + j * BAND_LD], so every diagonal
    // block, and every block within BAND_KL of the diagonal, is a
    // column-major matrix with leading dimension BAND_LD - 1, and the blocks
    // along the diagonal are a constant stride apart.
    const void* band = nullptr;
    // Where the composition of those inverses reads the triangle's blocks within
    // them: a, or a copy of those blocks when a has no unit stride.
    View tri;
};

constexpr int64_t BAND_KL = PB;
constexpr int64_t BAND_LD = 2 * BAND_KL + 1;

// Block (r, c) of the inverse in the band store (|r - c| + block size - 1 <= BAND_KL).
inline View band_view(const Solve& s, int64_t r, int64_t c) {
    return { (char*)const_cast<void*>(s.band) + ((r - c + BAND_KL) + c * BAND_LD) * (int64_t)dt_size(s.dt),
             1, BAND_LD - 1 };
}

inline void* offset(const View& v, int64_t i, int64_t j, size_t es) {
    return (char*)v.ptr + (i * v.rs + j * v.cs) * (int64_t)es;
}

// Inverses of `count` consecutive 64-row diagonal blocks into the band.
template <typename T>
void inverse_launch(const Solve& s, int count) {
    const View b0 = band_view(s, 0, 0);
    const dim3 grid((unsigned)(LB / INV_CPW / WPB), (unsigned)count), block(64 * WPB);
    const int64_t a_step = LB * (s.a.rs + s.a.cs), b_step = LB * BAND_LD;
    if (s.lower)
        hipLaunchKernelGGL((trsm_inverse_kernel<T, true, INV_CPW>), grid, block, 0, s.st,
                           (const T*)s.a.ptr, s.a.rs, s.a.cs, (T*)b0.ptr, b0.cs, (int)s.unit,
                           a_step, b_step);
    else
        hipLaunchKernelGGL((trsm_inverse_kernel<T, false, INV_CPW>), grid, block, 0, s.st,
                           (const T*)s.a.ptr, s.a.rs, s.a.cs, (T*)b0.ptr, b0.cs, (int)s.unit,
                           a_step, b_step);
    HIP_CHECK(hipGetLastError());
}

// X[r0 .. r0 + m - 1] = alpha * inv(L_rr) * R[r0 ..] by substitution, m <= SLAB.
template <typename T>
void slab(const Solve& s, int64_t r0, int64_t m, double alpha) {
    const size_t es = sizeof(T);
    // An upper triangle is a lower one with its rows and columns reversed.
    const int64_t d = s.lower ? 1 : -1, f = s.lower ? r0 : r0 + m - 1;
    const dim3 grid((unsigned)((s.n + 15) / 16)), block(512);
    const T* a = (const T*)offset(s.a, f, f, es);
    const T* b = (const T*)offset(s.rhs, f, 0, es);
    T* x = (T*)offset(s.x, f, 0, es);
    // Two or four 16-row tiles per wave (up to 256 or 512 rows).
    if (m <= 256)
        hipLaunchKernelGGL((trsm_slab_kernel<T, 2>), grid, block, 0, s.st, a, d * s.a.rs,
                           d * s.a.cs, b, d * s.rhs.rs, s.rhs.cs, x, d * s.x.rs, s.x.cs, (int)m,
                           s.n, (T)alpha, (int)s.unit);
    else
        hipLaunchKernelGGL((trsm_slab_kernel<T, 4>), grid, block, 0, s.st, a, d * s.a.rs,
                           d * s.a.cs, b, d * s.rhs.rs, s.rhs.cs, x, d * s.x.rs, s.x.cs, (int)m,
                           s.n, (T)alpha, (int)s.unit);
    HIP_CHECK(hipGetLastError());
}

// R[dst rows] := beta * R[dst rows] - L_eff[dst rows, src rows] * X[src rows]
void update(const Solve& s, int64_t dst0, int64_t dstn, int64_t src0, int64_t srcn,
            double beta) {
    const size_t es = dt_size(s.dt);
    GemmDesc d;
    d.dt = s.dt;
    d.m = dstn; d.n = s.n; d.k = srcn;
    d.a = { offset(s.a, dst0, src0, es), s.a.rs, s.a.cs };
    d.b = { offset(s.x, src0, 0, es), s.x.rs, s.x.cs };
    d.c = { offset(s.rhs, dst0, 0, es), s.rhs.rs, s.rhs.cs };
    d.alpha = -1.0;
    d.beta = beta;
    // FP64 updates of 1024 and 2048 rows (n = 1024, k = rows, operands in
    // the solve's layout), measured over the tile table with 1, 2 and 4 k
    // partitions: 1024 rows are fastest on 128x64x16 tiles of eight waves
    // in two partitions (53.1 us against 59.7 on 64x64x32 tiles and 57.8 on
    // the size heuristic's 32x32), 2048 rows on 128x64x32 tiles in one
    // (158 against 173 us on the heuristic's 64x64). Every tile gives the
    // same result; the partitioned sum rounds in another order.
    GemmConfig cfg;
    if (s.dt == Dt::F64 && dstn >= 1536 && srcn >= 1536) cfg.tile = 11;
    else if (s.dt == Dt::F64 && dstn >= 768 && srcn >= 768) { cfg.tile = 7; cfg.split_k = 2; }
    gemm_run(d, cfg.tile >= 0 ? &cfg : nullptr, s.st);
}

// X[r0 .. r0+511] = alpha * inv(L_pp) * R[r0 .. r0+511] for an aligned
// 512-row block: one product with its inverse.
void block_by_product(const Solve& s, int64_t r0, double alpha) {
    const size_t es = dt_size(s.dt);
    GemmDesc d;
    d.dt = s.dt;
    d.m = PB; d.n = s.n; d.k = PB;
    d.a = band_view(s, r0, r0);
    d.b = { offset(s.rhs, r0, 0, es), s.rhs.rs, s.rhs.cs };
    d.c = { offset(s.x, r0, 0, es), s.x.rs, s.x.cs };
    d.alpha = alpha;
    d.beta = 0.0;
    gemm_run(d, nullptr, s.st);
}

void solve(const Solve& s, int64_t r0, int64_t m, double alpha) {
    if (m <= SLAB) {
        if (s.band && m == PB) block_by_product(s, r0, alpha);
        else if (s.dt == Dt::F64) slab<double>(s, r0, m, alpha);
        else slab<float>(s, r0, m, alpha);
        return;
    }
    // Halves of whole tiles; with inverted blocks, of whole blocks, the
    // ragged rest at the end.
    const int64_t unit = s.band ? PB : 16;
    const int64_t m1 = (m / 2 + unit - 1) / unit * unit, m2 = m - m1;
    if (s.lower) {
        solve(s, r0, m1, alpha);
        update(s, r0 + m1, m2, r0, m1, alpha);
        solve(s, r0 + m1, m2, 1.0);
    } else {
        solve(s, r0 + m1, m2, alpha);
        update(s, r0, m1, r0 + m1, m2, alpha);
        solve(s, r0, m1, 1.0);
    }
}

// Inverses of 2b rows from those of b rows in the band store (b = 64, 128,
// 256), for every aligned pair: inv([[L11, 0], [L21, L22]]) =
// [[inv(L11), 0], [-inv(L22) L21 inv(L11), inv(L22)]] for a lower triangle,
// inv([[U11, U12], [0, U22]]) = [[inv(U11), -inv(U11) U12 inv(U22)],
// [0, inv(U22)]] for an upper one. Both products are one strided launch over
// the pairs: in the band the pairs are 2b * BAND_LD elements apart, in the
// triangle (or its copy) 2b (rs + cs). The blocks passed the dominance check, so the
// inverse applied first has condition number at most 48 and the product form
// loses at most that factor against the substitution it replaces.
void compose_band(const Solve& s, int64_t rows, int64_t b) {
    const size_t es = dt_size(s.dt);
    const int64_t npair = rows / (2 * b);
    if (npair < 1) return;
    void* t = workspace((size_t)npair * b * b * es, 19);
    const bool upper = !s.lower;
    const int64_t step = 2 * b * BAND_LD;
    GemmDesc d;
    d.dt = s.dt;
    d.m = b; d.n = b; d.k = b;
    // Lower: T_p = L21_p * inv(L11_p). Upper: T_p = U12_p * inv(U22_p).
    d.a = upper ? View{ offset(s.tri, 0, b, es), s.tri.rs, s.tri.cs }
                : View{ offset(s.tri, b, 0, es), s.tri.rs, s.tri.cs };
    d.b = upper ? band_view(s, b, b) : band_view(s, 0, 0);
    d.c = { t, 1, b };
    d.alpha = 1.0;
    d.beta = 0.0;
    gemm_strided_run(d, (int)npair, 2 * b * (s.tri.rs + s.tri.cs), step, b * b, s.st);
    // Lower: -inv(L22_p) * T_p below the diagonal. Upper: -inv(U11_p) * T_p
    // to its right.
    d.a = upper ? band_view(s, 0, 0) : band_view(s, b, b);
    d.b = { t, 1, b };
    d.c = upper ? band_view(s, 0, b) : band_view(s, b, 0);
    d.alpha = -1.0;
    gemm_strided_run(d, (int)npair, step, b * b, step, s.st);
}

} // namespace detail_trsm
using namespace detail_trsm;

// The stream of the diagonal-block check: created once, default priority,
// not ordered with the legacy default stream.
hipStream_t check_stream() {
    static hipStream_t cs = nullptr;
    if (!cs) HIP_CHECK(hipStreamCreateWithFlags(&cs, hipStreamNonBlocking));
    return cs;
}

static bool capturing(hipStream_t st) {
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    HIP_CHECK(hipStreamIsCapturing(st, &cap));
    return cap != hipStreamCaptureStatusNone;
}

void trsm_run(Dt dt, side_t side, uplo_t uplo, trans_t trans, diag_t diag, int64_t m,
              int64_t n, double alpha, View a, View b, hipStream_t st) {
    if (m <= 0 || n <= 0) return;
    const bool t = ((unsigned)trans & BLIS_TRANS_BIT) != 0;
    const bool lower = (uplo == BLIS_LOWER);
    Solve s;
    s.dt = dt;
    s.unit = (diag == BLIS_UNIT_DIAG);
    s.st = st;
    View bv;          // B'(i,j) = bv.ptr[i*bv.rs + j*bv.cs]
    int64_t rows;
    if (side == BLIS_LEFT) {
        // L_eff = op(A).
        s.a = { a.ptr, t ? a.cs : a.rs, t ? a.rs : a.cs };
        s.lower = t ? !lower : lower;
        bv = b;
        s.n = n;
        rows = m;
    } else {
        // X op(A) = alpha B  <=>  op(A)^T X^T = alpha B^T.
        s.a = { a.ptr, t ? a.rs : a.cs, t ? a.cs : a.rs };
        s.lower = t ? lower : !lower;
        bv = { b.ptr, b.cs, b.rs };
        s.n = m;
        rows = n;
    }
    s.rhs = bv;
    s.x = bv;
    // A large triangle over many columns: check its whole 512-row diagonal
    // blocks for dominance while they are inverted, and solve them by GEMM
    // products when all pass. The host reads the check's flags, so a solve that
    // is being captured is by substitution.
    const int64_t whole = rows / PB * PB;
    const int nblk = (int)(whole / NB);
    const size_t es = dt_size(dt);
    const bool gather = s.a.rs != 1 && s.a.cs != 1;
    int* d_ok = nullptr;
    void *band = nullptr, *blocks = nullptr;
    if (rows >= TRSM_INV_MIN_ROWS && s.n >= TRSM_INV_MIN_N && !capturing(st)) {
        d_ok = (int*)try_workspace(sizeof(int) * nblk, 15);
        band = try_workspace((size_t)(whole + 1) * BAND_LD * es, 13);
        if (gather) blocks = try_workspace((size_t)whole * (PB + 1) * es, 14);
    }
    // Substitution needs none of these, and is what is left without memory.
    if (d_ok && band && (blocks || !gather)) {
        // The check runs on a side stream, beside the inversion on the main
        // stream; only the host reads its flags (pinned memory, one wait).
        hipStream_t cs = check_stream();
        hipEvent_t ready, checked;
        HIP_CHECK(hipEventCreateWithFlags(&ready, hipEventDisableTiming));
        HIP_CHECK(hipEventCreateWithFlags(&checked, hipEventDisableTiming));
        HIP_CHECK(hipEventRecord(ready, st));
        HIP_CHECK(hipStreamWaitEvent(cs, ready, 0));
        if (dt == Dt::F64) {
            if (s.lower)
                hipLaunchKernelGGL((trsm_diag_check_kernel<double, true>), dim3(nblk), dim3(NB), 0,
                                   cs, (const double*)s.a.ptr, s.a.rs, s.a.cs, whole, (int)s.unit,
                                   d_ok);
            else
                hipLaunchKernelGGL((trsm_diag_check_kernel<double, false>), dim3(nblk), dim3(NB),
                                   0, cs, (const double*)s.a.ptr, s.a.rs, s.a.cs, whole,
                                   (int)s.unit, d_ok);
        } else {
            if (s.lower)
                hipLaunchKernelGGL((trsm_diag_check_kernel<float, true>), dim3(nblk), dim3(NB), 0,
                                   cs, (const float*)s.a.ptr, s.a.rs, s.a.cs, whole, (int)s.unit,
                                   d_ok);
            else
                hipLaunchKernelGGL((trsm_diag_check_kernel<float, false>), dim3(nblk), dim3(NB), 0,
                                   cs, (const float*)s.a.ptr, s.a.rs, s.a.cs, whole, (int)s.unit,
                                   d_ok);
        }
        HIP_CHECK(hipGetLastError());
        std::vector<int> ok(nblk, 0);
        static int* pinned = nullptr;
        constexpr int PINNED_FLAGS = 1 << 16;
        if (!pinned) HIP_CHECK(hipHostMalloc((void**)&pinned, sizeof(int) * PINNED_FLAGS));
        int* flags = nblk <= PINNED_FLAGS ? pinned : ok.data();
        HIP_CHECK(hipMemcpyAsync(flags, d_ok, sizeof(int) * nblk, hipMemcpyDeviceToHost, cs));
        HIP_CHECK(hipEventRecord(checked, cs));
        // 64-row inverses straight into the band, then 128-, 256- and 512-row
        // ones by composition, all before the wait for the check, so that the
        // GPU stays busy while the host reads the flags.
        s.band = band;
        s.tri = s.a;
        if (gather) {
            // The composition's products need a unit stride. The updates pack
            // their blocks of the triangle themselves, as every GEMM does.
            // FP64 4096 x 1024 with strides 2 and 8192: 582 us, by
            // substitution 895.
            const dim3 grid(28, (unsigned)(whole / PB)), block(256);
            if (dt == Dt::F64)
                hipLaunchKernelGGL(trsm_gather_kernel<double>, grid, block, 0, st,
                                   (const double*)s.a.ptr, s.a.rs, s.a.cs, (double*)blocks,
                                   (int)s.lower);
            else
                hipLaunchKernelGGL(trsm_gather_kernel<float>, grid, block, 0, st,
                                   (const float*)s.a.ptr, s.a.rs, s.a.cs, (float*)blocks,
                                   (int)s.lower);
            HIP_CHECK(hipGetLastError());
            s.tri = { blocks, 1, PB };
        }
        if (dt == Dt::F64) inverse_launch<double>(s, (int)(whole / LB));
        else inverse_launch<float>(s, (int)(whole / LB));
        compose_band(s, whole, LB);
        compose_band(s, whole, 2 * LB);
        compose_band(s, whole, 4 * LB);
        HIP_CHECK(hipEventSynchronize(checked));
        HIP_CHECK(hipEventDestroy(checked));
        HIP_CHECK(hipEventDestroy(ready));
        bool all = true;
        for (int i = 0; i < nblk; ++i) all = all && flags[i];
        void* xbuf = all ? try_workspace((size_t)rows * s.n * es, 16) : nullptr;
        if (xbuf) {
            // The right-hand side is updated in place and X is built in a
            // separate column-major buffer, copied over B once at the end.
            s.x = { xbuf, 1, rows };
            solve(s, 0, rows, alpha);
            if (bv.rs == 1 && bv.cs == rows) {
                // Column-stored without padding: one contiguous span, which
                // the runtime's copy moves at about 5.5 TB/s against 2.3 TB/s
                // for the tiled kernel (32 MB: 12 against 28 us).
                HIP_CHECK(hipMemcpyAsync(bv.ptr, s.x.ptr, (size_t)rows * s.n * es,
                                         hipMemcpyDeviceToDevice, st));
                return;
            }
            const int64_t tiles = ((rows + 63) / 64) * ((s.n + 63) / 64);
            const unsigned gc = (unsigned)std::max<int64_t>(1, std::min<int64_t>(tiles, 8192));
            if (dt == Dt::F64)
                hipLaunchKernelGGL(trsm_copy_kernel<double>, dim3(gc), dim3(256), 0, st,
                                   (const double*)s.x.ptr, s.x.rs, s.x.cs, (double*)bv.ptr, bv.rs,
                                   bv.cs, rows, s.n);
            else
                hipLaunchKernelGGL(trsm_copy_kernel<float>, dim3(gc), dim3(256), 0, st,
                                   (const float*)s.x.ptr, s.x.rs, s.x.cs, (float*)bv.ptr, bv.rs,
                                   bv.cs, rows, s.n);
            HIP_CHECK(hipGetLastError());
            return;
        }
        s.band = nullptr;
    }
    solve(s, 0, rows, alpha);
}

} // namespace blis_amd
