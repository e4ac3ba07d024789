// FP64 solves of the Tikhonov normal equations (G + shift I) y = b (Inverse::solve,
// src/solver/inverse.cpp:212-238), batched over frames.
//
// The factorisation eliminates [A | I] block column by block column, so that it ends with
// X = L^-1 (A = L L^T) instead of L, and every later solve is two products, z = X b and
// y = X^T z, over the whole chip instead of a substitution whose 2 n / 32 dependent steps run
// in one workgroup.  In place: column block k below the diagonal holds L until step k, the
// inverse's partial sums after it; X ends up in the lower triangle and X^T mirrored in the
// upper one, so both products read contiguous columns.
//
// Step k of n / 64: one launch forms the panel L_ik = A_ik X_kk^T (i > k) and finishes the
// rows X_kj = X_kk W_kj (j < k); one launch updates every tile (i, j <= i), i > k, and the
// block of tile (k+1, k+1), which comes first, factors and inverts it for the next step.
// Tiles are 64 x 64, products on v_mfma_f64_16x16x4_f64.  Bound by the chain of n / 64 diagonal
// factorisations for one frame (64 dependent columns each), by FP64 MFMA for many.
//
// Error against an extended-precision solve, n = 63, 200 and 321, condition 1e2 to 1e7: forward 1.0 to
// 1.75 times that of factor and substitutions (1.4e-10 against 0.9e-10 at 1e7), residual 1 to 6 times
// (7e-10 against 1e-10): far below what the normal equations carry in, which are FP32 sums.
//
// Measured (MI355X, n = 1024, against the 32-column factorisation in three launches per block
// column and one-workgroup substitutions): the first diagonal tile 41 -> 24 us, a step's panel
// 16.8 -> 7.4 us and update 48 -> 28 us (64 matrices 294 -> 138 us), the arrows from this file's
// first form (whole-tile eliminations, operands loaded one by one), which matched the former
// factorisation; one solve 1140 -> 16 us, 64 solves 1610 -> 153 us (3.5 TB/s), 64 against one
// factor 1120 -> 100 us.
#include "chip_dev.h"
#include "dense.h"

namespace mpf {

typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int kSB = 64;            // tile
constexpr int kSL = kSB + 2;       // LDS row
typedef double SpdTile[kSB][kSL];

static inline void check_launch() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw Error(MPF_EHIP, std::string("kernel launch: ") + hipGetErrorString(e));
}

// A64 = G + shift I; rows and columns past n are never read
__global__ void __launch_bounds__(256) k_spd_shift(int n, const float* __restrict__ G, size_t strideG, double shift,
                                                   double* __restrict__ A, size_t strideA) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int b = blockIdx.y;
    if (i >= (size_t)n * n) return;
    const int r = (int)(i % n), c = (int)(i / n);
    A[b * strideA + i] = (double)G[b * strideG + i] + (r == c ? shift : 0.0);
}

// A 64 x 64 tile's elements, 16 per thread: every load is issued (from a clamped place) before the
// first is used; a guarded load per element would wait for each in turn (16 us per launch
// instead of 7).
struct SpdElems {
    double v[kSB * kSB / 256];
    // element u of the thread: place (u * 256 + thread) of the tile
    static __device__ __forceinline__ int place(int u) { return u * 256 + threadIdx.x; }
    template <class F>
    __device__ __forceinline__ void load(F&& at) {
#pragma unroll
        for (int u = 0; u < kSB * kSB / 256; ++u) v[u] = *at(place(u) % kSB, place(u) / kSB);
    }
};

// rows r0.., columns c0.. of the column-major a (ld entries per column, rows and nc columns
// valid) as t[column][row]; entries past them are 0 (1 on the diagonal when `unit`)
__device__ __forceinline__ void tile_load(SpdTile& t, const double* a, size_t ld, int n, int r0, int c0, int nc,
                                          bool unit) {
    SpdElems e;
    e.load([&](int r, int c) { return a + (size_t)min(r0 + r, n - 1) + (size_t)min(c0 + c, nc - 1) * ld; });
#pragma unroll
    for (int u = 0; u < kSB * kSB / 256; ++u) {
        const int r = e.place(u) % kSB, c = e.place(u) / kSB;
        t[c][r] = r0 + r < n && c0 + c < nc ? e.v[u] : (unit && r == c ? 1.0 : 0.0);
    }
}

// acc += op over the tiles' 64 contraction steps: a[t][i], b[t][j]; wavefront w owns the 32 x 32
// quadrant (w / 2, w % 2).  Lane l: operand row l % 16, step l / 16; result row 4 v + l / 16,
// column l % 16.
__device__ __forceinline__ void tile_product(const SpdTile& a, const SpdTile& b, v4d (&acc)[2][2]) {
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, o = l & 15, q = l >> 4;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
#pragma unroll 4
    for (int t = 0; t < kSB; t += 4) {
        const double a0 = a[t + q][wi + o], a1 = a[t + q][wi + 16 + o];
        const double b0 = b[t + q][wj + o], b1 = b[t + q][wj + 16 + o];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
    }
}
__device__ __forceinline__ void tile_zero(v4d (&acc)[2][2]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
}
// the product as t[column][row]
__device__ __forceinline__ void tile_put(SpdTile& t, const v4d (&acc)[2][2]) {
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, o = l & 15, q = l >> 4;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) t[wj + 16 * j + o][wi + 16 * i + 4 * v + q] = acc[i][j][v];
}

// L L^T of the 16 x 16 diagonal block of t at o and its inverse into w's, by one wavefront: lane
// r + 16 g holds columns 4 g .. 4 g + 3 of row r of both; step j passes column j and row j of the
// inverse through LDS (two buffers, no block barrier)
__device__ __forceinline__ void factor16(const SpdTile& t, SpdTile& w, int o, double (*colb)[16], double (*rowb)[16],
                                         int* info) {
    const int l = threadIdx.x & 63, r = l & 15, g = l >> 4;
    double A[4], X[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int c = 4 * g + q;
        A[q] = r >= c ? t[o + c][o + r] : t[o + r][o + c];
        X[q] = r == c ? 1.0 : 0.0;
    }
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int b = j & 1;
        if (g == j / 4) colb[b][r] = A[j % 4];
        if (r == j)
#pragma unroll
            for (int q = 0; q < 4; ++q) rowb[b][4 * g + q] = X[q];
        wave_sync();
        double d = colb[b][j];
        if (!(d > 0.0)) {
            if (l == 0) atomicExch(info, 1);
            d = 1e-300;
        }
        const double rs = rsqrt(d), lr = r > j ? colb[b][r] * rs : 0.0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const double x = rowb[b][4 * g + q] * rs;
            A[q] -= lr * (colb[b][4 * g + q] * rs);
            X[q] = r == j ? x : X[q] - lr * x;
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) w[o + 4 * g + q][o + r] = 4 * g + q <= r ? X[q] : 0.0;
}

// one wavefront's 16 x 16 product over 16 steps: a(k, row), b(k, column)
template <class FA, class FB>
__device__ __forceinline__ v4d product16(FA&& a, FB&& b) {
    const int l = threadIdx.x & 63, o = l & 15, q = l >> 4;
    v4d acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < 16; k += 4) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a(k + q, o), b(k + q, o), acc, 0, 0, 0);
    return acc;
}

// L L^T of the tile t (its lower triangle, t[column][row]) and X = L^-1 (w, the same layout)
// written to rows and columns d0.. of a, mirrored: the elimination of the whole matrix again
// on 16 x 16 blocks, a wavefront per block product.  A 64-step elimination by all threads with
// a barrier per step made the launch of one tile 41 us against this one's 24.
__device__ __forceinline__ void diag_factor(SpdTile& t, SpdTile& w, double (*colb)[16], double (*rowb)[16], double* a,
                                            int n, int d0, int* info) {
    const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, lo = l & 15, lq = l >> 4;
    for (int i = threadIdx.x; i < kSB * kSB; i += 256) w[i / kSB][i % kSB] = 0.0;
    __syncthreads();
#pragma unroll 1
    for (int jb = 0; jb < 4; ++jb) {
        const int o = 16 * jb;
        if (wave == 0) factor16(t, w, o, colb, rowb, info);
        __syncthreads();
        // the panel L_i = A_io X_o^T (i > jb) and the finished rows X_oj = X_o W_oj (j < jb)
        if (wave < 3) {
            const int i = wave < jb ? wave : wave + 1;
            v4d p;
            if (i > jb)
                p = product16([&](int k, int r) { return t[o + k][16 * i + r]; },
                              [&](int k, int c) { return w[o + k][o + c]; });
            else
                p = product16([&](int k, int r) { return w[o + k][o + r]; },
                              [&](int k, int c) { return w[16 * i + c][o + k]; });
            wave_sync();
            SpdTile& out = i > jb ? t : w;
            const int c0 = i > jb ? o : 16 * i, r0 = i > jb ? 16 * i : o;
#pragma unroll
            for (int v = 0; v < 4; ++v) out[c0 + lo][r0 + 4 * v + lq] = p[v];
        }
        __syncthreads();
        // blocks (i, j <= i), i > jb: A_ij -= L_i L_j^T (j > jb), W_ij -= L_i X_oj (j <= jb)
        int task = 0;
        for (int i = jb + 1; i < 4; ++i)
            for (int j = 0; j <= i; ++j, ++task) {
                if ((task & 3) != wave) continue;
                SpdTile& out = j > jb ? t : w;
                const v4d p = product16([&](int k, int r) { return t[o + k][16 * i + r]; },
                                        [&](int k, int c) { return j > jb ? t[o + k][16 * j + c] : w[16 * j + c][o + k]; });
#pragma unroll
                for (int v = 0; v < 4; ++v) out[16 * j + lo][16 * i + 4 * v + lq] -= p[v];
            }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < kSB * kSB; i += 256) {
        const int r = i % kSB, c = i / kSB;
        if (d0 + r < n && d0 + c < n) a[(size_t)(d0 + r) + (size_t)(d0 + c) * n] = r >= c ? w[c][r] : w[r][c];
    }
}

__global__ void __launch_bounds__(256, 2) k_spd_first(int n, double* __restrict__ A, size_t strideA,
                                                   int* __restrict__ info) {
    __shared__ SpdTile t, w;
    __shared__ double colb[2][16], rowb[2][16];
    double* a = A + blockIdx.y * strideA;
    tile_load(t, a, n, n, 0, 0, n, true);
    __syncthreads();
    diag_factor(t, w, colb, rowb, a, n, 0, info);
}

// blocks b < k: X_kb = X_kk W_kb (lower tile and its mirror); blocks b >= k: the panel
// L_ik = A_ik X_kk^T, i = b + 1, into P [n x 64]
__global__ void __launch_bounds__(256, 2) k_spd_panel(int n, double* __restrict__ A, size_t strideA,
                                                   double* __restrict__ P, size_t strideP, int k) {
    __shared__ SpdTile ta, tb;
    double* a = A + blockIdx.y * strideA;
    double* p = P + blockIdx.y * strideP;
    const int d0 = k * kSB, b = blockIdx.x;
    v4d acc[2][2];
    tile_zero(acc);
    // X_kk as [column][row], lower triangle (the upper one holds the mirror)
    {
        SpdElems e;
        e.load([&](int r, int c) { return a + (size_t)min(d0 + r, n - 1) + (size_t)min(d0 + c, n - 1) * n; });
#pragma unroll
        for (int u = 0; u < kSB * kSB / 256; ++u) {
            const int r = e.place(u) % kSB, c = e.place(u) / kSB;
            tb[c][r] = d0 + r < n && d0 + c < n ? (r >= c ? e.v[u] : 0.0) : (r == c ? 1.0 : 0.0);
        }
    }
    if (b < k) {
        // out[r][c] = sum_t X_kk[r][t] W_kb[t][c]: operand a[t][r] = tb, b[t][c] transposed
        const int c0 = b * kSB;
        SpdElems e;
        e.load([&](int t, int c) { return a + (size_t)min(d0 + t, n - 1) + (size_t)(c0 + c) * n; });
#pragma unroll
        for (int u = 0; u < kSB * kSB / 256; ++u) {
            const int t = e.place(u) % kSB, c = e.place(u) / kSB;
            ta[t][c] = d0 + t < n ? e.v[u] : 0.0;
        }
        __syncthreads();
        tile_product(tb, ta, acc);
        __syncthreads();
        tile_put(ta, acc);
        __syncthreads();
#pragma unroll
        for (int i0 = 0; i0 < kSB * kSB; i0 += 256) {
            const int i = i0 + threadIdx.x, r = i % kSB, c = i / kSB;
            if (d0 + r < n) a[(size_t)(d0 + r) + (size_t)(c0 + c) * n] = ta[c][r];
            if (d0 + c < n) a[(size_t)(c0 + r) + (size_t)(d0 + c) * n] = ta[r][c];
        }
    } else {
        const int r0 = (b + 1) * kSB;
        tile_load(ta, a, n, n, r0, d0, n, false);
        __syncthreads();
        // out[i][c] = sum_t A_ik[i][t] X_kk[c][t]
        tile_product(ta, tb, acc);
        __syncthreads();
        tile_put(ta, acc);
        __syncthreads();
#pragma unroll
        for (int i0 = 0; i0 < kSB * kSB; i0 += 256) {
            const int i = i0 + threadIdx.x, r = i % kSB, c = i / kSB;
            if (r0 + r < n) p[(size_t)(r0 + r) + (size_t)c * n] = ta[c][r];
        }
    }
}

// tiles (i, j <= i), i > k, (k+1, k+1) first: j > k: A_ij -= L_ik L_jk^T; j < k:
// W_ij -= L_ik X_kj; j = k: W_ik = -L_ik X_kk
__global__ void __launch_bounds__(256, 2) k_spd_update(int n, double* __restrict__ A, size_t strideA,
                                                    const double* __restrict__ P, size_t strideP, int k,
                                                    int* __restrict__ info) {
    __shared__ SpdTile ta, tb;
    __shared__ double colb[2][16], rowb[2][16];
    double* a = A + blockIdx.y * strideA;
    const double* p = P + blockIdx.y * strideP;
    // row k + 1 has k + 2 tiles, its last one (the diagonal) taken by block 0
    int b = blockIdx.x, i = k + 1, j = k + 1;
    if (b > 0) {
        --b;
        if (b <= k) j = b;
        else {
            b -= k + 1;
            i = k + 2;
            while (b > i) { b -= i + 1; ++i; }
            j = b;
        }
    }
    const int d0 = k * kSB, r0 = i * kSB, c0 = j * kSB;
    v4d acc[2][2];
    tile_zero(acc);
    tile_load(ta, p, n, n, r0, 0, kSB, false);           // L_ik as [t][row]
    if (j > k) {
        if (j != i) tile_load(tb, p, n, n, c0, 0, kSB, false);
    } else {
        // X_k,j as [t][column]: row block k of X from its mirror; the diagonal tile's mirror is
        // its upper triangle
        SpdElems e;
        e.load([&](int c, int t) { return a + (size_t)(c0 + c) + (size_t)min(d0 + t, n - 1) * n; });
#pragma unroll
        for (int u = 0; u < kSB * kSB / 256; ++u) {
            const int c = e.place(u) % kSB, t = e.place(u) / kSB;
            tb[t][c] = d0 + t < n && (j < k || c <= t) ? e.v[u] : 0.0;
        }
    }
    __syncthreads();
    if (j > k && j == i) tile_product(ta, ta, acc);
    else tile_product(ta, tb, acc);
    __syncthreads();
    tile_put(ta, acc);
    __syncthreads();
    SpdElems e;
    if (j != k) e.load([&](int r, int c) { return a + (size_t)min(r0 + r, n - 1) + (size_t)min(c0 + c, n - 1) * n; });
    if (i == k + 1 && j == k + 1) {
        // the next diagonal tile: updated in LDS, factored here
#pragma unroll
        for (int u = 0; u < kSB * kSB / 256; ++u) {
            const int r = e.place(u) % kSB, c = e.place(u) / kSB;
            ta[c][r] = r0 + r < n && c0 + c < n ? e.v[u] - ta[c][r] : (r == c ? 1.0 : 0.0);
        }
        __syncthreads();
        diag_factor(ta, tb, colb, rowb, a, n, r0, info);
        return;
    }
#pragma unroll
    for (int u = 0; u < kSB * kSB / 256; ++u) {
        const int r = e.place(u) % kSB, c = e.place(u) / kSB;
        if (r0 + r < n && c0 + c < n)
            a[(size_t)(r0 + r) + (size_t)(c0 + c) * n] = (j == k ? 0.0 : e.v[u]) - ta[c][r];
    }
}

// out[b][c] = sum over rows of column c: `upper` rows 0..c (z = X x from the mirrored X^T), else
// rows c..n-1 (X^T x).  One wavefront per column and RB right-hand sides (shared factor).
template <int RB>
__global__ void __launch_bounds__(256) k_spd_apply(int n, int nb, const double* __restrict__ A, size_t strideA,
                                                   const double* __restrict__ x, size_t stridex,
                                                   double* __restrict__ out, size_t strideout, int upper) {
    const int c = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, b0 = blockIdx.y * RB;
    if (c >= n) return;
    const double* a = A + (RB == 1 ? (size_t)b0 * strideA : 0) + (size_t)c * n;
    const int lo = upper ? 0 : c, hi = upper ? c + 1 : n;
    double s[RB];
#pragma unroll
    for (int q = 0; q < RB; ++q) s[q] = 0.0;
#pragma unroll 4
    for (int r = lo + lane; r < hi; r += 64) {
        const double v = a[r];
#pragma unroll
        for (int q = 0; q < RB; ++q)
            if (b0 + q < nb) s[q] += v * x[(size_t)(b0 + q) * stridex + r];
    }
#pragma unroll
    for (int q = 0; q < RB; ++q) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s[q] += __shfl_xor(s[q], off, 64);
        if (lane == 0 && b0 + q < nb) out[(size_t)(b0 + q) * strideout + c] = s[q];
    }
}

size_t spd_factor_work(int n, int batch) { return (size_t)batch * n * kSB; }

void launch_spd_factor(int n, const float* G, size_t strideG, double shift, double* A, size_t strideA, int batch,
                       int* d_info, double* work, hipStream_t st) {
    dim3 g0((unsigned)(((size_t)n * n + 255) / 256), batch);
    k_spd_shift<<<g0, 256, 0, st>>>(n, G, strideG, shift, A, strideA);
    const int nblk = (n + kSB - 1) / kSB;
    const size_t sp = (size_t)n * kSB;
    k_spd_first<<<dim3(1, batch), 256, 0, st>>>(n, A, strideA, d_info);
    for (int k = 0; k < nblk; ++k) {
        if (nblk > 1) k_spd_panel<<<dim3(nblk - 1, batch), 256, 0, st>>>(n, A, strideA, work, sp, k);
        if (k + 1 == nblk) break;
        int tiles = 0;
        for (int i = k + 1; i < nblk; ++i) tiles += i + 1;
        k_spd_update<<<dim3(tiles, batch), 256, 0, st>>>(n, A, strideA, work, sp, k, d_info);
    }
    check_launch();
}

void launch_spd_solve(int n, const double* A, size_t strideA, const double* b, size_t strideb, double* y,
                      size_t stridey, int batch, double* work, hipStream_t st) {
    const int blocks = (n + 3) / 4;
    if (strideA == 0 && batch > 1) {
        constexpr int RB = 8;
        const dim3 g(blocks, (batch + RB - 1) / RB);
        k_spd_apply<RB><<<g, 256, 0, st>>>(n, batch, A, 0, b, strideb, work, n, 1);
        k_spd_apply<RB><<<g, 256, 0, st>>>(n, batch, A, 0, work, n, y, stridey, 0);
    } else {
        const dim3 g(blocks, batch);
        k_spd_apply<1><<<g, 256, 0, st>>>(n, batch, A, strideA, b, strideb, work, n, 1);
        k_spd_apply<1><<<g, 256, 0, st>>>(n, batch, A, strideA, work, n, y, stridey, 0);
    }
    check_launch();
}

}  // namespace mpf
