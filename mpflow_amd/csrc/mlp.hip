// Multilayer perceptron for the learned Gauss-Newton start: dense layers with GELU,
// trained with MSE and Adam.  No counterpart in the reference.
//
// Every GEMM runs on MFMA (v_mfma_f32_32x32x16_bf16): FP32 operands in HBM are rounded to
// BF16 (nearest even) while staged in LDS, products accumulate in FP32.  One kernel covers
// the three products of a layer:
//   forward   Z = H W (+ b)        A = H  (batch x in),  B = W   (in x out)
//   backward  dW = H^T dZ          A = H^T,              B = dZ
//             dH = dZ W^T          A = dZ,               B = W^T
#include <atomic>
#include <cmath>
#include <cstring>

#include "mlp.h"
#include "threads.h"

namespace mpf {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x) {
    return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// C[m][n] = sum_k A(m, k) B(k, n) with A(m, k) = A[m*pa + k] (AK) or A[k*pa + m], B(k, n) =
// B[n*pb + k] (BK) or B[k*pb + n], at any pitch: the 128-bit loads are aligned to 4 bytes.  epi 0: C = acc;  1: Z = acc + bias[n] (stored in C) and H =
// GELU(Z);  2: C = acc + bias[n].  With gridDim.z > 1 slice z sums the K steps [z per, (z + 1) per)
// alone and stores its sum in part[z][m][n] (k_mlp_split_sum adds them).
//
// T x T outputs per workgroup, wavefronts of T/2 x T/2.  Each tile pair is staged 64 K at a time,
// converted to BF16 and written to one of two LDS buffers while the MFMAs consume the other.
// Rows and columns past M and N read a neighbour's values instead of being tested for (their
// outputs are not stored); only K is padded with zeros.
//
// Bound by the FP32 operands' L2 and HBM reads: 128 x 128 where that fills the chip halves them,
// and a product with few tiles splits K until it has enough workgroups.  Measured (MI355X) on
// 1024 -> 2048 x 3 -> 9600: one forward pass of 64 rows 35 -> 11 + 5 us per layer (unsplit, the
// weights came at 0.9 TB/s; now 3), forward and backward of 4096 rows 234 -> 353 TFLOP/s.
constexpr int kGK = 64;                // K step
constexpr int kGL = kGK + 8;           // LDS row: 72 BF16 (144 bytes, 16-byte aligned)
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// one operand's T x 64 tile: rows r0.. (of `rows`), steps k0.. (of K)
template <bool ALONG_K, int T>
struct GemmTile {
    static constexpr int kVec = T / 16;          // float4 per thread
    float4 v[kVec];
    __device__ __forceinline__ void load(const float* __restrict__ P, long pitch, int r0, int rows, int k0, int K) {
        const int tid = threadIdx.x;
        if (ALONG_K) {
            // float4 u of thread t: row (t + 256 u) / 16, k from 4 ((t + 256 u) % 16)
            if (k0 + kGK <= K) {
#pragma unroll
                for (int u = 0; u < kVec; ++u) {
                    const int f = tid + 256 * u, r = min(r0 + (f >> 4), rows - 1), c = k0 + 4 * (f & 15);
                    const f32x4u_t w = *(const f32x4u_t*)(P + (size_t)r * pitch + c);
                    v[u] = make_float4(w.x, w.y, w.z, w.w);
                }
            } else {
#pragma unroll
                for (int u = 0; u < kVec; ++u) {
                    const int f = tid + 256 * u, r = min(r0 + (f >> 4), rows - 1), c = k0 + 4 * (f & 15);
                    float e[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = P[(size_t)r * pitch + min(c + i, K - 1)];
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = c + i < K ? e[i] : 0.0f;
                    v[u] = make_float4(e[0], e[1], e[2], e[3]);
                }
            }
        } else {
            // 4 x 4 blocks: float4 4 h + u of thread t is step 4 (b / (T / 4)) + u of the four rows
            // from 4 (b % (T / 4)), b = t + 256 h
            const bool whole = r0 + T <= rows;
#pragma unroll
            for (int h = 0; h < kVec / 4; ++h)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int b = tid + 256 * h, k = k0 + 4 * (b / (T / 4)) + u, c = r0 + 4 * (b % (T / 4));
                    const float* row = P + (size_t)min(k, K - 1) * pitch;
                    float4 e;
                    if (whole) {
                        const f32x4u_t w = *(const f32x4u_t*)(row + c);
                        e = make_float4(w.x, w.y, w.z, w.w);
                    } else {
                        e = make_float4(row[min(c, rows - 1)], row[min(c + 1, rows - 1)], row[min(c + 2, rows - 1)],
                                        row[min(c + 3, rows - 1)]);
                    }
                    v[4 * h + u] = e;
                }
            if (k0 + kGK > K) {
#pragma unroll
                for (int h = 0; h < kVec / 4; ++h)
#pragma unroll
                    for (int u = 0; u < 4; ++u)
                        if (k0 + 4 * ((tid + 256 * h) / (T / 4)) + u >= K) v[4 * h + u] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    }
    __device__ __forceinline__ void store(__bf16 (*s)[kGL]) const {
        const int tid = threadIdx.x;
        if (ALONG_K) {
#pragma unroll
            for (int u = 0; u < kVec; ++u) {
                const int f = tid + 256 * u;
                *reinterpret_cast<bf16x4_t*>(&s[f >> 4][4 * (f & 15)]) =
                    bf16x4_t{(__bf16)v[u].x, (__bf16)v[u].y, (__bf16)v[u].z, (__bf16)v[u].w};
            }
        } else {
#pragma unroll
            for (int h = 0; h < kVec / 4; ++h) {
                const int b = tid + 256 * h, kq = 4 * (b / (T / 4)), c = 4 * (b % (T / 4));
                const float4 *q = v + 4 * h;
                *reinterpret_cast<bf16x4_t*>(&s[c][kq]) =
                    bf16x4_t{(__bf16)q[0].x, (__bf16)q[1].x, (__bf16)q[2].x, (__bf16)q[3].x};
                *reinterpret_cast<bf16x4_t*>(&s[c + 1][kq]) =
                    bf16x4_t{(__bf16)q[0].y, (__bf16)q[1].y, (__bf16)q[2].y, (__bf16)q[3].y};
                *reinterpret_cast<bf16x4_t*>(&s[c + 2][kq]) =
                    bf16x4_t{(__bf16)q[0].z, (__bf16)q[1].z, (__bf16)q[2].z, (__bf16)q[3].z};
                *reinterpret_cast<bf16x4_t*>(&s[c + 3][kq]) =
                    bf16x4_t{(__bf16)q[0].w, (__bf16)q[1].w, (__bf16)q[2].w, (__bf16)q[3].w};
            }
        }
    }
};

template <bool AK, bool BK, int T>
__global__ void __launch_bounds__(256, 2) k_mlp_gemm(int M, int N, int K, const float* __restrict__ A, long pa,
                                                     const float* __restrict__ B, long pb, float* __restrict__ C,
                                                     int ldc, int epi, const float* __restrict__ bias,
                                                     float* __restrict__ H, float* __restrict__ part, int per) {
    constexpr int W = T / 64;                                        // 32 x 32 MFMA tiles per wavefront side
    __shared__ __attribute__((aligned(16))) __bf16 sa[2][T][kGL];    // [m][k]
    __shared__ __attribute__((aligned(16))) __bf16 sb[2][T][kGL];    // [n][k]
    const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wm = (wave >> 1) * (T / 2), wn = (wave & 1) * (T / 2);
    GemmTile<AK, T> ta;
    GemmTile<BK, T> tb;
    f32x16_t acc[W][W];
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    const int kt0 = blockIdx.z * per, kt1 = min((K + kGK - 1) / kGK, kt0 + per);
    ta.load(A, pa, m0, M, kt0 * kGK, K);
    tb.load(B, pb, n0, N, kt0 * kGK, K);
    ta.store(sa[0]);
    tb.store(sb[0]);
    __syncthreads();
    for (int kt = kt0; kt < kt1; ++kt) {
        const int buf = (kt - kt0) & 1;
        if (kt + 1 < kt1) {
            ta.load(A, pa, m0, M, (kt + 1) * kGK, K);
            tb.load(B, pb, n0, N, (kt + 1) * kGK, K);
        }
#pragma unroll
        for (int ks = 0; ks < kGK; ks += 16) {
            const int kq = ks + (lane >> 5) * 8;
            bf16x8_t a[W], b[W];
#pragma unroll
            for (int i = 0; i < W; ++i) {
                a[i] = *reinterpret_cast<const bf16x8_t*>(&sa[buf][wm + 32 * i + (lane & 31)][kq]);
                b[i] = *reinterpret_cast<const bf16x8_t*>(&sb[buf][wn + 32 * i + (lane & 31)][kq]);
            }
#pragma unroll
            for (int i = 0; i < W; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (kt + 1 < kt1) {
            ta.store(sa[buf ^ 1]);
            tb.store(sb[buf ^ 1]);
        }
        __syncthreads();
    }
    // accumulator layout: lane -> column (lane & 31) of the 32 x 32 sub-tile (stores
    // coalesce along rows of C), register v -> row 8*(v/4) + 4*(lane/32) + v%4
    const bool split = gridDim.z > 1;
    float* out = split ? part + (size_t)blockIdx.z * M * N : C;
    const int ld = split ? N : ldc;
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
        for (int j = 0; j < W; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = m0 + wm + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
                const int col = n0 + wn + 32 * j + (lane & 31);
                if (row < M && col < N) {
                    float z = acc[i][j][v];
                    if (!split && epi >= 1) z += bias[col];
                    out[(size_t)row * ld + col] = z;
                    if (!split && epi == 1) H[(size_t)row * ldc + col] = gelu(z);
                }
            }
}

// the slices' sums added in order, then the epilogue of k_mlp_gemm
__global__ void __launch_bounds__(256) k_mlp_split_sum(int M, int N, int slices, const float* __restrict__ part,
                                                       float* __restrict__ C, int ldc, int epi,
                                                       const float* __restrict__ bias, float* __restrict__ H) {
    const int col = blockIdx.x * 256 + threadIdx.x, row = blockIdx.y;
    if (col >= N) return;
    const size_t o = (size_t)row * N + col, step = (size_t)M * N;
    float z = 0.0f;
#pragma unroll 8
    for (int q = 0; q < slices; ++q) z += part[q * step + o];
    if (epi >= 1) z += bias[col];
    C[(size_t)row * ldc + col] = z;
    if (epi == 1) H[(size_t)row * ldc + col] = gelu(z);
}

// dZ = dH * GELU'(Z) elementwise (in place on dH)
__global__ void k_mlp_gelu_back(size_t n, const float* __restrict__ Z, float* __restrict__ dH) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dH[i] *= gelu_grad(Z[i]);
}

// bias gradient: db[n] = sum over rows of dZ.  A 256-thread block owns 64 columns: row
// group g (0..3) sums rows g, g + 4, ... (loads coalesced along the columns), then the
// four group sums are added in order (a fixed summation order).
__global__ void __launch_bounds__(256) k_mlp_colsum(int M, int N, const float* __restrict__ dZ,
                                                    float* __restrict__ db) {
    const int c = threadIdx.x & 63, g = threadIdx.x >> 6;
    const int n = blockIdx.x * 64 + c;
    float s = 0.0f;
    if (n < N)
#pragma unroll 8
        for (int m = g; m < M; m += 4) s += dZ[(size_t)m * N + n];
    __shared__ float red[4][64];
    red[g][c] = s;
    __syncthreads();
    if (g == 0 && n < N) db[n] = ((red[0][c] + red[1][c]) + red[2][c]) + red[3][c];
}

// MSE: dY = 2 (Y - T) / (M N); per-block partial sums of (Y - T)^2 in FP64
__global__ void __launch_bounds__(256) k_mlp_mse(size_t n, const float* __restrict__ Y, const float* __restrict__ T,
                                                 float scale, float* __restrict__ dY, double* __restrict__ part) {
    __shared__ double red[256];
    double s = 0.0;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
        const float d = Y[i] - T[i];
        dY[i] = 2.0f * d * scale;
        s += (double)d * (double)d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// out = scale * sum of the n partials: thread t sums t, t + 256, ..., then a tree sum
__global__ void __launch_bounds__(256) k_mlp_sum(int n, const double* __restrict__ part, double scale,
                                                 double* __restrict__ out) {
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) s += part[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0] * scale;
}

// Adam (Kingma & Ba 2015) with bias correction folded into the step size
__global__ void k_mlp_adam(size_t n, float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                           float* __restrict__ v, float lr_t, float b1, float b2, float eps) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr_t * mi / (sqrtf(vi) + eps);
}

// --------------------------------------------------------------------------------
// host
// --------------------------------------------------------------------------------
static int div_up(int a, int b) { return (a + b - 1) / b; }

// slices of K: products of few tiles split it until the chip has two workgroups per CU, as long as
// a slice keeps two K steps and the partial sums' traffic (8 bytes per slice and output) stays
// below the weights' (4 K bytes per column).  slices * M * N never exceeds kSplitWork floats.
constexpr size_t kSplitWork = 512 * 64 * 64;
static int gemm_slices(int M, int N, int K) {
    const int tiles = div_up(M, 64) * div_up(N, 64);
    if (tiles > 256) return 1;
    return std::max(1, std::min({512 / tiles, K / (2 * kGK), K / (2 * M)}));
}

template <bool AK, bool BK>
static void gemm(int M, int N, int K, const float* A, long pa, const float* B, long pb, float* C, int ldc, int epi,
                 const float* bias, float* H, float* work, hipStream_t st) {
    // 128 x 128 tiles where they fill the chip (4096 rows: 267 -> 170 us per forward product)
    const bool large = (long long)div_up(M, 128) * div_up(N, 128) >= 256;
    const int nk = div_up(K, kGK), want = large || !work ? 1 : gemm_slices(M, N, K);
    const int per = div_up(nk, want), slices = div_up(nk, per);
    if (large)
        k_mlp_gemm<AK, BK, 128><<<dim3(div_up(N, 128), div_up(M, 128)), 256, 0, st>>>(M, N, K, A, pa, B, pb, C, ldc,
                                                                                     epi, bias, H, nullptr, per);
    else
        k_mlp_gemm<AK, BK, 64><<<dim3(div_up(N, 64), div_up(M, 64), slices), 256, 0, st>>>(
            M, N, K, A, pa, B, pb, C, ldc, epi, bias, H, work, per);
    if (slices > 1)
        k_mlp_split_sum<<<dim3(div_up(N, 256), M), 256, 0, st>>>(M, N, slices, work, C, ldc, epi, bias, H);
    MPF_HIP(hipGetLastError());
}

Mlp::Mlp(hipStream_t s, const std::vector<int>& d, uint64_t seed) : st(s), dims(d) {
    MPF_REQUIRE(dims.size() >= 2, "mlp: need at least one layer");
    for (int v : dims) MPF_REQUIRE(v >= 1 && v <= (1 << 20), "mlp: layer width out of range");
    L = (int)dims.size() - 1;
    W.resize(L); b.resize(L); gW.resize(L); gb.resize(L); mW.resize(L); vW.resize(L); mb.resize(L); vb.resize(L);
    uint64_t state = seed;
    auto next = [&]() {   // SplitMix64
        state += 0x9E3779B97F4A7C15ULL;
        uint64_t z = state;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
        return z ^ (z >> 31);
    };
    for (int l = 0; l < L; ++l) {
        const size_t nw = (size_t)dims[l] * dims[l + 1];
        // Glorot-uniform weights, zero biases
        const double lim = std::sqrt(6.0 / (dims[l] + dims[l + 1]));
        std::vector<float> hw(nw);
        for (auto& x : hw) x = (float)(lim * (2.0 * ((next() >> 11) * (1.0 / 9007199254740992.0)) - 1.0));
        W[l].alloc(nw); W[l].upload(hw.data(), nw, st);
        b[l].alloc(dims[l + 1]); MPF_HIP(hipMemsetAsync(b[l].p, 0, b[l].bytes(), st));
        gW[l].alloc(nw); gb[l].alloc(dims[l + 1]);
        mW[l].alloc(nw); vW[l].alloc(nw); mb[l].alloc(dims[l + 1]); vb[l].alloc(dims[l + 1]);
        MPF_HIP(hipMemsetAsync(mW[l].p, 0, mW[l].bytes(), st));
        MPF_HIP(hipMemsetAsync(vW[l].p, 0, vW[l].bytes(), st));
        MPF_HIP(hipMemsetAsync(mb[l].p, 0, mb[l].bytes(), st));
        MPF_HIP(hipMemsetAsync(vb[l].p, 0, vb[l].bytes(), st));
    }
    loss.alloc(1);
    MPF_HIP(hipStreamSynchronize(st));
}

void Mlp::ensure_batch(int B) {
    if (B <= cap) return;
    cap = B;
    Z.clear(); H.clear();
    Z.resize(L); H.resize(L);
    int wmax = 0;
    for (int l = 0; l < L; ++l) {
        Z[l].alloc((size_t)B * dims[l + 1]);
        H[l].alloc((size_t)B * dims[l + 1]);
        wmax = std::max(wmax, dims[l + 1]);
    }
    wmax = std::max(wmax, dims[0]);
    dA.alloc((size_t)B * wmax);
    dB.alloc((size_t)B * wmax);
    part.alloc(1024);
    if (!work.p) {
        try {
            work.alloc(kSplitWork);
        } catch (const Error& e) {
            if (e.code != MPF_ENOMEM) throw;   // no room: no product is split
        }
    }
}

void Mlp::forward(int B, const float* X, float* Y) {
    MPF_REQUIRE(B >= 1, "mlp: batch < 1");
    ensure_batch(B);
    const float* in = X;
    for (int l = 0; l < L; ++l) {
        const int ni = dims[l], no = dims[l + 1];
        const bool last = l == L - 1;
        gemm<true, false>(B, no, ni, in, ni, W[l].p, no, Z[l].p, no, last ? 2 : 1, b[l].p, H[l].p, work.p, st);
        in = H[l].p;
    }
    x_in = X;
    batch = B;
    if (Y) MPF_HIP(hipMemcpyAsync(Y, Z[L - 1].p, sizeof(float) * (size_t)B * dims[L], hipMemcpyDeviceToDevice, st));
}

double Mlp::backward(const float* T) {
    MPF_REQUIRE(batch > 0 && x_in, "mlp: backward needs a forward pass first");
    const int B = batch;
    const size_t ny = (size_t)B * dims[L];
    // dZ_L = 2 (Y - T) / (B * out) into dA
    const int nb = (int)std::min<size_t>(1024, (ny + 255) / 256);
    k_mlp_mse<<<nb, 256, 0, st>>>(ny, Z[L - 1].p, T, 1.0f / (float)ny, dA.p, part.p);
    k_mlp_sum<<<1, 256, 0, st>>>(nb, part.p, 1.0 / (double)ny, loss.p);
    float* dz = dA.p;
    float* dh = dB.p;
    for (int l = L - 1; l >= 0; --l) {
        const int ni = dims[l], no = dims[l + 1];
        const float* hin = l == 0 ? x_in : H[l - 1].p;
        // dW = H_in^T dZ ; db = column sums of dZ
        gemm<false, false>(ni, no, B, hin, ni, dz, no, gW[l].p, no, 0, nullptr, nullptr, work.p, st);
        k_mlp_colsum<<<(no + 63) / 64, 256, 0, st>>>(B, no, dz, gb[l].p);
        if (l > 0) {
            // dH_in = dZ W^T, then dZ_in = dH_in * GELU'(Z_in)
            gemm<true, true>(B, ni, no, dz, no, W[l].p, no, dh, ni, 0, nullptr, nullptr, work.p, st);
            const size_t n = (size_t)B * ni;
            k_mlp_gelu_back<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(n, Z[l - 1].p, dh);
            std::swap(dz, dh);
        }
    }
    MPF_HIP(hipGetLastError());
    double h = 0.0;
    MPF_HIP(hipMemcpyAsync(&h, loss.p, sizeof(double), hipMemcpyDeviceToHost, st));
    MPF_HIP(hipStreamSynchronize(st));
    return h;
}

void Mlp::adam(float lr, float b1, float b2, float eps) {
    ++t;
    const float lr_t = lr * (float)(std::sqrt(1.0 - std::pow((double)b2, (double)t)) / (1.0 - std::pow((double)b1, (double)t)));
    for (int l = 0; l < L; ++l) {
        const size_t nw = (size_t)dims[l] * dims[l + 1];
        k_mlp_adam<<<(unsigned)((nw + 255) / 256), 256, 0, st>>>(nw, W[l].p, gW[l].p, mW[l].p, vW[l].p, lr_t, b1, b2, eps);
        k_mlp_adam<<<(dims[l + 1] + 255) / 256, 256, 0, st>>>(dims[l + 1], b[l].p, gb[l].p, mb[l].p, vb[l].p, lr_t,
                                                             b1, b2, eps);
    }
    MPF_HIP(hipGetLastError());
}

int64_t Mlp::count() const {
    int64_t n = 0;
    for (int l = 0; l < L; ++l) n += (int64_t)dims[l] * dims[l + 1] + dims[l + 1];
    return n;
}

// Copies of device memory to pageable host memory by kReadThreads threads, a chunk at a time: each
// enqueues its copy into a pinned buffer of its own, waits for it and moves it on.  Bound by the
// first touch of the caller's memory, which the runtime's own copy does on one thread.  Measured
// into new arrays: 120 MB 12.0 -> 3.5 ms (first read, with the pinned buffers made, 12.6 -> 4.7), 25
// MB 1.5 -> 0.8 ms (2.4 -> 3.6), hence kReadMin: above it the first read is not slower either.
bool Mlp::read(const std::vector<Span>& spans) {
    constexpr size_t kChunk = (size_t)1 << 21;
    std::vector<Span> chunks;
    size_t total = 0;
    for (const Span& s : spans)
        for (size_t o = 0; o < s.bytes; o += kChunk) {
            chunks.push_back(Span{s.dst + o, s.src + o, std::min(kChunk, s.bytes - o)});
            total += chunks.back().bytes;
        }
    if (total < kReadMin) return false;
    if (!pinned && hipHostMalloc((void**)&pinned, kReadThreads * kChunk, hipHostMallocDefault) != hipSuccess) {
        (void)hipGetLastError();
        pinned = nullptr;
        return false;
    }
    for (auto& e : copied)
        if (!e) MPF_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    int device = 0;
    MPF_HIP(hipGetDevice(&device));
    std::atomic<size_t> next{0};
    std::atomic<int> failed{(int)hipSuccess};
    auto work = [&](int t) {
        char* buf = pinned + t * kChunk;
        hipError_t e = hipSetDevice(device);
        while (e == hipSuccess) {
            const size_t c = next.fetch_add(1);
            if (c >= chunks.size()) return;
            e = hipMemcpyAsync(buf, chunks[c].src, chunks[c].bytes, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(copied[t], st);
            if (e == hipSuccess) e = hipEventSynchronize(copied[t]);
            if (e == hipSuccess) std::memcpy(chunks[c].dst, buf, chunks[c].bytes);
        }
        failed = (int)e;
    };
    on_threads(kReadThreads, work);
    MPF_HIP((hipError_t)failed.load());
    return true;
}

Mlp::~Mlp() {
    for (auto& e : copied)
        if (e) (void)hipEventDestroy(e);
    if (pinned) (void)hipHostFree(pinned);
}

// flat order: W_0, b_0, W_1, b_1, ... (W row-major in x out)
void Mlp::params(int which, bool set, float* host) {
    MPF_REQUIRE(which == 0 || which == 1, "mlp: which must be 0 (parameters) or 1 (gradients)");
    MPF_REQUIRE(!(set && which == 1), "mlp: gradients are read-only");
    size_t off = 0;
    std::vector<Span> spans;
    for (int l = 0; l < L; ++l) {
        const size_t nw = (size_t)dims[l] * dims[l + 1];
        DBuf<float>& w = which == 0 ? W[l] : gW[l];
        DBuf<float>& bb = which == 0 ? b[l] : gb[l];
        if (set) {
            w.upload(host + off, nw, st);
            bb.upload(host + off + nw, dims[l + 1], st);
        } else {
            spans.push_back(Span{(char*)(host + off), (const char*)w.p, nw * sizeof(float)});
            spans.push_back(Span{(char*)(host + off + nw), (const char*)bb.p, dims[l + 1] * sizeof(float)});
        }
        off += nw + dims[l + 1];
    }
    if (!set && read(spans)) return;
    for (const Span& s : spans) MPF_HIP(hipMemcpyAsync(s.dst, s.src, s.bytes, hipMemcpyDeviceToHost, st));
    MPF_HIP(hipStreamSynchronize(st));
}

}  // namespace mpf
