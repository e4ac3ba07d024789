// On-chip conjugate gradients of the complex-conductivity model: a whole (frame, harmonic, lane
// group) in one workgroup, as chip.hip does for real conductivity, with the recurrences of
// complex.hip (FP32 complex vectors, FP64 complex scalars and vector updates, COCG or the
// reference's conjugated dot products).  p and the inverse diagonal in LDS (16 bytes per row and
// lane), r, x and q in registers, the matrix (16-bit positions, FP32 complex values) from L2.
//
// Bound by the chain of an iteration (two block sums with their barriers, two complex divisions,
// the gathers), not by any pipe.  Measured (MI355X): two frames x 3 harmonics of 1261 nodes, 16
// patterns, 216 steps of the reference rule: 10.8 -> 0.88 ms per forward solve (before: six launches
// per iteration).
#include <climits>

#include "chip_dev.h"
#include "complex.h"

namespace mpf {

// values S + alpha_c R of every (job, slice): cval [C][width / 8][4][np] float4 (two entries each)
__global__ void __launch_bounds__(256) k_c_chip_pack(const CJob* __restrict__ jobs, const int2* __restrict__ js,
                                                     int* __restrict__ progress, int nprogress) {
    const int at = (blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
    if (at < nprogress) progress[at] = 0;
    const int2 pr = js[blockIdx.y];
    const CJob& J = jobs[pr.x];
    const int s = pr.y, np = J.np, pos = blockIdx.x * 256 + threadIdx.x;
    const int row = J.crow[pos];
    const float al = J.alpha[s];
    const int noct = J.width / 8;
    for (int o = 0; o < noct; ++o) {
        float2 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t e = (size_t)(8 * o + u) * np + row;
            const float2 sv = J.sv[e], rv = J.rv[e];
            v[u] = make_float2(sv.x + al * rv.x, sv.y + al * rv.y);
        }
        float4* out = J.cval + ((size_t)(s * noct + o) * 4) * np + pos;
#pragma unroll
        for (int h = 0; h < 4; ++h)
            out[(size_t)h * np] = make_float4(v[2 * h].x, v[2 * h].y, v[2 * h + 1].x, v[2 * h + 1].y);
    }
}

// the lane's own component and its partner's as one complex number (columns 2 g + component,
// wave_sum's order)
template <int W>
__device__ __forceinline__ zd whole(double v, int l) {
    const double o = W == 4 ? dpp<kXor2>(v) : dpp<kXor1>(v);
    const bool im = W == 4 ? (l & 2) != 0 : (l & 1) != 0;
    return im ? zd{o, v} : zd{v, o};
}

// a / b by Smith's algorithm as cplx.h's, without its branch (the lanes of a wavefront hold other
// columns) and with what depends on b alone apart
struct ZDiv {
    double r, d;
    bool swap;
    __device__ explicit ZDiv(zd b) {
        swap = !(fabs(b.x) >= fabs(b.y));
        const double big = swap ? b.y : b.x, small = swap ? b.x : b.y;
        r = small / big;
        d = big + small * r;
    }
    __device__ zd of(zd a) const {
        const double u = swap ? a.y : a.x, w = swap ? a.x : a.y;
        const double im = w - u * r;
        return zd{(u + w * r) / d, (swap ? -im : im) / d};
    }
};

// HOLD: one 8-slot group per row, kept in registers over the iterations
template <int G, int K, int NT, bool HOLD>
__global__ void __launch_bounds__(NT, NT / 256) k_c_chip(const CJob* __restrict__ jobs, const int4* __restrict__ items,
                                                         const int2* __restrict__ gin, int2* __restrict__ gout,
                                                         int* progress, int phase) {
    constexpr int NP = K * NT, W = 2 * G;
    typedef typename ChipVec<W>::type VecW;        // G complex columns
    __shared__ VecW ps[NP];
    __shared__ float2 ds[NP];
    __shared__ double red1[NT / 64][2 * W], red2[NT / 64][W + G];
    __shared__ int told;                           // the leader's word
    const int4 it = items[blockIdx.x];
    const CJob& J = jobs[it.x];
    const int s = it.y, lane0 = it.z * G, me = it.w + it.z;
    const int tid = threadIdx.x, nt = K > 1 ? NT : (int)blockDim.x, l = tid & 63, nw = nt >> 6;
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int np = J.np, n = J.n, Rq = J.Rq;
    const int col = col_of<G>(l), lane = lane0 + col;   // the lane's pattern column (both components)
    const bool reference = J.rule == MPF_STOP_REFERENCE, herm = J.herm != 0, dc = s == 0;
    const int lead = J.col0 / G;
    const size_t base = (size_t)s * np * Rq + lane0;
    float2 *X = J.x + base, *Rs = J.r + base, *Ps = J.p + base;
    int target = INT_MAX, steps = 0;
    if (phase == 0) {
        if (lane0 >= J.Ru) {
            for (int pos = tid; pos < np; pos += nt)
#pragma unroll
                for (int g = 0; g < G; ++g) X[(size_t)pos * Rq + g] = make_float2(0.0f, 0.0f);
            if (tid == 0) gout[me] = make_int2(0, kChipEmpty);
            return;
        }
    } else {
        const int2 own = gin[me];
        if (reference) target = gin[it.w + lead].x;
        else {
            target = 0;
            for (int g = 0; g * G < J.Ru; ++g) target = max(target, gin[it.w + g].x);
        }
        if (own.y || own.x == target) {
            if (tid == 0) gout[me] = own;
            return;
        }
        target = min(target, J.maxit);
        steps = own.x;
    }
    const bool decides = phase == 0 && reference && it.z == lead, follows = phase == 0 && reference && !decides;
    int* const word = progress + it.w;
    const int noct = J.width / 8;
    int npu = np;
    const __amdgpu_buffer_rsrc_t ids = uniform_rsrc(J.cid, (size_t)noct * np * 16);
    const __amdgpu_buffer_rsrc_t val = uniform_rsrc(J.cval + (size_t)s * noct * 4 * np, (size_t)noct * 4 * np * 16);
    auto load = [&](__amdgpu_buffer_rsrc_t rs, int first) {
        return __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)tid * 16u, first * 16, 0);
    };
    auto has = [&](int k) { return (wave + k * nw) * 64 < npu; };
    float r[K][W], x[K][W], q[K][W];               // q: A p, then z
    v4u hid[HOLD ? K : 1], hval[HOLD ? K : 1][4];
    uint64_t more = 0;
    uint32_t real = 0;
    // one term a . b of a Krylov dot product
    auto dot = [&](zd a, zd b) { return herm ? a * zconj(b) : a * b; };
    // z = D^-1 r into q; r.z and r.r
    auto precondition = [&](double (&vz)[W], double (&vr)[G]) {
#pragma unroll
        for (int g = 0; g < G; ++g) { vz[2 * g] = 0.0; vz[2 * g + 1] = 0.0; vr[g] = 0.0; }
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const zd d = zf(ds[tid + k * nt]);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const zd rn = zmake((double)r[k][2 * g], (double)r[k][2 * g + 1]);
                const float2 z = fz(d * rn);
                q[k][2 * g] = z.x;
                q[k][2 * g + 1] = z.y;
                const zd t = dot(rn, zf(z));
                vz[2 * g] += t.x;
                vz[2 * g + 1] += t.y;
                vr[g] += zabs2(rn);
            }
        });
    };
    // totals of a complex and a real quantity per column (one barrier)
    auto sum_zr = [&](const double (&vz)[W], const double (&vr)[G], zd& z, double& rr) {
        const double a = wave_sum<W>(vz, l), b = wave_sum<G>(vr, l);
        if (l < W) red2[wave][col_of<W>(l)] = a;
        if (l < G) red2[wave][W + col] = b;
        __syncthreads();
        z = whole<W>(across_waves<W>(&red2[0][0], W + G, nw, l), l);
        rr = across_waves<G>(&red2[0][W], W + G, nw, l);
    };

    // ---- start -----------------------------------------------------------------
    zd rho;
    double bb;
    {
        const bool resume = steps > 0;
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const int pos = tid + k * nt;
            float2 d = make_float2(0.0f, 0.0f);
            float p[W];
#pragma unroll
            for (int c = 0; c < W; ++c) { r[k][c] = 0.0f; x[k][c] = 0.0f; q[k][c] = 0.0f; p[c] = 0.0f; }
            if (has(k)) {
                const int row = J.crow[pos];
                const size_t o = (size_t)row * Rq;
                if constexpr (HOLD) {
                    hid[k] = load(ids, k * nt);
#pragma unroll
                    for (int h = 0; h < 4; ++h) hval[k][h] = load(val, h * np + k * nt);
                }
                if (noct > 1)
                    more |= (uint64_t)(__builtin_amdgcn_readfirstlane((int)J.cocts[wave + k * nw]) - 1) << (2 * k);
                if (row < n) {
                    d = J.dinv[(size_t)s * np + row];
                    real |= 1u << k;
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    if (resume) {
                        const float2 a = Rs[o + g], b = X[o + g], c = Ps[o + g];
                        r[k][2 * g] = a.x; r[k][2 * g + 1] = a.y;
                        x[k][2 * g] = b.x; x[k][2 * g + 1] = b.y;
                        p[2 * g] = c.x; p[2 * g + 1] = c.y;
                    } else if (lane0 + g < J.Ru) {
                        r[k][2 * g] = (float)((double)J.beta[s] * J.F[(size_t)row * J.Fp + lane0 + g]);
                    }
                }
            }
            ds[pos] = d;
            ps[pos] = pack<W>(p);
        });
        if (resume) {
            rho = J.sc[((size_t)ZF_RHO * J.C + s) * Rq + lane];
            bb = J.sc[((size_t)ZF_BB * J.C + s) * Rq + lane].x;
        } else {
            double vz[W], vr[G];
            precondition(vz, vr);
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                ps[tid + k * nt] = pack<W>(q[k]);
            });
            sum_zr(vz, vr, rho, bb);
        }
    }
    __syncthreads();

    // ---- iterations ------------------------------------------------------------
    int flags = 0;
    bool late = false;
    while (true) {
        asm volatile("" : "+s"(npu), "+s"(wave), "+v"(real));   // as in chip.hip
        int seen = 0;
        if (follows && tid == 0) seen = lead_seen(word);
        double pq[W], pu[W];
#pragma unroll
        for (int c = 0; c < W; ++c) { pq[c] = 0.0; pu[c] = 0.0; }
        v4u idn, vn[4];
        if constexpr (!HOLD) {
            idn = load(ids, 0);
#pragma unroll
            for (int h = 0; h < 4; ++h) vn[h] = load(val, h * npu);
        }
        const ZDiv by_rho(rho);
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            if constexpr (!HOLD) __builtin_amdgcn_sched_barrier(0);
            v4u id, v[4];
            if constexpr (HOLD) {
                id = hid[k];
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h] = hval[k][h];
            } else {
                id = idn;
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h] = vn[h];
                if (k + 1 < K) {
                    idn = load(ids, (k + 1) * nt);
#pragma unroll
                    for (int h = 0; h < 4; ++h) vn[h] = load(val, h * npu + (k + 1) * nt);
                }
            }
            if (has(k)) {
                float acc[W];
#pragma unroll
                for (int c = 0; c < W; ++c) acc[c] = 0.0f;
                for (int o = 0;;) {
#pragma unroll
                    for (int h = 0; h < 4; ++h)
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const float ar = __uint_as_float(v[h][2 * u]), ai = __uint_as_float(v[h][2 * u + 1]);
                            float g[W];
                            unpack<W>(ps[(id[h] >> (16 * u)) & 0xFFFF], g);
#pragma unroll
                            for (int c = 0; c < G; ++c) {
                                acc[2 * c] += ar * g[2 * c] - ai * g[2 * c + 1];
                                acc[2 * c + 1] += ar * g[2 * c + 1] + ai * g[2 * c];
                            }
                        }
                    if (HOLD || o++ >= (int)((more >> (2 * k)) & 3)) break;
                    id = load(ids, o * npu + k * nt);
#pragma unroll
                    for (int h = 0; h < 4; ++h) v[h] = load(val, (4 * o + h) * npu + k * nt);
                }
                float own[W];
                unpack<W>(ps[tid + k * nt], own);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    q[k][2 * g] = acc[2 * g];
                    q[k][2 * g + 1] = acc[2 * g + 1];
                    const zd p = zmake(own[2 * g], own[2 * g + 1]), t = dot(p, zmake(acc[2 * g], acc[2 * g + 1]));
                    pq[2 * g] += t.x;
                    pq[2 * g + 1] += t.y;
                    pu[2 * g] += p.x;
                    pu[2 * g + 1] += p.y;
                }
            }
        });
        // alpha = rho / (p.q + (1^T p) . (1^T p) on the dcFree harmonic)
        zd tq, tu = zmake(0.0);
        {
            const double a = wave_sum<W>(pq, l);
            if (l < W) red1[wave][col_of<W>(l)] = a;
            if (dc) {
                const double b = wave_sum<W>(pu, l);
                if (l < W) red1[wave][W + col_of<W>(l)] = b;
            }
            __syncthreads();
            tq = whole<W>(across_waves<W>(&red1[0][0], 2 * W, nw, l), l);
            if (dc) {
                tu = whole<W>(across_waves<W>(&red1[0][W], 2 * W, nw, l), l);
                tq += dot(tu, tu);
            }
        }
        const bool pz = zzero(tq);
        const zd al = pz ? zmake(0.0) : ZDiv(tq).of(rho);
        // the columns' scalars: column g sits in lane lane_of<G>(g)
        zd a[G], un[G];
        bool zero[G];
        const uint64_t zeros = __ballot(pz);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            a[g] = zmake(__shfl(al.x, lane_of<G>(g), 64), __shfl(al.y, lane_of<G>(g), 64));
            un[g] = zmake(__shfl(tu.x, lane_of<G>(g), 64), __shfl(tu.y, lane_of<G>(g), 64));
            zero[g] = (zeros >> lane_of<G>(g)) & 1;
        }
        // r -= alpha (q + 1 1^T p), x += alpha p; a zero denominator zeroes both
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            float own[W];
            unpack<W>(ps[tid + k * nt], own);
            const bool row = (real >> k) & 1;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                zd qf = zmake(q[k][2 * g], q[k][2 * g + 1]);
                if (dc && row) qf += un[g];
                const float2 ro = fz(zmake(r[k][2 * g], r[k][2 * g + 1]) - a[g] * qf);
                const float2 xo = fz(zmake(x[k][2 * g], x[k][2 * g + 1]) + a[g] * zmake(own[2 * g], own[2 * g + 1]));
                r[k][2 * g] = zero[g] ? 0.0f : ro.x;
                r[k][2 * g + 1] = zero[g] ? 0.0f : ro.y;
                x[k][2 * g] = zero[g] ? 0.0f : xo.x;
                x[k][2 * g + 1] = zero[g] ? 0.0f : xo.y;
            }
        });
        double vz[W], vr[G], rr;
        precondition(vz, vr);
        zd rz;
        if (follows && tid == 0) told = lead_word(word, steps + 1, seen);
        sum_zr(vz, vr, rz, rr);
        const bool rz0 = zzero(rho);
        const zd be = rz0 ? zmake(0.0) : by_rho.of(rz);
        const uint64_t bzeros = __ballot(rz0);
        rho = rz;
        ++steps;
        // stop rules as k_c_state
        const bool mine = lane < J.Ru;
        bool open;
        if (reference) open = lane == J.col0 && sqrt(sqrt(zabs2(rz)) / bb) >= 1.1920928955078125e-07;
        else open = mine && bb > 0.0 && !(rr <= J.tol * J.tol * bb);
        const bool live = __ballot(open) != 0;
        const bool bad = __ballot(mine && !(isfinite(rr) && isfinite(rz.x) && isfinite(rz.y))) != 0;
        bool stop;
        if (follows) {
            const int v = told;
            late = v < 0;
            stop = late || v == 2 * steps + 1;
        } else if (reference && it.z != lead) stop = steps >= target;
        else {
            stop = (!live && (phase == 0 || steps >= target)) || steps >= J.maxit;
            // the iteration cap reports, converged in its last step or not
            if (steps >= J.maxit) flags = kChipCapped;
        }
        if (bad) { stop = true; flags = kChipNan; }
        if (decides && tid == 0) lead_tell(word, 2 * steps + stop);
        zd b[G];
#pragma unroll
        for (int g = 0; g < G; ++g)
            b[g] = zmake(__shfl(be.x, lane_of<G>(g), 64), __shfl(be.y, lane_of<G>(g), 64));
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            float own[W];
            unpack<W>(ps[tid + k * nt], own);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float2 p = fz(zmake(q[k][2 * g], q[k][2 * g + 1]) + b[g] * zmake(own[2 * g], own[2 * g + 1]));
                const bool bz = (bzeros >> lane_of<G>(g)) & 1;
                own[2 * g] = bz ? 0.0f : p.x;
                own[2 * g + 1] = bz ? 0.0f : p.y;
            }
            ps[tid + k * nt] = pack<W>(own);
        });
        __syncthreads();
        if (stop) break;
    }

    // ---- result and state ------------------------------------------------------
    const bool keep = !reference || late;
    each_row<K>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        if (has(k)) {
            const size_t o = (size_t)J.crow[tid + k * nt] * Rq;
            float p[W];
            unpack<W>(ps[tid + k * nt], p);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                X[o + g] = make_float2(x[k][2 * g], x[k][2 * g + 1]);
                if (keep) {
                    Rs[o + g] = make_float2(r[k][2 * g], r[k][2 * g + 1]);
                    Ps[o + g] = make_float2(p[2 * g], p[2 * g + 1]);
                }
            }
        }
    });
    if (wave == 0 && l < G && keep) {
        J.sc[((size_t)ZF_RHO * J.C + s) * Rq + lane] = rho;
        J.sc[((size_t)ZF_BB * J.C + s) * Rq + lane] = zmake(bb);
    }
    if (tid == 0) gout[me] = make_int2(steps, flags);
}

static inline void check_launch() { MPF_HIP(hipGetLastError()); }

// Two lanes halve the matrix reads, one lane puts a solve on twice the CUs: one while every group
// has a CU of its own, and where two lanes need more registers than a thread has.  512 threads
// where their K rows fit: 1280 rows 2.45 -> 1.85 ms per call against 1024 threads, whose every
// wavefront repeats the scalar recurrence
ChipShape c_chip_shape(int np, long long lanes) {
    ChipShape c;
    c.G = lanes > kChipCus && np <= 512 * 8 ? 2 : 1;
    c.threads = np <= 512 * 8 ? 512 : 1024;
    const int k = (np + c.threads - 1) / c.threads;
    for (int q : {8, 6, 5, 4, 3, 2, 1})
        if (k <= q) c.K = q;
    if (c.K == 1) c.threads = np;
    return c;
}

void launch_c_chip_pack(const CJob* d_jobs, const int2* d_js, int njs, int np, int* progress, int nprogress,
                        hipStream_t st) {
    MPF_REQUIRE(nprogress <= njs * np, "on-chip solver: more lane groups than threads");
    k_c_chip_pack<<<dim3(np / 256, njs), 256, 0, st>>>(d_jobs, d_js, progress, nprogress);
    check_launch();
}

template <int G, int NT>
static void c_chip_dispatch(const CJob* d_jobs, const int4* d_items, int n, const ChipShape& c, bool one_oct,
                            const int2* gin, int2* gout, int* progress, int phase, hipStream_t st) {
    // (1024 threads take more than 4096 rows.)  Rows of one 8-slot group: the matrix stays in registers where they have room for it (20 per
    // row; 1280 rows 1.85 -> 1.54 ms per call)
#define MPF_CHIP(k)                                                                                \
    case k:                                                                                        \
        if constexpr (G == 1 && NT == 512 && k <= 5)                                               \
            if (one_oct) {                                                                         \
                k_c_chip<G, k, NT, true><<<n, c.threads, 0, st>>>(d_jobs, d_items, gin, gout, progress, phase); \
                return;                                                                            \
            }                                                                                      \
        if constexpr (NT == 512 || k > 4) {                                                        \
            k_c_chip<G, k, NT, false><<<n, c.threads, 0, st>>>(d_jobs, d_items, gin, gout, progress, phase); \
            return;                                                                                \
        }                                                                                          \
        break;
    switch (c.K) {
        MPF_CHIP(1) MPF_CHIP(2) MPF_CHIP(3) MPF_CHIP(4) MPF_CHIP(5) MPF_CHIP(6) MPF_CHIP(8)
        default: break;
    }
#undef MPF_CHIP
    throw Error(MPF_EINVAL, "on-chip solver: no kernel for this size");
}

void launch_c_chip(const CJob* d_jobs, const int4* d_items, int n, const ChipShape& c, int width, const int2* gin,
                   int2* gout, int* progress, int phase, hipStream_t st) {
    const bool one_oct = width == 8;
    if (c.G == 2) c_chip_dispatch<2, 512>(d_jobs, d_items, n, c, one_oct, gin, gout, progress, phase, st);
    else if (c.threads <= 512) c_chip_dispatch<1, 512>(d_jobs, d_items, n, c, one_oct, gin, gout, progress, phase, st);
    else c_chip_dispatch<1, 1024>(d_jobs, d_items, n, c, one_oct, gin, gout, progress, phase, st);
    check_launch();
}

}  // namespace mpf
