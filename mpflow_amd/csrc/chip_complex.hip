// On-chip conjugate gradients of the complex-conductivity model: a whole (frame, harmonic, lane
// group) in one workgroup, as chip.hip does for real conductivity, with the recurrences of
// complex.hip (FP32 complex vectors, FP64 complex scalars and vector updates, COCG or the
// reference's conjugated dot products).  p and the inverse diagonal in LDS (16 bytes per row and
// lane), r, x and q in registers, the matrix (16-bit positions, FP32 complex values) from L2.
//
// Every sum runs in the order of complex.hip's kernels, so that both solvers take the same steps to
// the same bits.  COCG needs that: it has no guard against near-breakdown, the reference rule
// looks at one column only, and the order of the sums alone moves the voltages' error by ten times
// and more on some inputs (240 problems of 600 to 1261 nodes in four orders each, restated on the
// CPU: median 1.7e-7, worst 3.5e-6; one problem has 1.5e-7 in three orders and 3.2e-6 in the
// fourth).  The streamed order is: a thread adds the rows rr, rr + rpp, ... of its tile (rpp =
// 512 / Rq rows per pass), one lane adds the tile's rpp sums, then the tiles.  Hence a wavefront
// owns whole tiles, its lane the rows l, l + 64, ...  (A column that breaks down stops its lane group
// alone, not every column of its pair as there; the pair reports it all the same.)
//
// Bound by the chain of an iteration (two block sums with their barriers, two complex divisions,
// the gathers), not by any pipe.  Measured (MI355X): two frames x 3 harmonics of 1261 nodes, 16
// patterns, 216 steps of the reference rule: 10.8 -> 1.10 ms per forward solve (before: six launches
// per iteration; sums in the order that suits the lanes: 0.88 ms).
#include <climits>

#include "chip_dev.h"
#include "complex.h"

namespace mpf {

// values S + alpha_c R of every (job, slice): cval [C][width / 8][4][np] float4 (two entries each);
// one block per (pair, tile)
__global__ void __launch_bounds__(256) k_c_chip_pack(const CJob* __restrict__ jobs, const int2* __restrict__ js,
                                                     int tiles, int* __restrict__ progress, int nprogress) {
    const int at = blockIdx.x * 256 + threadIdx.x;
    if (at < nprogress) progress[at] = 0;
    const int2 pr = js[blockIdx.x / tiles];
    const CJob& J = jobs[pr.x];
    const int s = pr.y, np = J.np, row = blockIdx.x % tiles * 256 + threadIdx.x;
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
        float4* out = J.cval + ((size_t)(s * noct + o) * 4) * np + row;
#pragma unroll
        for (int h = 0; h < 4; ++h)
            out[(size_t)h * np] = make_float4(v[2 * h].x, v[2 * h].y, v[2 * h + 1].x, v[2 * h + 1].y);
    }
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

// f(acc, value) over the values of the rows l % rpp, l % rpp + rpp, ... of 64 consecutive rows (one per
// lane) in that order, rpp = 2^RL: what one thread of the streamed kernels adds in their passes
template <int RL, class F>
__device__ __forceinline__ void add_rows(double v, F&& f) {
    if constexpr (RL >= 6) f(v);
    else {
        double half[2], at[8];
        both_halves<32>(v, half);
        constexpr int N = 64 >> RL;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (RL == 5) at[h] = half[h];
            else {
                double quarter[2];
                both_halves<16>(half[h], quarter);
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    if constexpr (RL == 4) at[2 * h + g] = quarter[g];
                    else {
                        // 8 rows: the other half of the 16 lanes by a rotation
                        const double o = dpp<kRor8>(quarter[g]);
                        const bool hi = threadIdx.x & 8;
                        at[4 * h + 2 * g] = hi ? o : quarter[g];
                        at[4 * h + 2 * g + 1] = hi ? quarter[g] : o;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < N; ++i) f(at[i]);
    }
}
// the rpp sums of one tile (lane l: sum l % rpp of value q, q < Q) added from the first on: part[q].
// red: 32 columns of them at a time, of this wavefront alone
template <int RL, int Q>
__device__ __forceinline__ void add_lanes(const double (&v)[Q], double (*red)[34], double* part, int l) {
    constexpr int RPP = 1 << RL, W = RPP < 32 ? RPP : 32;
    double a = 0.0;
#pragma unroll
    for (int c = 0; c < RPP; c += W) {
        if (l >= c && l < c + W)
#pragma unroll
            for (int q = 0; q < Q; ++q) red[q][l - c] = v[q];
        wave_sync();
        if (l < Q)
#pragma unroll
            for (int k = 0; k < W; ++k) a += red[l][k];
        wave_sync();
    }
    if (l < Q) part[l] = a;
}

// K rows per thread: K / 4 tiles per wavefront, the tiles wave, wave + nw.  RL: log2 of the streamed
// kernels' rows per pass.  HOLD: one 8-slot group per row, kept in registers over the iterations.
template <int G, int K, int NT, bool HOLD, int RL>
__global__ void __launch_bounds__(NT, NT / 256) k_c_chip(const CJob* __restrict__ jobs, const int4* __restrict__ items,
                                                         const int2* __restrict__ gin, int2* __restrict__ gout,
                                                         int* progress, int polls, int phase) {
    static_assert(K == 4 || K == 8, "a wavefront owns one or two tiles");
    constexpr int NP = K * NT, W = 2 * G, NTL = NP / kTileRows;
    typedef typename ChipVec<W>::type VecW;        // G complex columns
    __shared__ VecW ps[NP];
    __shared__ float2 ds[NP];
    __shared__ double red[NT / 64][2 * W][34];
    __shared__ double part1[NTL][2 * W], part2[NTL][W + G];
    __shared__ int told;                           // the leader's word
    const int4 it = items[blockIdx.x];
    const CJob& J = jobs[it.x];
    const int s = it.y, lane0 = it.z * G, me = it.w + it.z;
    // K = 4: a wavefront per tile of the mesh; K = 8: NT threads, so that offsets are constants
    const int tid = threadIdx.x, nt = K > 4 ? NT : (int)blockDim.x, l = tid & 63, nw = nt >> 6;
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int np = J.np, n = J.n, Rq = J.Rq;
    const int col = l % G, lane = lane0 + col;     // the lane's pattern column
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
    // the k-th row of the thread, and whether its tile exists (uniform over a wavefront).  Rows whose
    // tile does not are neither loaded nor gathered: their vectors stay zero
    auto row_of = [&](int k) { return (wave + (k >> 2) * nw) * kTileRows + (k & 3) * 64 + l; };
    auto has = [&](int k) { return k < 4 || (wave + (k >> 2) * nw) * kTileRows < npu; };
    const __amdgpu_buffer_rsrc_t ids = uniform_rsrc(J.cid, (size_t)noct * np * 16);
    const __amdgpu_buffer_rsrc_t val = uniform_rsrc(J.cval + (size_t)s * noct * 4 * np, (size_t)noct * 4 * np * 16);
    // element `first` + the k-th row of a table of 16-byte elements: the thread's first row plus a
    // uniform offset, so no address registers
    auto load = [&](__amdgpu_buffer_rsrc_t rs, int k, int first) {
        return __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)(wave * kTileRows + l) * 16u,
                                                     (first + (k >> 2) * nw * kTileRows + (k & 3) * 64) * 16, 0);
    };
    float r[K][W], x[K][W], q[K][W];               // q: A p, then z
    v4u hid[HOLD ? K : 1], hval[HOLD ? K : 1][4];
    uint64_t more = 0;
    uint32_t real = 0;
    // one term a . b of a Krylov dot product
    auto dot = [&](zd a, zd b) { return zdot(herm, a, b); };
    // adds the values of the k-th rows to the tile's sums, and after its last rows those to part; those after
    // the first W only if `all`
    auto rows_done = [&](auto kc, auto& v, auto& acc, double* part, bool all) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value, Q = sizeof(acc) / sizeof(double);
        auto add = [&](int c) __attribute__((always_inline)) {
            // opaque before and after, so that the values' lanes are spread out one value after the other
            // (registers): few rows per pass, two tiles or two lanes
            constexpr bool apart = RL < 4 || !HOLD;
            if constexpr (apart) asm volatile("" : "+v"(v[c]));
            add_rows<RL>(v[c], [&](double t) { acc[c] += t; });
            if constexpr (apart) asm volatile("" : "+v"(acc[c]));
        };
#pragma unroll
        for (int c = 0; c < W; ++c) add(c);
        if (all)
#pragma unroll
            for (int c = W; c < Q; ++c) add(c);
        if constexpr (k % 4 == 3) {
            if (has(k)) add_lanes<RL, Q>(acc, red[wave], part + (wave + (k >> 2) * nw) * Q, l);
#pragma unroll
            for (int c = 0; c < Q; ++c) acc[c] = 0.0;
        }
    };
    // the tiles' sums of the lane's column: a complex value, a real one.  Tiles past the mesh's hold 0,
    // so that every read is issued before the first sum waits for one
    auto tiles = [&](const double* part, int Q, int at) __attribute__((always_inline)) {
        zd a = zmake(0.0);
#pragma unroll 8
        for (int t = 0; t < NTL; ++t) a += zmake(part[t * Q + at], part[t * Q + at + 1]);
        return a;
    };
    auto tiles_real = [&](const double* part, int Q, int at) __attribute__((always_inline)) {
        double a = 0.0;
#pragma unroll 8
        for (int t = 0; t < NTL; ++t) a += part[t * Q + at];
        return a;
    };
    for (int i = tid; i < NTL * 2 * W; i += nt) (&part1[0][0])[i] = 0.0;
    for (int i = tid; i < NTL * (W + G); i += nt) (&part2[0][0])[i] = 0.0;
    __syncthreads();
    // z = D^-1 r into q; r.z and r.r of the lane's column (one barrier)
    auto precondition = [&](zd& rz, double& rr) {
        double acc[W + G];
#pragma unroll
        for (int c = 0; c < W + G; ++c) acc[c] = 0.0;
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            double v[W + G];
            const zd d = zf(ds[row_of(k)]);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const zd rn = zmake((double)r[k][2 * g], (double)r[k][2 * g + 1]);
                const float2 z = fz(zprod(d, rn));
                q[k][2 * g] = z.x;
                q[k][2 * g + 1] = z.y;
                const zd t = dot(rn, zf(z));
                v[2 * g] = t.x;
                v[2 * g + 1] = t.y;
                v[W + g] = znorm2(rn);
            }
            rows_done(kc, v, acc, &part2[0][0], true);
        });
        __syncthreads();
        rz = tiles(&part2[0][0], W + G, 2 * col);
        rr = tiles_real(&part2[0][0], W + G, W + col);
    };

    // ---- start -----------------------------------------------------------------
    zd rho;
    double bb;
    {
        const bool resume = steps > 0;
        double acc[W + G];
#pragma unroll
        for (int c = 0; c < W + G; ++c) acc[c] = 0.0;
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const int row = row_of(k);
            float2 d = make_float2(0.0f, 0.0f);
            float p[W];
            double b[G];
#pragma unroll
            for (int c = 0; c < W; ++c) { r[k][c] = 0.0f; x[k][c] = 0.0f; q[k][c] = 0.0f; p[c] = 0.0f; }
#pragma unroll
            for (int g = 0; g < G; ++g) b[g] = 0.0;
            if (has(k)) {
                const size_t o = (size_t)row * Rq;
                if constexpr (HOLD) {
                    hid[k] = load(ids, k, 0);
#pragma unroll
                    for (int h = 0; h < 4; ++h) hval[k][h] = load(val, k, h * np);
                }
                if (noct > 1)
                    more |= (uint64_t)(__builtin_amdgcn_readfirstlane((int)J.cocts[row >> 6]) - 1) << (2 * k);
                if (row < n) {
                    d = J.dinv[(size_t)s * np + row];
                    real |= 1u << k;
                }
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    if (resume) {
                        const float2 rv = Rs[o + g], xv = X[o + g], pv = Ps[o + g];
                        r[k][2 * g] = rv.x; r[k][2 * g + 1] = rv.y;
                        x[k][2 * g] = xv.x; x[k][2 * g + 1] = xv.y;
                        p[2 * g] = pv.x; p[2 * g + 1] = pv.y;
                    } else if (lane0 + g < J.Ru) {
                        b[g] = (double)J.beta[s] * J.F[(size_t)row * J.Fp + lane0 + g];
                        r[k][2 * g] = (float)b[g];
                    }
                }
            }
            if (!resume) {
                // r.z, b.b and p = z from the right-hand side before its rounding to FP32
                double v[W];
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const float2 z = fz(zprod(zf(d), zmake(b[g])));
                    p[2 * g] = z.x;
                    p[2 * g + 1] = z.y;
                    const zd t = dot(zmake((double)r[k][2 * g], 0.0), zf(z));
                    v[2 * g] = t.x;
                    v[2 * g + 1] = t.y;
                }
#pragma unroll
                for (int c = 0; c < W; ++c) add_rows<RL>(v[c], [&](double t) { acc[c] += t; });
#pragma unroll
                for (int g = 0; g < G; ++g) add_rows<RL>(b[g], [&](double t) { acc[W + g] = fma(t, t, acc[W + g]); });
                if constexpr (k % 4 == 3) {
                    if (has(k))
                        add_lanes<RL, W + G>(acc, red[wave], &part2[wave + (k >> 2) * nw][0], l);
#pragma unroll
                    for (int c = 0; c < W + G; ++c) acc[c] = 0.0;
                }
            }
            ds[row] = d;
            ps[row] = pack<W>(p);
        });
        __syncthreads();
        if (resume) {
            rho = J.sc[((size_t)ZF_RHO * J.C + s) * Rq + lane];
            bb = J.sc[((size_t)ZF_BB * J.C + s) * Rq + lane].x;
        } else {
            rho = tiles(&part2[0][0], W + G, 2 * col);
            bb = tiles_real(&part2[0][0], W + G, W + col);
        }
    }

    // ---- iterations ------------------------------------------------------------
    int flags = 0;
    bool late = false;
    while (true) {
        asm volatile("" : "+s"(npu), "+s"(wave), "+v"(real));   // as in chip.hip
        int seen = 0;
        if (follows && tid == 0) seen = lead_seen(word);
        double acc[2 * W];
#pragma unroll
        for (int c = 0; c < 2 * W; ++c) acc[c] = 0.0;
        v4u idn, vn[4];
        if constexpr (!HOLD) {
            idn = load(ids, 0, 0);
#pragma unroll
            for (int h = 0; h < 4; ++h) vn[h] = load(val, 0, h * npu);
        }
        const ZDiv by_rho(rho);
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
                v4u id, v[4];
            if constexpr (HOLD) {
                id = hid[k];
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h] = hval[k][h];
            } else {
                id = idn;
#pragma unroll
                for (int h = 0; h < 4; ++h) v[h] = vn[h];
                if (k + 1 < K && has(k + 1)) {
                    idn = load(ids, k + 1, 0);
#pragma unroll
                    for (int h = 0; h < 4; ++h) vn[h] = load(val, k + 1, h * npu);
                }
            }
            double t[2 * W];
#pragma unroll
            for (int c = 0; c < 2 * W; ++c) t[c] = 0.0;
            if (has(k)) {
                float a[W];
#pragma unroll
                for (int c = 0; c < W; ++c) a[c] = 0.0f;
                // odd: whether the one lane is (two lanes are an even and an odd one)
                auto gather = [&](auto odd) __attribute__((always_inline)) {
                    for (int o = 0;;) {
#pragma unroll
                        for (int h = 0; h < 4; ++h)
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const float ar = __uint_as_float(v[h][2 * u]), ai = __uint_as_float(v[h][2 * u + 1]);
                                float g[W];
                                unpack<W>(ps[(id[h] >> (16 * u)) & 0xFFFF], g);
                                add_entry(odd, a[0], a[1], ar, ai, g[0], g[1]);
                                if constexpr (G == 2) add_entry(true, a[2], a[3], ar, ai, g[2], g[3]);
                            }
                        if (HOLD || o++ >= (int)((more >> (2 * k)) & 3)) break;
                        id = load(ids, k, o * npu);
#pragma unroll
                        for (int h = 0; h < 4; ++h) v[h] = load(val, k, (4 * o + h) * npu);
                    }
                };
                // a loop for either; with 128 registers one loop that forms both parts (150 spilled
                // registers against 40)
                if constexpr (NT > 512) gather((lane0 & 1) != 0);
                else if (G == 1 && (lane0 & 1)) gather(std::true_type());
                else gather(std::false_type());
                float own[W];
                unpack<W>(ps[row_of(k)], own);
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    q[k][2 * g] = a[2 * g];
                    q[k][2 * g + 1] = a[2 * g + 1];
                    const zd p = zmake(own[2 * g], own[2 * g + 1]), pq = dot(p, zmake(a[2 * g], a[2 * g + 1]));
                    t[2 * g] = pq.x;
                    t[2 * g + 1] = pq.y;
                    t[W + 2 * g] = p.x;
                    t[W + 2 * g + 1] = p.y;
                }
            }
            rows_done(kc, t, acc, &part1[0][0], dc);
        });
        __syncthreads();
        // alpha = rho / (p.q + (1^T p) . (1^T p) on the dcFree harmonic)
        zd tq = tiles(&part1[0][0], 2 * W, 2 * col), tu = zmake(0.0);
        if (dc) {
            tu = tiles(&part1[0][0], 2 * W, W + 2 * col);
            tq = tq + dot(tu, tu);
        }
        const bool pz = zzero(tq);
        const zd al = pz ? zmake(0.0) : ZDiv(tq).of(rho);
        // the columns' scalars: column g sits in lane g
        zd a[G], un[G];
        bool zero[G];
        const uint64_t zeros = __ballot(pz);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            a[g] = zmake(__shfl(al.x, g, 64), __shfl(al.y, g, 64));
            un[g] = zmake(__shfl(tu.x, g, 64), __shfl(tu.y, g, 64));
            zero[g] = (zeros >> g) & 1;
        }
        // r -= alpha (q + 1 1^T p), x += alpha p; a zero denominator zeroes both
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            float own[W];
            unpack<W>(ps[row_of(k)], own);
            const bool row = (real >> k) & 1;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                zd qf = zmake(q[k][2 * g], q[k][2 * g + 1]);
                if (dc && row) qf = qf + un[g];
                const float2 ro = fz(zmake(r[k][2 * g], r[k][2 * g + 1]) - zprod(qf, a[g]));
                const float2 xo = fz(zmake(x[k][2 * g], x[k][2 * g + 1]) + zprod(a[g], zmake(own[2 * g], own[2 * g + 1])));
                r[k][2 * g] = zero[g] ? 0.0f : ro.x;
                r[k][2 * g + 1] = zero[g] ? 0.0f : ro.y;
                x[k][2 * g] = zero[g] ? 0.0f : xo.x;
                x[k][2 * g + 1] = zero[g] ? 0.0f : xo.y;
            }
        });
        zd rz;
        double rr;
        if (follows && tid == 0) told = lead_word(word, steps + 1, seen, polls);
        precondition(rz, rr);
        const bool rz0 = zzero(rho);
        const zd be = rz0 ? zmake(0.0) : by_rho.of(rz);
        const uint64_t bzeros = __ballot(rz0);
        rho = rz;
        ++steps;
        // stop rules as k_c_state
        const bool mine = lane < J.Ru;
        bool open;
        if (reference) open = lane == J.col0 && sqrt(sqrt(znorm2(rz)) / bb) >= 1.1920928955078125e-07;
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
            b[g] = zmake(__shfl(be.x, g, 64), __shfl(be.y, g, 64));
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            float own[W];
            const int pos = row_of(k);
            unpack<W>(ps[pos], own);
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float2 p = fz(zmake(q[k][2 * g], q[k][2 * g + 1]) + zprod(b[g], zmake(own[2 * g], own[2 * g + 1])));
                const bool bz = (bzeros >> g) & 1;
                own[2 * g] = bz ? 0.0f : p.x;
                own[2 * g + 1] = bz ? 0.0f : p.y;
            }
            ps[pos] = pack<W>(own);
        });
        __syncthreads();
        if (stop) break;
    }

    // ---- result and state ------------------------------------------------------
    const bool keep = !reference || late;
    each_row<K>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        if (has(k)) {
            const size_t o = (size_t)row_of(k) * Rq;
            float p[W];
            unpack<W>(ps[row_of(k)], p);
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

// A wavefront per tile up to 8 tiles, then two per wavefront.  Two lanes halve the matrix reads, one lane
// puts a solve on twice the CUs and keeps the rows of one 8-slot group in registers.  One lane up to 8
// tiles (forward solves, one lane against two: 1261 nodes x 3 harmonics, 16 lanes, 8 frames 1.15 /
// 1.82 ms, 40 frames 3.35 / 3.76; P2 of 1873 nodes, 16 frames 3.01 / 3.55, 40 frames 7.30 / 7.04) and
// where every group has a CU of its own; two above (3997 nodes, 20 frames 16.1 / 7.6 ms, 60 frames 26.9 /
// 21.7; 2791 nodes x 2, 32 lanes, 8 frames 4.9 / 6.3, 20 frames 13.8 / 12.6); one again where two lanes need
// more registers than a thread has
ChipShape c_chip_shape(int np, long long lanes) {
    const int tiles = np / kTileRows;
    ChipShape c;
    c.G = tiles > 8 && tiles <= 16 && lanes > kChipCus ? 2 : 1;
    c.K = tiles <= 8 ? 4 : 8;
    c.threads = tiles <= 8 ? 64 * tiles : (tiles <= 16 ? 512 : 1024);
    return c;
}

void launch_c_chip_pack(const CJob* d_jobs, const int2* d_js, int njs, int np, int* progress, int nprogress,
                        hipStream_t st) {
    MPF_REQUIRE(nprogress <= njs * np, "on-chip solver: more lane groups than threads");
    k_c_chip_pack<<<njs * (np / 256), 256, 0, st>>>(d_jobs, d_js, np / 256, progress, nprogress);
    check_launch();
}

template <int G, int K, int NT, bool HOLD>
static void c_chip_dispatch(const CJob* d_jobs, const int4* d_items, int n, const ChipShape& c, int Rq,
                            const int2* gin, int2* gout, int* progress, int polls, int phase, hipStream_t st) {
    switch (Rq) {
#define MPF_CHIP(rq, rl)                                                                                    \
    case rq:                                                                                                \
        k_c_chip<G, K, NT, HOLD, rl><<<n, c.threads, 0, st>>>(d_jobs, d_items, gin, gout, progress, polls, phase); \
        return
        MPF_CHIP(8, 6);
        MPF_CHIP(16, 5);
        MPF_CHIP(32, 4);
        MPF_CHIP(64, 3);
#undef MPF_CHIP
        default: break;
    }
    throw Error(MPF_EINVAL, "on-chip solver: no kernel for this lane stride");
}

void launch_c_chip(const CJob* d_jobs, const int4* d_items, int n, const ChipShape& c, int width, int Rq,
                   const int2* gin, int2* gout, int* progress, int polls, int phase, hipStream_t st) {
    // rows of one 8-slot group: the matrix stays in registers where they have room for it (20 per row;
    // 1280 rows 1.85 -> 1.54 ms per call, measured with the sums in the lanes' own order)
    const auto launch = c.K == 8 ? (c.threads > 512 ? c_chip_dispatch<1, 8, 1024, false>
                                    : c.G == 2      ? c_chip_dispatch<2, 8, 512, false>
                                                    : c_chip_dispatch<1, 8, 512, false>)
                        : width == 8 ? c_chip_dispatch<1, 4, 512, true>
                                     : c_chip_dispatch<1, 4, 512, false>;
    launch(d_jobs, d_items, n, c, Rq, gin, gout, progress, polls, phase, st);
    check_launch();
}

}  // namespace mpf
