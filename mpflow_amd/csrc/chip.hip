// On-chip PCG: ConjugateGradient::solve (src/numeric/conjugate_gradient.cpp:61-161) of a
// whole (job, harmonic, lane group) inside one workgroup.
//
// The columns of one matrix iterate independently except for the stop test, so a
// workgroup takes G of them: p lives in LDS (the neighbour gathers read LDS only), r, x and
// q in registers, and an iteration touches memory only for the matrix (ids of 16 bits and
// FP32 values, from L2) and the coarse inverse.  The five-launch iteration moves 9.25 vector
// passes through HBM instead and pays its launches and their gaps whatever the size.
//
// What bounds it: the chain of an iteration (gathers, two block sums, the coarse product)
// more than any pipe -- at 4 lanes x 5120 rows about 30% of the cycles issue VALU and 20% LDS
// instructions -- so sums stay on the VALU (DPP and half swaps instead of LDS shuffles), the
// first coarse entries are loaded before the barrier that the sums wait for, and 512 threads
// with 256 VGPRs beat 1024 with 128 where there are lanes enough for every CU.
//
// Measured (MI355X, whole calls): one 2D forward solve of 817 nodes, 168 steps, 4.60 -> 0.42
// ms (1.02 ms with the deciding group of the reference rule run before the others); 64 frames x 5
// harmonics of 4921 nodes to 1e-6 18.1 -> 5.75 ms (1024 threads 7.2 ms against 5.5 at the time); a caller's 4921-row
// matrix with 32 columns 2.02 -> 0.56 ms.
//
// The recurrences, the FP64 scalars, the stop rules and the breakdown rules are those of the
// streaming kernels (sparse.hip); sums run in a fixed order.  One difference: a column that breaks
// down (NaN) stops its lane group alone, not every column of its pair; the pair reports it all the
// same.  A solve is one launch: it ends at its stop rule or after max_iter iterations.
#include <climits>

#include "chip_dev.h"

namespace mpf {

// --------------------------------------------------------------------------------
// chip order and matrix
// --------------------------------------------------------------------------------
__global__ void __launch_bounds__(kTileRows) k_chip_order(const uint8_t* __restrict__ tpos,
                                                          uint16_t* __restrict__ rowof,
                                                          uint16_t* __restrict__ posof) {
    const int row = blockIdx.x * kTileRows + threadIdx.x;
    const int pos = tpos ? blockIdx.x * kTileRows + tpos[row] : row;
    posof[row] = (uint16_t)pos;
    rowof[pos] = (uint16_t)row;
}

// one 64-thread block per 64 positions
__global__ void __launch_bounds__(64) k_chip_ids(int np, int width, const int32_t* __restrict__ ids,
                                                 const uint8_t* __restrict__ gw, const uint16_t* __restrict__ rowof,
                                                 const uint16_t* __restrict__ posof, uint4* __restrict__ cid,
                                                 uint8_t* __restrict__ octs) {
    const int pos = blockIdx.x * 64 + threadIdx.x;
    const int row = rowof[pos];
    const int w = gw[row / 16];      // slots past the row group's widest row are padding
    for (int o = 0; o < width / 8; ++o) {
        uint16_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int slot = 8 * o + u;
            v[u] = slot < w ? posof[ids[(size_t)slot * np + row]] : (uint16_t)pos;
        }
        uint4 p;
        p.x = v[0] | ((uint32_t)v[1] << 16);
        p.y = v[2] | ((uint32_t)v[3] << 16);
        p.z = v[4] | ((uint32_t)v[5] << 16);
        p.w = v[6] | ((uint32_t)v[7] << 16);
        cid[(size_t)o * np + pos] = p;
    }
    int m = (w + 7) / 8;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) m = max(m, __shfl_xor(m, off, 64));
    if (threadIdx.x == 0) octs[blockIdx.x] = (uint8_t)max(m, 1);
}

// the values of one (job, slice) pair: S + alpha_c R in FP32, as the SpMV stages them
__global__ void __launch_bounds__(256) k_chip_pack(const JobDev* __restrict__ jobs, const int2* __restrict__ js,
                                                   int* __restrict__ progress, int nprogress) {
    const int at = (blockIdx.y * gridDim.x + blockIdx.x) * 256 + threadIdx.x;
    if (at < nprogress) progress[at] = 0;
    const int2 pr = js[blockIdx.y];
    const JobDev& J = jobs[pr.x];
    const int s = pr.y, np = J.np, pos = blockIdx.x * 256 + threadIdx.x;
    if (pos >= np) return;
    const int row = J.crow[pos];
    const float al = J.alpha[s];
    const MPF_GLOBAL float* Sv = gp((const float*)J.s);
    const MPF_GLOBAL float* Rv = gp((const float*)J.r);
    const int noct = J.width / 8;
    for (int o = 0; o < noct; ++o) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t e = (size_t)(8 * o + u) * np + row;
            v[u] = Sv[e] + al * Rv[e];
        }
        MPF_GLOBAL float4* out = (MPF_GLOBAL float4*)gp(J.cval) + ((size_t)(s * noct + o) * 2) * np + pos;
        out[0] = make_float4(v[0], v[1], v[2], v[3]);
        out[np] = make_float4(v[4], v[5], v[6], v[7]);
    }
}

// --------------------------------------------------------------------------------
// the solver
// --------------------------------------------------------------------------------
// LDS of a block: p, the Jacobi inverse (where it fits beside p), the coarse vectors
template <int G, int NP>
constexpr bool chip_dinv_in_lds() { return (size_t)NP * 4 * (G + 1) <= 140 * 1024; }

// NT = 512: two wavefronts per SIMD with 256 VGPRs each, the most right-hand sides per
// iteration; NT = 1024: four per SIMD with 128 VGPRs, the shortest iteration of two lanes.
// HOLD: one 8-slot group per row, kept in registers over the iterations.
template <int G, int K, int NT, bool HOLD>
__global__ void __launch_bounds__(NT, NT / 256) k_pcg_chip(const JobDev* __restrict__ jobs, const int4* __restrict__ items,
                                                    const int2* __restrict__ gin, int2* __restrict__ gout,
                                                    int* progress, int polls, int phase) {
    typedef typename ChipVec<G>::type VecG;
    constexpr int NP = K * NT, NA = NP / kAggRows;
    constexpr bool DLDS = chip_dinv_in_lds<G, NP>();
    __shared__ VecG ps[NP];                        // p (0 past the rows)
    __shared__ float ds[DLDS ? NP : 1];            // Jacobi inverse
    __shared__ double gs[NA * G];                  // (W^T r)_a
    __shared__ VecG cgs[NA];                       // c_a (W^T r)_a
    __shared__ VecG cys[NA];                       // coarse correction
    __shared__ float cs[NA];                       // c_a
    __shared__ double red1[NT / 64][2 * G], red2[NT / 64][2 * G];
    __shared__ int told;                           // the leader's word
    const int4 it = items[blockIdx.x];
    const JobDev& J = jobs[it.x];
    const int s = it.y, lane0 = it.z * G, me = it.w + it.z;
    // several rows per thread: NT threads, so that every row's offset is a constant
    const int tid = threadIdx.x, nt = K > 1 ? NT : (int)blockDim.x, l = tid & 63, nw = nt >> 6;
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int np = J.np, n = J.n, Rp = J.Rp, col = col_of<G>(l), lane = lane0 + col;
    const bool reference = J.rule == MPF_STOP_REFERENCE;
    const int lead = J.col0 / G;                   // reference rule: the group that decides
    const MPF_GLOBAL uint16_t* rowof = gp(J.crow);
    const size_t base = (size_t)s * np * Rp + lane0;
    MPF_GLOBAL float* X = gp(J.x) + base;
    MPF_GLOBAL float* Rs = gp(J.rv) + base;
    MPF_GLOBAL float* Ps = gp(J.p) + base;
    int target = INT_MAX, steps = 0;
    if (phase == 0) {
        if (lane0 >= J.R) {
            // lanes past the right-hand sides stay zero
            for (int pos = tid; pos < np; pos += nt)
#pragma unroll
                for (int c = 0; c < G; ++c) X[(size_t)pos * Rp + c] = 0.0f;
            if (tid == 0) gout[me] = make_int2(0, kChipEmpty);
            return;
        }
    } else {
        const int2 own = gin[me];
        if (reference) target = gin[it.w + lead].x;
        else {
            target = 0;
            for (int g = 0; g * G < J.R; ++g) target = max(target, gin[it.w + g].x);
        }
        if (own.y || own.x == target) {
            if (tid == 0) gout[me] = own;
            return;
        }
        target = min(target, J.maxit);             // every loop below ends by the iteration cap
        steps = own.x;
    }
    const bool decides = phase == 0 && reference && it.z == lead, follows = phase == 0 && reference && !decides;
    int* const word = progress + it.w;
    const bool coarse = J.cinv != nullptr, dc = s == J.dc;
    const int na = np / kAggRows, noct = J.width / 8;
    int npu = np;
    // 16-byte elements [..][np]: a thread's offset plus a uniform one, so no address registers
    const __amdgpu_buffer_rsrc_t ids = uniform_rsrc(J.cid, (size_t)noct * np * 16);
    const __amdgpu_buffer_rsrc_t val = uniform_rsrc(J.cval + (size_t)s * noct * 2 * np, (size_t)noct * 2 * np * 16);
    auto load = [&](__amdgpu_buffer_rsrc_t rs, int first) {
        return __builtin_amdgcn_raw_buffer_load_b128(rs, (uint32_t)tid * 16u, first * 16, 0);
    };
    // positions past np: zero vectors, no gather.  Only the gather and the memory accesses
    // test for them (a uniform test: a wavefront's k-th 64 positions are one aggregate)
    auto has = [&](int k) { return (wave + k * nw) * kAggRows < npu; };
    float r[K][G], x[K][G], q[K][G];               // q: A p, then z
    float di[DLDS ? 1 : K];
    v4u hid[HOLD ? K : 1], hva[HOLD ? K : 1], hvb[HOLD ? K : 1];
    uint64_t more = 0;                             // 2 bits per k: 8-slot groups after the first
    uint32_t real = 0;                             // bit k: a row of the matrix, not padding
    auto dinv = [&](int k) {
        if constexpr (DLDS) return ds[tid + k * nt];
        else return di[k];
    };
    const __amdgpu_buffer_rsrc_t cinv =
        uniform_rsrc(coarse ? J.cinv + (size_t)s * na * J.cld : nullptr, coarse ? (size_t)na * J.cld * 4 : 0);
    // z = D^-1 r + W C cinv C W^T r into q (two barriers with a coarse level) and, added to vz, r.z as
    // r.D^-1 r over the rows and W^T r . y over the aggregates, in FP64.  W^T r is as wide as the
    // streamed kernels': FP64 at the start, in the iteration FP32 sums of 16 rows added in FP64 (FP64
    // throughout: 4% more per forward solve of 64 frames x 5 harmonics of 4921 nodes).  The coarse
    // product runs in items of 4 coarse rows (16 lanes each) x 64 columns per wavefront, four of
    // them loaded ahead: the first four before the barrier that the sums wait for.
    auto precondition = [&](double (&vz)[G], auto at_start) __attribute__((always_inline)) {
        if (coarse) {
            constexpr int PF = 4;
            int lo = l;
            asm volatile("" : "+v"(lo));           // the items' offsets are not kept across iterations
            const int nu = (na + 63) / 64, nitem = (na / 4 + nw - 1) / nw * nu;
            v4u e[PF];
            auto fetch = [&](int i0) {
#pragma unroll
                for (int i = 0; i < PF; ++i) {
                    const int iq = (i0 + i) / nu, u = (lo & 15) * 4 + 64 * ((i0 + i) - iq * nu);
                    const int a = (wave + iq * nw) * 4 + (lo >> 4);
                    e[i] = __builtin_amdgcn_raw_buffer_load_b128(
                        cinv, i0 + i < nitem && a < na && u < na ? (uint32_t)(a * J.cld + u) * 4u : 0xFFFFFFF0u, 0, 0);
                }
            };
            fetch(0);
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                double t;
                if constexpr (decltype(at_start)::value) {
                    double rd[G];
#pragma unroll
                    for (int c = 0; c < G; ++c) rd[c] = (double)r[k][c];
                    t = wave_sum<G>(rd, l);
                } else {
                    t = wave_sum_wide<G>(r[k], l);
                }
                const int a = wave + k * nw;
                if (l < G) {
                    gs[a * G + col] = t;
                    reinterpret_cast<float*>(cgs)[a * G + col] = (float)((double)cs[a] * t);
                }
            });
            __syncthreads();
            float y[G];
            for (int i0 = 0; i0 < nitem; i0 += PF) {
#pragma unroll
                for (int i = 0; i < PF; ++i) {
                    const int iq = (i0 + i) / nu, us = (i0 + i) - iq * nu, u = (lo & 15) * 4 + 64 * us;
                    const int a = (wave + iq * nw) * 4 + (lo >> 4);
                    if (i0 + i >= nitem || a - (lo >> 4) >= na) continue;
                    if (us == 0)
#pragma unroll
                        for (int c = 0; c < G; ++c) y[c] = 0.0f;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        // columns past na: the entry is 0, any finite g will do
                        float g[G];
                        unpack<G>(cgs[min(u, na - 4) + j], g);
#pragma unroll
                        for (int c = 0; c < G; ++c) y[c] = fmaf(__uint_as_float(e[i][j]), g[c], y[c]);
                    }
                    if (us == nu - 1) {
                        float o[G];
#pragma unroll
                        for (int c = 0; c < G; ++c) {
                            float t = y[c];
                            t += dpp<kXor1>(t);
                            t += dpp<kXor2>(t);
                            t += dpp<kRor4>(t);
                            t += dpp<kRor8>(t);
                            o[c] = t * cs[a];
                        }
                        if ((lo & 15) == 0) cys[a] = pack<G>(o);
                    }
                }
                if (i0 + PF < nitem) fetch(i0 + PF);
            }
            __syncthreads();
            if (tid < na) {
                float y[G];
                unpack<G>(cys[tid], y);
#pragma unroll
                for (int c = 0; c < G; ++c) vz[c] += gs[tid * G + c] * (double)y[c];
            }
        }
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const float d = dinv(k);
            float y[G];
#pragma unroll
            for (int c = 0; c < G; ++c) y[c] = 0.0f;
            if (coarse) {
                unpack<G>(cys[wave + k * nw], y);
                if (!((real >> k) & 1))
#pragma unroll
                    for (int c = 0; c < G; ++c) y[c] = 0.0f;
            }
#pragma unroll
            for (int c = 0; c < G; ++c) {
                vz[c] += (double)r[k][c] * (double)(d * r[k][c]);
                q[k][c] = fmaf(d, r[k][c], y[c]);
            }
        });
    };
    // per-lane column totals of two quantities over the block (one barrier)
    auto block_sum = [&](double (*red)[2 * G], const double (&u)[G], const double (&v)[G], bool second, double& a,
                         double& b) {
        const double wu = wave_sum<G>(u, l);
        if (l < G) red[wave][col] = wu;
        if (second) {
            const double wv = wave_sum<G>(v, l);
            if (l < G) red[wave][G + col] = wv;
        }
        __syncthreads();
        a = across_waves<G>(&red[0][0], 2 * G, nw, l);
        b = second ? across_waves<G>(&red[0][G], 2 * G, nw, l) : 0.0;
    };
    auto norms = [&](double (&vr)[G]) {
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
#pragma unroll
            for (int c = 0; c < G; ++c) vr[c] += (double)r[k][c] * (double)r[k][c];
        });
    };

    // ---- start -----------------------------------------------------------------
    double rho, bb;
    {
        const float xs = J.xscale[s];
        const bool resume = steps > 0;
        if (coarse)
            for (int a = tid; a < NA; a += nt) cs[a] = a < na ? gp((const float*)J.csc)[a] : 0.0f;
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            const int pos = tid + k * nt;
            float d = 0.0f;
            float p[G];
#pragma unroll
            for (int c = 0; c < G; ++c) { r[k][c] = 0.0f; x[k][c] = 0.0f; q[k][c] = 0.0f; p[c] = 0.0f; }
            if (has(k)) {
                const int row = rowof[pos];
                const size_t o = (size_t)row * Rp;
                if constexpr (HOLD) { hid[k] = load(ids, k * nt); hva[k] = load(val, k * nt); hvb[k] = load(val, np + k * nt); }
                if (noct > 1)
                    more |= (uint64_t)(__builtin_amdgcn_readfirstlane((int)gp(J.cocts)[wave + k * nw]) - 1) << (2 * k);
                if (row < n) {
                    d = gp((const float*)J.dinv)[(size_t)s * np + row];
                    real |= 1u << k;
                }
#pragma unroll
                for (int c = 0; c < G; ++c) {
                    if (resume) {
                        r[k][c] = Rs[o + c];
                        x[k][c] = X[o + c];
                        p[c] = Ps[o + c];
                    } else if (lane0 + c < J.R) {
                        r[k][c] = J.use_rhs ? (gp(J.rhs) + base)[o + c]
                                            : (float)(xs * gp(J.F)[s * J.fstride + o + lane0 + c]);
                    }
                }
            }
            if constexpr (DLDS) ds[pos] = d;
            else di[k] = d;
            ps[pos] = pack<G>(p);
        });
        if (resume) {
            rho = sc_ptr(J, SC_RHO, s)[lane];
            bb = sc_ptr(J, SC_BB, s)[lane];
        } else {
            __syncthreads();                       // cs
            double vb[G], vz[G];
#pragma unroll
            for (int c = 0; c < G; ++c) { vb[c] = 0.0; vz[c] = 0.0; }
            precondition(vz, std::true_type());
            norms(vb);
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                ps[tid + k * nt] = pack<G>(q[k]);
            });
            block_sum(red1, vz, vb, true, rho, bb);
            // a correction solve stops relative to the full right-hand side ||beta_c F||^2
            // left in SC_X2 by the FP64 residual
            if (J.ref_b) bb = sc_ptr(J, SC_X2, s)[lane];
        }
    }
    __syncthreads();

    // ---- iterations ------------------------------------------------------------
    int flags = 0;
    bool late = false;
    while (true) {
        // opaque per iteration: the offsets and tests derived from these are formed where they
        // are used instead of being kept in (spilled) registers across the loop
        asm volatile("" : "+s"(npu), "+s"(wave), "+v"(real));
        int seen = 0;
        if (follows && tid == 0) seen = lead_seen(word);
        double pq[G];
#pragma unroll
        for (int c = 0; c < G; ++c) pq[c] = 0.0;
        // the next positions' first 8 slots are loaded while the current ones are gathered
        v4u idn, van, vbn;
        if constexpr (!HOLD) { idn = load(ids, 0); van = load(val, 0); vbn = load(val, npu); }
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            if constexpr (!HOLD) __builtin_amdgcn_sched_barrier(0);
            v4u id, va, vb;
            if constexpr (HOLD) { id = hid[k]; va = hva[k]; vb = hvb[k]; }
            else { id = idn; va = van; vb = vbn; }
            if (!HOLD && k + 1 < K) {
                const int next = chip_step(k + 1, wave, nw, npu);   // past the rows: another row's, unused
                idn = load(ids, next);
                van = load(val, next);
                vbn = load(val, npu + next);
            }
            if (has(k)) {
                float acc[G];
#pragma unroll
                for (int c = 0; c < G; ++c) acc[c] = 0.0f;
                for (int o = 0;;) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        // four gathers in flight (registers)
                        if constexpr (!HOLD) __builtin_amdgcn_sched_barrier(0);
                        const v4u w = h ? vb : va;
                        float g[4][G];
#pragma unroll
                        for (int u = 0; u < 4; ++u)
                            unpack<G>(ps[(id[2 * h + (u >> 1)] >> (16 * (u & 1))) & 0xFFFF], g[u]);
#pragma unroll
                        for (int u = 0; u < 4; ++u)
#pragma unroll
                            for (int c = 0; c < G; ++c) acc[c] = fmaf(__uint_as_float(w[u]), g[u][c], acc[c]);
                    }
                    if (HOLD || o++ >= (int)((more >> (2 * k)) & 3)) break;
                    id = load(ids, o * npu + k * nt);
                    va = load(val, 2 * o * npu + k * nt);
                    vb = load(val, (2 * o + 1) * npu + k * nt);
                }
                float own[G];
                unpack<G>(ps[tid + k * nt], own);
#pragma unroll
                for (int c = 0; c < G; ++c) {
                    q[k][c] = acc[c];
                    pq[c] += (double)own[c] * (double)acc[c];
                }
            }
        });
        double pu[G];
#pragma unroll
        for (int c = 0; c < G; ++c) pu[c] = 0.0;
        if (dc)
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                float own[G];
                unpack<G>(ps[tid + k * nt], own);
#pragma unroll
                for (int c = 0; c < G; ++c) pu[c] += (double)own[c];
            });
        // alpha = rho / p.q; with dcFree q = A p + 1 1^T p, so p.q += (1^T p)^2
        double tq, tu;
        block_sum(red1, pq, pu, dc, tq, tu);
        tq += tu * tu;
        const float al = tq != 0.0 ? (float)(rho / tq) : 0.0f;
        // a zero p.q zeroes r and x (updateVectorKernel, conjugate_gradient_kernel.cu:77-89):
        // columns that have converged exactly, or have broken down
        const uint64_t zeros = __ballot(tq == 0.0 && lane < J.R);
        float a[G];
#pragma unroll
        for (int c = 0; c < G; ++c) a[c] = lane_value(al, lane_of<G>(c));
        if (dc) {
            float un[G];
#pragma unroll
            for (int c = 0; c < G; ++c) un[c] = lane_value((float)tu, lane_of<G>(c));
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                const bool row = (real >> k) & 1;
#pragma unroll
                for (int c = 0; c < G; ++c) q[k][c] += row ? un[c] : 0.0f;
            });
        }
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
#pragma unroll
            for (int c = 0; c < G; ++c) r[k][c] = fmaf(-a[c], q[k][c], r[k][c]);
        });
        if (zeros)
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
#pragma unroll
                for (int c = 0; c < G; ++c)
                    if ((zeros >> lane_of<G>(c)) & 1) r[k][c] = 0.0f;
            });
        double vz[G], vr[G], rz, rr;
#pragma unroll
        for (int c = 0; c < G; ++c) { vz[c] = 0.0; vr[c] = 0.0; }
        precondition(vz, std::false_type());
        norms(vr);
        if (follows && tid == 0) told = lead_word(word, steps + 1, seen, polls);
        block_sum(red2, vz, vr, true, rz, rr);
        // beta = rho' / rho (rho == 0 zeroes p)
        const float be = rho != 0.0 ? (float)(rz / rho) : 0.0f;
        const uint64_t bzeros = __ballot(rho == 0.0 && lane < J.R);
        rho = rz;
        ++steps;
        // stop rules (conjugate_gradient.cpp:118-150): the reference's, sqrt(r.z / b.b) >=
        // FLT_EPSILON, looks at column 0 only and its NaN (b = 0 among others) stops; a NaN
        // residual with a nonzero right-hand side is a breakdown
        bool open;
        if (reference) open = lane == J.col0 && bb > 0.0 && rz >= (double)FLT_EPSILON * (double)FLT_EPSILON * bb;
        else open = lane < J.R && bb > 0.0 && rr > J.tol * J.tol * bb;
        const bool live = __ballot(open) != 0;
        const bool nan = __ballot(lane < J.R && bb > 0.0 && rr != rr) != 0;
        bool stop;
        if (follows) {
            const int v = told;
            late = v < 0;
            stop = late || v == 2 * steps + 1;
        } else if (reference && it.z != lead) stop = steps >= target;
        else {
            stop = (!live && (phase == 0 || steps >= target)) || steps >= J.maxit;
            if (live && steps >= J.maxit) flags = kChipCapped;
        }
        if (nan) { stop = true; flags = kChipNan; }
        if (decides && tid == 0) lead_tell(word, 2 * steps + stop);
        // x += alpha p, p = z + beta p
        float b[G];
#pragma unroll
        for (int c = 0; c < G; ++c) b[c] = lane_value(be, lane_of<G>(c));
        each_row<K>([&](auto kc) __attribute__((always_inline)) {
            constexpr int k = decltype(kc)::value;
            float own[G];
            unpack<G>(ps[tid + k * nt], own);
#pragma unroll
            for (int c = 0; c < G; ++c) {
                x[k][c] = fmaf(a[c], own[c], x[k][c]);
                own[c] = fmaf(b[c], own[c], q[k][c]);
            }
            ps[tid + k * nt] = pack<G>(own);
        });
        if (zeros | bzeros)
            each_row<K>([&](auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                float own[G];
                unpack<G>(ps[tid + k * nt], own);
#pragma unroll
                for (int c = 0; c < G; ++c) {
                    if ((zeros >> lane_of<G>(c)) & 1) x[k][c] = 0.0f;
                    if ((bzeros >> lane_of<G>(c)) & 1) own[c] = 0.0f;
                }
                ps[tid + k * nt] = pack<G>(own);
            });
        __syncthreads();
        if (stop) break;
    }

    // ---- result, and the state from which a later phase goes on -----------------
    const bool keep = !reference || late;
    each_row<K>([&](auto kc) __attribute__((always_inline)) {
        constexpr int k = decltype(kc)::value;
        if (has(k)) {
            const size_t o = (size_t)rowof[tid + k * nt] * Rp;
            float p[G];
            unpack<G>(ps[tid + k * nt], p);
#pragma unroll
            for (int c = 0; c < G; ++c) {
                X[o + c] = x[k][c];
                if (keep) { Rs[o + c] = r[k][c]; Ps[o + c] = p[c]; }
            }
        }
    });
    if (wave == 0 && l < G && keep) {
        sc_ptr(J, SC_RHO, s)[lane] = rho;
        sc_ptr(J, SC_BB, s)[lane] = bb;
    }
    if (tid == 0) gout[me] = make_int2(steps, flags);
}

// --------------------------------------------------------------------------------
// launch wrappers
// --------------------------------------------------------------------------------
static inline void check_launch() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw Error(MPF_EHIP, std::string("kernel launch: ") + hipGetErrorString(e));
}

ChipShape chip_shape(int np, int width, long long lanes) {
    // the largest lane group whose rows fit the registers
    const int fit = np <= 512 * 10 ? 4 : (np <= 512 * 20 ? 2 : 1);
    ChipShape c;
    c.threads = fit == 1 ? 1024 : 512;
    c.G = fit;
    while (c.G > 1 && lanes <= (c.G / 2) * kChipCus) c.G /= 2;
    // few lanes: 1024 threads where 128 VGPRs hold the rows without spills, but one lane of a
    // small mesh takes 512 -- half the wavefronts repeat the scalars, and 256 VGPRs hold the matrix
    // of rows of one 8-slot group.  817 rows: 0.58 ms per call at 1024 threads, 0.49 at 512, 0.42
    // with the matrix held; a 4921-row matrix with 32 columns 0.62, 0.58, 0.54 ms; one
    // Gauss-Newton step of 4921 nodes 3.77, 3.87, 3.72 ms, hence half the rows without it.
    c.hold = c.G == 1 && width == 8 && np <= 512 * 10;
    if (c.G == 1) c.threads = c.hold || np <= 512 * 5 ? 512 : 1024;
    if (c.G == 2 && lanes <= 2 * kChipCus && np <= 1024 * 8) c.threads = 1024;
    const int k = (np + c.threads - 1) / c.threads;
    for (int q : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20})
        if (k <= q) { c.K = q; break; }
    if (c.K == 1) c.threads = np;
    return c;
}

void launch_chip_order(int np, const uint8_t* tpos, uint16_t* rowof, uint16_t* posof, hipStream_t st) {
    k_chip_order<<<np / kTileRows, kTileRows, 0, st>>>(tpos, rowof, posof);
    check_launch();
}

void launch_chip_ids(int np, int width, const int32_t* ids, const uint8_t* gw, const uint16_t* rowof,
                     const uint16_t* posof, uint4* cid, uint8_t* octs, hipStream_t st) {
    k_chip_ids<<<np / 64, 64, 0, st>>>(np, width, ids, gw, rowof, posof, cid, octs);
    check_launch();
}

void launch_chip_pack(const JobDev* d_jobs, const int2* d_js, int njs, int max_np, int* progress, int nprogress,
                      hipStream_t st) {
    MPF_REQUIRE(nprogress <= njs * max_np, "on-chip solver: more lane groups than threads");
    k_chip_pack<<<dim3(max_np / 256, njs), 256, 0, st>>>(d_jobs, d_js, progress, nprogress);
    check_launch();
}

// kernels for MINK..MAXK rows per thread; up to MAXH the matrix may stay in registers
template <int G, int NT, int MINK, int MAXK, int MAXH>
static void chip_dispatch(const JobDev* d_jobs, const int4* d_items, int n, const ChipShape& c, const int2* gin,
                          int2* gout, int* progress, int polls, int phase, hipStream_t st) {
#define MPF_CHIP(k)                                                                                           \
    case k:                                                                                                   \
        if constexpr (k <= MAXH)                                                                              \
            if (c.hold) {                                                                                     \
                k_pcg_chip<G, k, NT, true><<<n, c.threads, 0, st>>>(d_jobs, d_items, gin, gout, progress, polls, phase); \
                return;                                                                                       \
            }                                                                                                 \
        if constexpr (k >= MINK && k <= MAXK) {                                                               \
            k_pcg_chip<G, k, NT, false><<<n, c.threads, 0, st>>>(d_jobs, d_items, gin, gout, progress, polls, phase); \
            return;                                                                                           \
        }                                                                                                     \
        break;
    switch (c.K) {
        MPF_CHIP(1) MPF_CHIP(2) MPF_CHIP(3) MPF_CHIP(4) MPF_CHIP(5) MPF_CHIP(6) MPF_CHIP(8) MPF_CHIP(10)
        MPF_CHIP(12) MPF_CHIP(16) MPF_CHIP(20)
        default: break;
    }
#undef MPF_CHIP
    throw Error(MPF_EINVAL, "on-chip solver: no kernel for this size");
}

void launch_chip(const JobDev* d_jobs, const int4* d_items, int n, const ChipShape& c, const int2* gin, int2* gout,
                 int* progress, int polls, int phase, hipStream_t st) {
    if (!n) return;
    if (c.G == 4) chip_dispatch<4, 512, 1, 10, 0>(d_jobs, d_items, n, c, gin, gout, progress, polls, phase, st);
    else if (c.G == 2 && c.threads <= 512)
        chip_dispatch<2, 512, 1, 20, 0>(d_jobs, d_items, n, c, gin, gout, progress, polls, phase, st);
    else if (c.G == 2) chip_dispatch<2, 1024, 1, 8, 0>(d_jobs, d_items, n, c, gin, gout, progress, polls, phase, st);
    else if (c.threads <= 512)
        chip_dispatch<1, 512, 1, 5, 10>(d_jobs, d_items, n, c, gin, gout, progress, polls, phase, st);
    else chip_dispatch<1, 1024, 3, 20, 0>(d_jobs, d_items, n, c, gin, gout, progress, polls, phase, st);
    check_launch();
}

}  // namespace mpf
