// Two-level PCG with inverse diagonal blocks in place of the inverse diagonal, for the meshes
// that the streaming kernels solve.
//
//   M^-1 = D^-1/2 B D^-1/2 + W Einv W^T
//
// D: the frame's diagonal; B: per 32-row leaf of the node bisection the inverse of the leaf's
// block of D1^-1/2 A(1) D1^-1/2, the unit-diagonal matrix at sigma = 1 -- one set of blocks per
// mesh and harmonic, shared by all frames, no factorisation per frame.  The blocks follow
// the frame's conductivity through D; exact blocks of the frame's matrix need as many
// iterations (measured on an ellipse phantom with contrasts 0.2 to 5).  Conductivities are not
// constrained to be positive: a frame with a negative diagonal entry has no D^-1/2 and takes the
// signed diagonal, by the kernels of the jobs without blocks (the model leaves its bloc null).
//
// Iterations of the coupled electrode model on the 81181-node mesh to 1e-4, harmonics 0-4:
// diagonal 68 / 53 / 44 / 37 / 31, blocks of 16 rows 51 / 35 / 28 / 24 / 20, of 32 48 / 31 / 25 /
// 21 / 18, of 64 48 / 30 / 24 / 20 / 17: 32 rows take nearly all of the gain at half of the
// 64-row blocks' products and bytes.
//
// The update kernel holds the tile's r in LDS in bisection order, wavefront w the w-th
// aggregate: two blocks, each 32 x 32 by 32 x Rp on v_mfma_f32_16x16x4_f32.  A lane's operand
// entries of r and its result entries of z are the same (row, column) pairs, so r.z, r.r and
// W^T r come from registers and z replaces r in LDS.  Bound by memory: q, r read, r, z written
// (one pass more than with the diagonal, whose z the direction kernel forms itself) and 32 KB
// of blocks per tile: 23.8 ms per 32-iteration solve of 32 frames against 23.0 ms for the
// direction kernel's 4.25 passes.  Work lists that run the frames of one (harmonic, tile) back
// to back, to keep its blocks in an XCD's L2, were slower (775 against 742 us per launch: the
// direction kernel's too).
//
// Measured (MI355X, one Gauss-Newton step on the 81181-node mesh, 5 harmonics): slice-iterations
// of 32 frames 11488 -> 6624, 332 -> 227 ms; of one frame 359 -> 207, 16.6 -> 12.2 ms.
#include "blockjac.h"
#include "krylov_dev.h"

namespace mpf {

typedef float v4f __attribute__((ext_vector_type(4)));
static_assert(kBlkRows == 32 && kAggRows == 64, "two 32-row blocks per wavefront's aggregate");

static inline void check_launch() {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) throw Error(MPF_EHIP, std::string("kernel launch: ") + hipGetErrorString(e));
}

// --------------------------------------------------------------------------------
// set-up: one 256-thread workgroup per (block, harmonic), FP64 Gauss-Jordan in LDS
// --------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_block_inverse(const JobDev* __restrict__ jobs, float* __restrict__ bloc,
                                                       int* __restrict__ bad) {
    constexpr int B = kBlkRows;
    const JobDev& J = jobs[0];
    const int np = J.np, s = blockIdx.y, blk = blockIdx.x, per = kTileRows / B;
    const int tile0 = blk / per * kTileRows, b0 = blk % per * B;
    __shared__ double T[B][B + 1];
    __shared__ double d[B];
    for (int i = threadIdx.x; i < B * B; i += 256) T[i / B][i % B] = i / B == i % B ? 1.0 : 0.0;
    __syncthreads();
    // rows of the block: sums of the element contributions (element -1: sigma independent)
    for (int i = threadIdx.x; i < kTileRows; i += 256) {
        const int row = tile0 + i, a = (int)J.tpos[row] - b0;
        if (a < 0 || a >= B || row >= J.n) continue;
        for (int q = 0; q < J.width; ++q) {
            const size_t ent = (size_t)q * np + row;
            const int id = J.ids[ent], c0 = J.ctb_off[ent], c1 = J.ctb_off[ent + 1];
            if (c0 == c1 || id < tile0 || id >= tile0 + kTileRows || id >= J.n) continue;
            const int b = (int)J.tpos[id] - b0;
            if (b < 0 || b >= B) continue;
            double v = 0.0;
            for (int e = c0; e < c1; ++e) v += J.ctb_k[e] + J.alpha64[s] * J.ctb_m[e];
            T[a][b] = v;
        }
    }
    __syncthreads();
    if (threadIdx.x < B) {
        const double v = T[threadIdx.x][threadIdx.x];
        d[threadIdx.x] = v > 0.0 ? sqrt(v) : 0.0;
    }
    __syncthreads();
    for (int k = 0; k < B; ++k) {
        const double p = T[k][k];
        if (!(p > 0.0) && threadIdx.x == 0) atomicOr(bad, 1);
        const double ip = p > 0.0 ? 1.0 / p : 0.0;
        double v[B * B / 256];
#pragma unroll
        for (int u = 0; u < B * B / 256; ++u) {
            const int i = (threadIdx.x + 256 * u) / B, j = threadIdx.x % B;
            const double t = T[i][j];
            v[u] = i == k ? (j == k ? ip : t * ip) : (j == k ? -t * ip : t - T[i][k] * ip * T[k][j]);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < B * B / 256; ++u) T[(threadIdx.x + 256 * u) / B][threadIdx.x % B] = v[u];
        __syncthreads();
    }
    // operand order: fragment (ib, kc) of 16 rows x 16 columns, lane l the row l % 16 and the
    // columns 4 (l / 16) .. + 3
    for (int i = threadIdx.x; i < B * B; i += 256) {
        const int j = i & 3, l = (i >> 2) & 63, f = i >> 8, ib = f >> 1, kc = f & 1;
        const int row = 16 * ib + (l & 15), col = 16 * kc + 4 * (l >> 4) + j;
        // symmetric to the last bit: the mean of both triangles
        const double v = 0.5 * (T[row][col] + T[col][row]) * d[row] * d[col];
        bloc[((size_t)s * gridDim.x + blk) * B * B + i] = (float)v;
    }
}

// --------------------------------------------------------------------------------
// one tile's z = D^-1/2 B D^-1/2 r
// --------------------------------------------------------------------------------
// rs: r of the tile as [place][column], replaced by z; sd: D^-1/2 per place.  Adds r.z, r.r and W^T r
// (FP64) of the lane's entries: columns 16 ct + l % 16 of the wavefront's aggregate.
template <int LG>
struct BlockTile {
    static constexpr int Rp = 1 << LG, CT = Rp / 16, LD = Rp + 4;
    typedef float Rows[kTileRows][LD];
    // the wavefront's 2 x 4 operand fragments
    static __device__ __forceinline__ void load(const JobDev& J, int s, int tile, float4 (&a)[8]) {
        const int wave = threadIdx.x >> 6, l = threadIdx.x & 63;
        const MPF_GLOBAL float4* b = (const MPF_GLOBAL float4*)gp(J.bloc) +
                                     ((size_t)s * (J.np / kBlkRows) + (size_t)tile * 8 + 2 * wave) * 256 + l;
#pragma unroll
        for (int f = 0; f < 8; ++f) a[f] = b[64 * f];
    }
    static __device__ __forceinline__ void apply(Rows& rs, const float* sd, const float4 (&a)[8], double (&rz)[CT],
                                                 double (&rr)[CT], double (&g)[CT]) {
        const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, o = l & 15, q4 = 4 * (l >> 4);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int p0 = wave * kAggRows + b * kBlkRows;
            float rv[2][4][CT], sv[2][4];
#pragma unroll
            for (int kc = 0; kc < 2; ++kc)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int p = p0 + 16 * kc + q4 + j;
                    sv[kc][j] = sd[p];
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) rv[kc][j][ct] = rs[p][16 * ct + o];
                }
            v4f acc[2][CT];
#pragma unroll
            for (int ib = 0; ib < 2; ++ib)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) acc[ib][ct] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kc = 0; kc < 2; ++kc)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float x[CT];
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) x[ct] = sv[kc][j] * rv[kc][j][ct];
#pragma unroll
                    for (int ib = 0; ib < 2; ++ib) {
                        const float4 f = a[4 * b + 2 * ib + kc];
                        const float fv[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
                        for (int ct = 0; ct < CT; ++ct)
                            acc[ib][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(fv[j], x[ct], acc[ib][ct], 0, 0, 0);
                    }
                }
            // result rows 16 ib + q4 + v: the places the operand entries came from
#pragma unroll
            for (int ib = 0; ib < 2; ++ib)
#pragma unroll
                for (int v = 0; v < 4; ++v)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        const float r = rv[ib][v][ct], z = sv[ib][v] * acc[ib][ct][v];
                        rz[ct] += (double)r * (double)z;
                        rr[ct] += (double)r * (double)r;
                        g[ct] += (double)r;
                        rs[p0 + 16 * ib + q4 + v][16 * ct + o] = z;
                    }
        }
    }
    // the wavefronts' sums: rz and rr as the tile's partials of channels c0 and c0 + 1, W^T r of
    // aggregate w in its channel and, scaled, for the coarse kernel
    static __device__ __forceinline__ void sums(const JobDev& J, int s, int tile, int c0, double (&rz)[CT],
                                                double (&rr)[CT], double (&g)[CT], double (*red)[4][Rp]) {
        const int wave = threadIdx.x >> 6, l = threadIdx.x & 63, o = l & 15;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
#pragma unroll
            for (int off = 16; off < 64; off <<= 1) {
                rz[ct] += __shfl_xor(rz[ct], off, 64);
                rr[ct] += __shfl_xor(rr[ct], off, 64);
                g[ct] += __shfl_xor(g[ct], off, 64);
            }
            if (l < 16) {
                const int col = 16 * ct + o, a = kAggPerTile * tile + wave;
                red[0][wave][col] = rz[ct];
                red[1][wave][col] = rr[ct];
                part_ptr(J, agg_channel(wave), s, tile)[col] = g[ct];
                gp(J.cg)[((size_t)s * kAggPerTile * J.ntiles + a) * Rp + col] = (float)((double)J.csc[a] * g[ct]);
            }
        }
        __syncthreads();
        if ((int)threadIdx.x < 2 * Rp) {
            const int c = threadIdx.x / Rp, col = threadIdx.x % Rp;
            double t = 0.0;
#pragma unroll
            for (int w = 0; w < 4; ++w) t += red[c][w][col];
            part_ptr(J, c0 + c, s, tile)[col] = t;
        }
    }
};

// start (k_pcg_init): x = 0, r = b, p = D^-1/2 B D^-1/2 b; partials b.z (channel 0) and b.b (1)
template <int LG>
__global__ void __launch_bounds__(256, 4) k_block_init(const JobDev* __restrict__ jobs, const int4* __restrict__ tiles) {
    typedef BlockTile<LG> BT;
    constexpr int Rp = 1 << LG, LPR = Rp / 4, ROWS = 256 / LPR, PER = kTileRows / ROWS, CT = BT::CT;
    const int4 t = tiles[blockIdx.x];
    const JobDev& J = jobs[t.x];
    if (!J.bloc) return;  // k_pcg_init
    const int s = t.y, tile0 = t.z * kTileRows;
    __shared__ typename BT::Rows rs;
    __shared__ float sd[kTileRows];
    __shared__ double red[2][4][Rp];
    const int c4 = threadIdx.x % LPR, r0 = threadIdx.x / LPR;
    const size_t base = (size_t)s * J.np * LPR;
    MPF_GLOBAL float4* X = (MPF_GLOBAL float4*)gp(J.x) + base;
    MPF_GLOBAL float4* Rr = (MPF_GLOBAL float4*)gp(J.rv) + base;
    MPF_GLOBAL float4* P = (MPF_GLOBAL float4*)gp(J.p) + base;
    float4 a[8];
    BT::load(J, s, t.z, a);
    sd[J.tpos[tile0 + threadIdx.x]] = sqrtf(J.dinv[(size_t)s * J.np + tile0 + threadIdx.x]);
    const float xs = J.xscale[s];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int row = tile0 + r0 + k * ROWS;
        const size_t i = (size_t)row * LPR + c4;
        float b[4];
        if (J.use_rhs) {
            const float4 v = ((const MPF_GLOBAL float4*)gp((const float*)J.rhs) + base)[i];
            b[0] = v.x; b[1] = v.y; b[2] = v.z; b[3] = v.w;
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = (float)(xs * J.F[s * J.fstride + (size_t)row * Rp + 4 * c4 + j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (4 * c4 + j >= J.R) b[j] = 0.0f;
        X[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        Rr[i] = make_float4(b[0], b[1], b[2], b[3]);
        *(float4*)&rs[J.tpos[row]][4 * c4] = make_float4(b[0], b[1], b[2], b[3]);
    }
    __syncthreads();
    double rz[CT], rr[CT], g[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) { rz[ct] = 0.0; rr[ct] = 0.0; g[ct] = 0.0; }
    BT::apply(rs, sd, a, rz, rr, g);
    BT::sums(J, s, t.z, 0, rz, rr, g, red);
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int row = tile0 + r0 + k * ROWS;
        P[(size_t)row * LPR + c4] = *(const float4*)&rs[J.tpos[row]][4 * c4];
    }
}

// update (k_pcg_update4): alpha = rho / p.q, r -= alpha (q + dc), then z into q; tile partials of
// r.z (channel 2), r.r (3) and W^T r.  The tile's loads are all issued before the sums of
// the chunk partials that alpha waits for.
template <int LG>
__global__ void __launch_bounds__(256, 4) k_block_update(const JobDev* __restrict__ jobs,
                                                         const int4* __restrict__ tiles, int iter) {
    typedef BlockTile<LG> BT;
    constexpr int Rp = 1 << LG, LPR = Rp / 4, ROWS = 256 / LPR, PER = kTileRows / ROWS, CT = BT::CT;
    const int par = iter & 1, k4 = iter & (kRing - 1);
    const int4 t = tiles[blockIdx.x];
    const JobDev& J = jobs[t.x];
    if (!J.bloc) return;  // k_pcg_update4
    const int s = t.y, tile0 = t.z * kTileRows;
    const bool live = slice_active(J, s);
    if (t.z == 0 && threadIdx.x == 0) J.st[s * kStInts + 3] = live ? 1 : 0;
    if (!live) return;
    __shared__ typename BT::Rows rs;
    __shared__ float sd[kTileRows];
    __shared__ double red[2][4][Rp];
    const int c4 = threadIdx.x % LPR, r0 = threadIdx.x / LPR;
    const size_t base = (size_t)s * J.np * LPR;
    MPF_GLOBAL float4* Q = (MPF_GLOBAL float4*)gp(J.q) + base;
    MPF_GLOBAL float4* Rr = (MPF_GLOBAL float4*)gp(J.rv) + base;
    float4 q4[PER], rv[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const size_t i = (size_t)(tile0 + r0 + k * ROWS) * LPR + c4;
        q4[k] = Q[i];
        rv[k] = Rr[i];
    }
    sd[J.tpos[tile0 + threadIdx.x]] = sqrtf(gp((const float*)J.dinv)[(size_t)s * J.np + tile0 + threadIdx.x]);
    // p.q and 1^T p arrive as one partial per kChunkTiles-tile chunk (k_pcg_chunks), summed by
    // every block in the same order; the buffers share LDS with r
    double* acc = reinterpret_cast<double*>(&rs[0][0]);        // [2][256 / Rp][Rp], then the results
    {
        constexpr int NG = 256 / Rp;
        const int cnt = coarse_chunks(J), lane = threadIdx.x & (Rp - 1), gr = threadIdx.x >> LG;
        const bool dc = s == J.dc;
        double u = 0.0, v = 0.0;
#pragma unroll 4
        for (int c = gr; c < cnt; c += NG) {
            u += part_ptr(J, 5, s, c)[lane];
            if (dc) v += part_ptr(J, 6, s, c)[lane];
        }
        acc[threadIdx.x] = u;
        acc[256 + threadIdx.x] = v;
        __syncthreads();
        if ((int)threadIdx.x < Rp) {
            double pq = 0.0, ps = 0.0;
#pragma unroll
            for (int c = 0; c < NG; ++c) { pq += acc[c * Rp + lane]; ps += acc[256 + c * Rp + lane]; }
            pq += ps * ps;
            const double al = pq != 0.0 ? sc_ptr(J, rho_slot(par), s)[lane] / pq : 0.0;
            float* res = reinterpret_cast<float*>(acc + 512);
            res[lane] = (float)al;
            res[Rp + lane] = (float)ps;
            res[2 * Rp + lane] = pq == 0.0 ? 1.0f : 0.0f;
            if (t.z == 0) {
                sc_ptr(J, SC_PQ0 + k4, s)[lane] = pq;
                sc_ptr(J, SC_PSUM, s)[lane] = ps;
                sc_ptr(J, SC_PA0 + k4, s)[lane] = al;
            }
        }
        __syncthreads();
    }
    float a4[4], dcv[4];
    bool zero[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int col = 4 * c4 + j;
        const float* res = reinterpret_cast<const float*>(acc + 512);
        a4[j] = res[col];
        dcv[j] = res[Rp + col];
        zero[j] = res[2 * Rp + col] != 0.0f;
    }
    __syncthreads();       // read before r takes their place
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int row = tile0 + r0 + k * ROWS;
        const float dc = row < J.n ? 1.0f : 0.0f;
        const float qv[4] = {q4[k].x, q4[k].y, q4[k].z, q4[k].w};
        float o[4] = {rv[k].x, rv[k].y, rv[k].z, rv[k].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = zero[j] ? 0.0f : o[j] - a4[j] * (qv[j] + dc * dcv[j]);
        const float4 n = make_float4(o[0], o[1], o[2], o[3]);
        Rr[(size_t)row * LPR + c4] = n;
        *(float4*)&rs[J.tpos[row]][4 * c4] = n;
    }
    float4 a[8];
    BT::load(J, s, t.z, a);
    __syncthreads();
    double rz[CT], rr[CT], g[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) { rz[ct] = 0.0; rr[ct] = 0.0; g[ct] = 0.0; }
    BT::apply(rs, sd, a, rz, rr, g);
    BT::sums(J, s, t.z, 2, rz, rr, g, red);
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int row = tile0 + r0 + k * ROWS;
        Q[(size_t)row * LPR + c4] = *(const float4*)&rs[J.tpos[row]][4 * c4];
    }
}

void launch_block_inverse(const JobDev* d_jobs, int C, int np, float* bloc, int* bad, hipStream_t st) {
    k_block_inverse<<<dim3(np / kBlkRows, C), 256, 0, st>>>(d_jobs, bloc, bad);
    check_launch();
}

void launch_block_init(const JobDev* d_jobs, const int4* d_tiles, int ntiles, int lg, hipStream_t st) {
    if (lg == 6) k_block_init<6><<<ntiles, 256, 0, st>>>(d_jobs, d_tiles);
    else if (lg == 5) k_block_init<5><<<ntiles, 256, 0, st>>>(d_jobs, d_tiles);
    else k_block_init<4><<<ntiles, 256, 0, st>>>(d_jobs, d_tiles);
    check_launch();
}

void launch_block_update(const JobDev* d_jobs, const int4* d_tiles, int ntiles, int iter, int lg, hipStream_t st) {
    if (lg == 6) k_block_update<6><<<ntiles, 256, 0, st>>>(d_jobs, d_tiles, iter);
    else if (lg == 5) k_block_update<5><<<ntiles, 256, 0, st>>>(d_jobs, d_tiles, iter);
    else k_block_update<4><<<ntiles, 256, 0, st>>>(d_jobs, d_tiles, iter);
    check_launch();
}

}  // namespace mpf
