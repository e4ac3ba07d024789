// Krylov driver (see krylov.h).
//
// ConjugateGradient::solve / BiCGSTAB::solve (src/numeric/conjugate_gradient.cpp:61-161,
// src/numeric/bicgstab.cpp:83-193) copy the residual matrix to the host and synchronise
// after every iteration, for one harmonic of one frame at a time.  Here all (job,
// harmonic) pairs iterate in the same launches; the host polls the device state every
// `check_every` iterations and then drops converged pairs from the work lists.  With
// opts.graphs the iterations between polls are captured once as a HIP graph and replayed
// while the lists do not change (lists are compacted only when a quarter of their tiles
// belong to finished pairs).
#include "krylov.h"

#include <algorithm>
#include <cstring>

#include "blockjac.h"
#include "model.h"

namespace mpf {

constexpr int kXcds = 8;

// Workgroups are dispatched round-robin over the XCDs (block b runs on XCD b % 8), and
// each XCD has its own L2.  Reorder a work list so that XCD x receives a contiguous run
// of consecutive tiles: neighbouring rows gathered by the SpMV then hit the same L2.
void xcd_order(const int4* in, int n, int4* out) {
    const int base = n / kXcds, extra = n % kXcds;
    int start[kXcds + 1];
    start[0] = 0;
    for (int x = 0; x < kXcds; ++x) start[x + 1] = start[x] + base + (x < extra ? 1 : 0);
    for (int b = 0; b < n; ++b) out[b] = in[start[b % kXcds] + b / kXcds];
}

KrylovDriver::KrylovDriver(mpf_ctx* c, std::vector<std::vector<JobDev>*> sources)
    : ctx(c), src(std::move(sources)) {
    for (size_t m = 0; m < src.size(); ++m)
        for (size_t f = 0; f < src[m]->size(); ++f) {
            origin.emplace_back((int)m, (int)f);
            h.push_back((*src[m])[f]);
        }
    const int nj = (int)h.size();
    MPF_REQUIRE(nj > 0, "krylov: no jobs");
    jobs.alloc(nj);
    st.alloc((size_t)nj * kMaxSlices * kStInts);
    active.alloc(1);
    hipStream_t s0 = ctx->stream;
    MPF_HIP(hipMemsetAsync(st.p, 0, st.bytes(), s0));
    // groups by (lane count, padded width)
    std::vector<int4> all_tiles, str_tiles;
    std::vector<int2> all_js, str_js;
    for (int j = 0; j < nj; ++j) {
        const JobDev& J = h[j];
        const bool chip = J.np <= kChipMaxRows && J.width <= kChipMaxWidth && J.gw;
        Group* g = nullptr;
        for (auto& q : groups)
            if (q.lg == J.lg && q.wpad == J.width && q.chip == chip) g = &q;
        if (!g) {
            groups.emplace_back();
            g = &groups.back();
            g->lg = J.lg;
            g->wpad = J.width;
            g->chip = chip;
        }
        g->jobs.push_back(j);
        // the 128-bit gather kernels keep byte offsets of a slice vector in 31 bits
        if ((long long)J.np * J.Rp * 4 >= (1LL << 31) - (1LL << 16)) g->wide = true;
        for (int c = 0; c < J.C; ++c) {
            all_js.push_back(make_int2(j, c));
            for (int t = 0; t < J.ntiles; ++t) all_tiles.push_back(make_int4(j, c, t, 0));
            if (chip) continue;
            str_js.push_back(make_int2(j, c));
            for (int t = 0; t < J.ntiles; ++t) str_tiles.push_back(make_int4(j, c, t, 0));
        }
    }
    size_t total = 0;
    for (auto& g : groups) {
        std::vector<int4> lst, lst_t, flst;
        std::vector<int2> gjs;
        long long rows = 0;
        for (int j : g.jobs) {
            for (int c = 0; c < h[j].C; ++c) {
                gjs.push_back(make_int2(j, c));
                for (int t = 0; t < h[j].ntiles; ++t) lst.push_back(make_int4(j, c, t, 0));
            }
            for (int t = 0; t < h[j].ntiles; ++t) {
                for (int c = 0; c < h[j].C; ++c) lst_t.push_back(make_int4(j, c, t, 0));
                flst.push_back(make_int4(j, 0, t, 0));
            }
            rows += (long long)h[j].C * h[j].np;
            g.nchunk = std::max(g.nchunk, (h[j].ntiles + kChunkTiles - 1) / kChunkTiles);
            if (h[j].cinv) init_nchunk = std::max(init_nchunk, g.nchunk);
        }
        g.njs = (int)gjs.size();
        g.js.alloc(g.njs);
        g.js.upload(gjs.data(), gjs.size(), s0);
        g.nall = (int)lst.size();
        const std::vector<int4>* src_o[2] = {&lst, &lst_t};
        for (int o = 0; o < 2; ++o) {
            g.base_o[o] = *src_o[o];
            g.all_o[o].resize(lst.size());
            xcd_order(src_o[o]->data(), g.nall, g.all_o[o].data());
            g.tiles_o[o].alloc(g.nall);
            g.tiles_o[o].upload(g.all_o[o].data(), g.all_o[o].size(), s0);
        }
        g.act.alloc(g.nall);
        g.hoff = total;
        total += g.nall;
        g.nfall = (int)flst.size();
        g.fbase = flst;
        g.fall.resize(flst.size());
        xcd_order(flst.data(), g.nfall, g.fall.data());
        g.ftiles.alloc(g.nfall);
        g.ftiles.upload(g.fall.data(), g.fall.size(), s0);
        g.fact.alloc(g.nfall);
        g.fhoff = total;
        total += g.nfall;
        // autotune key: lane count, width, and the power-of-two bucket of the rows per
        // launch (small launches favour different kernels than large ones)
        int bucket = 0;
        while ((1LL << bucket) < rows) ++bucket;
        g.key = ((long long)g.lg << 40) | ((long long)g.wpad << 32) | bucket;
    }
    n_init_tiles = (int)all_tiles.size();
    n_init_js = (int)all_js.size();
    std::vector<int4> ordered(all_tiles.size());
    xcd_order(all_tiles.data(), n_init_tiles, ordered.data());
    init_tiles.alloc(n_init_tiles);
    init_tiles.upload(ordered.data(), ordered.size(), s0);
    init_js.alloc(n_init_js);
    init_js.upload(all_js.data(), all_js.size(), s0);
    n_stream_tiles = (int)str_tiles.size();
    n_stream_js = (int)str_js.size();
    if (n_stream_js) {
        std::vector<int4> so(str_tiles.size());
        xcd_order(str_tiles.data(), n_stream_tiles, so.data());
        stream_tiles.alloc(n_stream_tiles);
        stream_tiles.upload(so.data(), so.size(), s0);
        stream_js.alloc(n_stream_js);
        stream_js.upload(str_js.data(), str_js.size(), s0);
        MPF_HIP(hipStreamSynchronize(s0));   // so goes out of scope
    }
    MPF_HIP(hipHostMalloc((void**)&h_active, sizeof(int), hipHostMallocDefault));
    MPF_HIP(hipHostMalloc((void**)&h_st, st.bytes(), hipHostMallocDefault));
    std::memset(h_st, 0, st.bytes());
    h_tiles_cap = total;
    MPF_HIP(hipHostMalloc((void**)&h_tiles, sizeof(int4) * h_tiles_cap, hipHostMallocDefault));
    MPF_HIP(hipStreamSynchronize(s0));
}

KrylovDriver::~KrylovDriver() {
    drop_graph();
    if (cap) (void)hipStreamDestroy(cap);
    if (h_active) (void)hipHostFree(h_active);
    if (h_st) (void)hipHostFree(h_st);
    if (h_tiles) (void)hipHostFree(h_tiles);
    drop_chip();
}

// the on-chip solver's tables, streams and events
void KrylovDriver::drop_chip() {
    if (h_gst) (void)hipHostFree(h_gst);
    for (auto& c : chips) {
        if (c.done) (void)hipEventDestroy(c.done);
        if (c.stream) (void)hipStreamDestroy(c.stream);
    }
    if (chip_fork) (void)hipEventDestroy(chip_fork);
    h_gst = nullptr;
    chip_fork = nullptr;
    chips.clear();
    chip_meshes.clear();
    cval.release(); chip_js.release(); progress.release();
    for (auto& g : gst) g.release();
}

// Tables of the on-chip PCG (chip.hip), once per driver: the chip order and 16-bit matrix of
// every mesh, room for the values of every (job, slice), and the work items per class.
bool KrylovDriver::ensure_chip() {
    if (chip_tried) return chip_ok;
    chip_tried = true;
    const int nj = (int)h.size();
    chip_mesh_of.assign(nj, -1);
    cval_off.assign(nj, 0);
    std::vector<int> jobs_on;
    for (const auto& g : groups)
        if (g.chip) jobs_on.insert(jobs_on.end(), g.jobs.begin(), g.jobs.end());
    if (jobs_on.empty()) return false;
    std::sort(jobs_on.begin(), jobs_on.end());
    hipStream_t s0 = ctx->stream;
    try {
        size_t nval = 0;
        for (int j : jobs_on) {
            const JobDev& J = h[j];
            int m = -1;
            for (size_t i = 0; i < chip_meshes.size(); ++i)
                if (chip_meshes[i]->ids == J.ids) m = (int)i;
            if (m < 0) {
                m = (int)chip_meshes.size();
                chip_meshes.emplace_back(new ChipMesh);
                ChipMesh& M = *chip_meshes.back();
                M.ids = J.ids;
                M.crow.alloc(J.np);
                M.cpos.alloc(J.np);
                M.cid.alloc((size_t)J.width / 8 * J.np);
                M.octs.alloc(J.np / 64);
                launch_chip_order(J.np, J.tpos, M.crow.p, M.cpos.p, s0);
                launch_chip_ids(J.np, J.width, J.ids, J.gw, M.crow.p, M.cpos.p, M.cid.p, M.octs.p, s0);
            }
            chip_mesh_of[j] = m;
            cval_off[j] = nval;
            nval += (size_t)J.C * J.width / 4 * J.np;
            chip_max_np = std::max(chip_max_np, J.np);
        }
        cval.alloc(nval);
        long long lanes = 0;
        for (int j : jobs_on) lanes += (long long)h[j].C * h[j].R;
        // the longest pairs (low harmonics) first
        int total = 0, cmax = 0;
        for (int j : jobs_on) cmax = std::max(cmax, h[j].C);
        for (int c = 0; c < cmax; ++c)
            for (int j : jobs_on) {
                const JobDev& J = h[j];
                if (c >= J.C) continue;
                const ChipShape sh = chip_shape(J.np, J.width, lanes);
                ChipClass* cl = nullptr;
                for (auto& q : chips)
                    if (q.shape.G == sh.G && q.shape.K == sh.K && q.shape.threads == sh.threads &&
                        q.shape.hold == sh.hold)
                        cl = &q;
                if (!cl) {
                    chips.emplace_back();
                    cl = &chips.back();
                    cl->shape = sh;
                }
                h_chip_js.push_back(make_int2(j, c));
                chip_first.push_back(total);
                for (int g = 0; g < J.Rp / sh.G; ++g) cl->h_items.push_back(make_int4(j, c, g, total));
                total += J.Rp / sh.G;
            }
        // the groups of a pair on one XCD (block b runs on XCD b % 8), which then reads the
        // pair's matrix into its L2 once: pair i goes to XCD i % 8
        for (auto& cl : chips) {
            std::vector<std::vector<int4>> on(kXcds);
            int pairs = -1, last = -1;
            for (const int4& it : cl.h_items) {
                if (it.w != last) { ++pairs; last = it.w; }
                on[pairs % kXcds].push_back(it);
            }
            cl.h_items.clear();
            size_t longest = 0;          // pairs of 16 and of 32 lanes have different group counts
            for (const auto& x : on) longest = std::max(longest, x.size());
            for (size_t i = 0; i < longest; ++i)
                for (const auto& x : on)
                    if (i < x.size()) cl.h_items.push_back(x[i]);
        }
        chip_first.push_back(total);
        size_t listed = 0;
        for (const auto& cl : chips) listed += cl.h_items.size();
        MPF_REQUIRE((int)listed == total, "krylov: on-chip work list incomplete");
        std::sort(chips.begin(), chips.end(), [](const ChipClass& a, const ChipClass& b) {
            return a.shape.K * a.shape.threads > b.shape.K * b.shape.threads;
        });
        for (size_t i = 0; i < chips.size(); ++i) {
            ChipClass& c = chips[i];
            c.items.alloc(c.h_items.size());
            c.items.upload(c.h_items.data(), c.h_items.size(), s0);
            if (i == 0) continue;
            MPF_HIP(hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking));
            MPF_HIP(hipEventCreateWithFlags(&c.done, hipEventDisableTiming));
        }
        if (chips.size() > 1) MPF_HIP(hipEventCreateWithFlags(&chip_fork, hipEventDisableTiming));
        chip_js.alloc(h_chip_js.size());
        chip_js.upload(h_chip_js.data(), h_chip_js.size(), s0);
        gst[0].alloc(total);
        gst[1].alloc(total);
        progress.alloc(total);
        MPF_HIP(hipMemsetAsync(gst[0].p, 0, gst[0].bytes(), s0));
        MPF_HIP(hipMemsetAsync(gst[1].p, 0, gst[1].bytes(), s0));
        h_gst = pinned_alloc<int2>(total);
        MPF_HIP(hipStreamSynchronize(s0));
    } catch (const Error& e) {
        if (e.code != MPF_ENOMEM) throw;
        // no room for the tables: the jobs are streamed
        drop_chip();
        return false;
    }
    chip_ok = true;
    return true;
}

// One solve of every on-chip pair: phase 0, then phase 1 until the lane groups of every pair
// have taken the same number of steps (usually once: it takes every group on to the step at
// which the pair's slowest group stopped).  Step counts and flags go to h_st.
void KrylovDriver::run_chip() {
    hipStream_t s0 = ctx->stream;
    const int total = chip_first.back();
    launch_chip_pack(jobs.p, chip_js.p, (int)h_chip_js.size(), chip_max_np, progress.p, total, s0);
    auto phase = [&](int ph, int in) {
        if (chips.size() > 1) MPF_HIP(hipEventRecord(chip_fork, s0));
        for (auto& c : chips) {
            hipStream_t s = c.stream ? c.stream : s0;
            if (c.stream) MPF_HIP(hipStreamWaitEvent(s, chip_fork, 0));
            launch_chip(jobs.p, c.items.p, (int)c.h_items.size(), c.shape, gst[in].p, gst[in ^ 1].p, progress.p,
                        ctx->lead_polls, ph, s);
            if (c.stream) {
                MPF_HIP(hipEventRecord(c.done, s));
                MPF_HIP(hipStreamWaitEvent(s0, c.done, 0));
            }
        }
    };
    phase(0, 1);
    int in = 0;
    for (bool open = true; open;) {
        phase(1, in);
        in ^= 1;
        MPF_HIP(hipMemcpyAsync(h_gst, gst[in].p, sizeof(int2) * total, hipMemcpyDeviceToHost, s0));
        MPF_HIP(hipStreamSynchronize(s0));
        open = false;
        for (size_t i = 0; i < h_chip_js.size() && !open; ++i) {
            int steps = 0;
            for (int g = chip_first[i]; g < chip_first[i + 1]; ++g) steps = std::max(steps, h_gst[g].x);
            for (int g = chip_first[i]; g < chip_first[i + 1]; ++g)
                if (!h_gst[g].y && h_gst[g].x != steps) open = true;
        }
    }
    for (size_t i = 0; i < h_chip_js.size(); ++i) {
        int steps = 0, flags = 0;
        for (int g = chip_first[i]; g < chip_first[i + 1]; ++g) {
            steps = std::max(steps, h_gst[g].x);
            flags |= h_gst[g].y & (kChipCapped | kChipNan);
        }
        int* sp = &h_st[((size_t)h_chip_js[i].x * kMaxSlices + h_chip_js[i].y) * kStInts];
        sp[0] = 0;
        sp[1] = steps;
        sp[2] = flags ? 1 : 0;
    }
}

void KrylovDriver::drop_graph() {
    if (gexec) (void)hipGraphExecDestroy(gexec);
    gexec = nullptr;
}

void KrylovDriver::launch_group_iter(Group& g, int iter, bool bicg, hipStream_t s, hipEvent_t e0,
                                     hipEvent_t e1) {
    if (g.ncur == 0) return;
    if (bicg)
        launch_bicg_iter(jobs.p, g.cur, g.ncur, active.p, iter, g.lg, g.wpad, s, e0, e1);
    else
        launch_pcg_iter(jobs.p, g.cur, g.ncur, active.p, iter, g.lg, g.wpad, g.variant, s, e0, e1, g.js.p, g.njs,
                        g.nchunk, g.fcur, g.nfcur, g.upd);
}

// Time each SpMV candidate that supports the group's width on the live job data (the
// SpMV only writes q and the SpMV partials, which the next iteration recomputes) and keep
// the fastest in the context's cache.  Candidates: the 128-bit gather kernel over
// (job, slice, tile) and over (job, tile, slice) work lists (in the second, the harmonics
// of one tile run back to back on one XCD and share its L2 copy of the tile's matrix),
// the 32-bit gather kernel, and the harmonic-fused kernel over (job, tile).
void KrylovDriver::tune(Group& g) {
    int choice = -1;
    {
        std::lock_guard<std::mutex> lk(ctx->tune.mu);
        auto it = ctx->tune.spmv.find(g.key);
        if (it != ctx->tune.spmv.end()) choice = it->second;
    }
    if (choice < 0) {
        hipStream_t s0 = ctx->stream;
        hipEvent_t a, b;
        MPF_HIP(hipEventCreate(&a));
        MPF_HIP(hipEventCreate(&b));
        float best = 1e30f;
        choice = g.wpad <= 24 && !g.wide ? 0 : 1;
        const int cand[4][2] = {{0, 0}, {0, 1}, {1, 0}, {2, 0}};
        for (const auto& c : cand) {
            const int v = c[0], o = c[1];
            if (v != 1 && (g.wpad > 24 || g.wide)) continue;
            const int4* lst = v == 2 ? g.ftiles.p : g.tiles_o[o].p;
            const int n = v == 2 ? g.nfall : g.nall;
            launch_pcg_spmv(jobs.p, lst, n, g.lg, g.wpad, v, s0);   // warm-up
            MPF_HIP(hipEventRecord(a, s0));
            for (int r = 0; r < 8; ++r) launch_pcg_spmv(jobs.p, lst, n, g.lg, g.wpad, v, s0);
            MPF_HIP(hipEventRecord(b, s0));
            MPF_HIP(hipEventSynchronize(b));
            float ms = 0.0f;
            MPF_HIP(hipEventElapsedTime(&ms, a, b));
            if (ms < best) { best = ms; choice = v | (o << 4); }
        }
        (void)hipEventDestroy(a);
        (void)hipEventDestroy(b);
        std::lock_guard<std::mutex> lk(ctx->tune.mu);
        ctx->tune.spmv[g.key] = choice;
    }
    g.variant = choice & 15;
    g.order = choice >> 4;
}

// whether every group's SpMV choice is in the context's cache
bool KrylovDriver::tuned() {
    std::lock_guard<std::mutex> lk(ctx->tune.mu);
    for (const auto& g : groups)
        if (!ctx->tune.spmv.count(g.key)) return false;
    return true;
}

bool KrylovDriver::run(const mpf_solve_opts& o, int rule, double tol, bool use_rhs, bool ref_b,
                       mpf_solve_stats* stats) {
    hipStream_t s0 = ctx->stream;
    const bool bicg = o.krylov == MPF_KRYLOV_BICGSTAB;
    const int nj = (int)h.size();
    // the two-level preconditioner (jobs with a coarse level; CG only)
    const bool want_coarse = !bicg && o.preconditioner == MPF_PRECOND_TWO_LEVEL;
    if (want_coarse != coarse) drop_graph();
    coarse = want_coarse && init_nchunk > 0;
    // small meshes run on chip; profiled runs stream, their SpMV launches are what is timed
    const bool chip = !bicg && !ctx->prof && ensure_chip();
    for (int j = 0; j < nj; ++j) {
        JobDev& J = h[j];
        J = (*src[origin[j].first])[origin[j].second];
        if (!coarse) J.cinv = nullptr;
        if (!J.cinv) J.bloc = nullptr;
        J.st = st.p + (size_t)j * kMaxSlices * kStInts;
        J.rule = rule;
        J.tol = tol;
        J.maxit = o.max_iter > 0 ? o.max_iter : 10 * J.n;
        J.use_rhs = use_rhs ? 1 : 0;
        J.ref_b = ref_b ? 1 : 0;
        if (chip && chip_mesh_of[j] >= 0) {
            const ChipMesh& M = *chip_meshes[chip_mesh_of[j]];
            J.crow = M.crow.p;
            J.cid = M.cid.p;
            J.cocts = M.octs.p;
            J.cval = cval.p + cval_off[j];
        }
    }
    for (auto& g : groups) {
        size_t with = 0;
        for (int j : g.jobs) with += h[j].bloc != nullptr;
        g.upd = with == 0 ? kUpdDiagonal : (with == g.jobs.size() ? kUpdBlocks : kUpdBoth);
    }
    jobs.upload(h.data(), h.size(), s0);
    MPF_HIP(hipMemsetAsync(active.p, 0, sizeof(int), s0));
    // the start: jobs with inverse blocks by their own kernel, the others by k_pcg_init
    auto start = [&](const int4* lt, int nt, const int2* lj, int nj2) {
        for (auto& g : groups)
            if (g.upd != kUpdDiagonal) launch_block_init(jobs.p, g.tiles_o[0].p, g.nall, g.lg, s0);
        launch_pcg_init(jobs.p, lt, nt, lj, nj2, active.p, s0, coarse ? init_nchunk : 0);
    };
    const int4* itiles = chip ? stream_tiles.p : init_tiles.p;
    const int2* ijs = chip ? stream_js.p : init_js.p;
    const int nit = chip ? n_stream_tiles : n_init_tiles, nij = chip ? n_stream_js : n_init_js;
    if (bicg) {
        launch_bicg_init(jobs.p, init_tiles.p, n_init_tiles, init_js.p, n_init_js, active.p, 0, s0);
    } else {
        if (chip && !tuned()) {
            // the candidates are timed on initialised pairs, streamed or not
            start(init_tiles.p, n_init_tiles, init_js.p, n_init_js);
            for (auto& g : groups) tune(g);
            MPF_HIP(hipMemsetAsync(active.p, 0, sizeof(int), s0));
        }
        if (nij) start(itiles, nit, ijs, nij);
    }
    for (auto& g : groups) {
        if (!bicg) tune(g);
        else g.order = 0;
        g.cur = g.tiles_o[g.order].p;
        g.ncur = chip && g.chip ? 0 : g.nall;
        g.fcur = g.ftiles.p;
        g.nfcur = g.nfall;
    }
    int every = o.check_every > 0 ? o.check_every : 16;
    every = (every + kRing - 1) / kRing * kRing;   // whole direction-ring cycles per poll
    const bool graphs = o.graphs != 0 && !ctx->prof;
    int maxit = 0;
    for (const auto& J : h) maxit = std::max(maxit, J.maxit);
    drop_graph();
    int it = 0;
    while (nij > 0 || bicg) {
        if (graphs) {
            if (!gexec || gbicg != bicg || gevery != every) {
                drop_graph();
                if (!cap) MPF_HIP(hipStreamCreateWithFlags(&cap, hipStreamNonBlocking));
                hipGraph_t graph;
                MPF_HIP(hipStreamBeginCapture(cap, hipStreamCaptureModeThreadLocal));
                for (int i = 0; i < every; ++i)
                    for (auto& g : groups) launch_group_iter(g, i, bicg, cap, nullptr, nullptr);
                MPF_HIP(hipStreamEndCapture(cap, &graph));
                const hipError_t e = hipGraphInstantiate(&gexec, graph, nullptr, nullptr, 0);
                (void)hipGraphDestroy(graph);
                MPF_HIP(e);
                gbicg = bicg;
                gevery = every;
            }
            MPF_HIP(hipGraphLaunch(gexec, s0));
        } else {
            for (int i = 0; i < every; ++i)
                for (auto& g : groups) {
                    std::pair<hipEvent_t, hipEvent_t> ev{nullptr, nullptr};
                    if (ctx->prof && g.ncur) ev = ctx->next_events();
                    launch_group_iter(g, it + i, bicg, s0, ev.first, ev.second);
                }
        }
        it += every;
        MPF_HIP(hipMemcpyAsync(h_active, active.p, sizeof(int), hipMemcpyDeviceToHost, s0));
        MPF_HIP(hipMemcpyAsync(h_st, st.p, st.bytes(), hipMemcpyDeviceToHost, s0));
        MPF_HIP(hipStreamSynchronize(s0));
        if (ctx->prof) ctx->collect_events();
        if (*h_active <= 0 || it >= maxit + every) break;
        // compact the work lists: always without graphs, otherwise once a quarter of the
        // listed tiles belong to finished pairs (finished pairs' blocks exit at once)
        for (auto& g : groups) {
            if (chip && g.chip) continue;
            // the survivors in (job, slice, tile) or (job, tile, slice) order (a filter of
            // the unstriped list keeps its order), then striped over the XCDs again so that
            // XCD x gets a contiguous run of them
            std::vector<int4> un;
            un.reserve(g.ncur);
            for (const int4& t : g.base_o[g.order])
                if (h_st[((size_t)t.x * kMaxSlices + t.y) * kStInts]) un.push_back(t);
            const int nt = (int)un.size();
            if (nt == g.ncur) continue;
            if (graphs && nt * 4 > g.ncur * 3 && nt > 0) continue;
            int4* ordered = h_tiles + g.hoff;
            xcd_order(un.data(), nt, ordered);
            if (nt) MPF_HIP(hipMemcpyAsync(g.act.p, ordered, sizeof(int4) * nt, hipMemcpyHostToDevice, s0));
            // the group's staging region is rewritten only after the next poll's
            // synchronisation
            g.cur = g.act.p;
            g.ncur = nt;
            // the fused SpMV's (job, tile) items: jobs with a live harmonic
            std::vector<int4> fun;
            fun.reserve(g.nfall);
            for (const int4& t : g.fbase) {
                bool live = false;
                for (int c = 0; c < h[t.x].C; ++c) live = live || h_st[((size_t)t.x * kMaxSlices + c) * kStInts];
                if (live) fun.push_back(t);
            }
            const int nf = (int)fun.size();
            int4* fordered = h_tiles + g.fhoff;
            xcd_order(fun.data(), nf, fordered);
            if (nf) MPF_HIP(hipMemcpyAsync(g.fact.p, fordered, sizeof(int4) * nf, hipMemcpyHostToDevice, s0));
            g.fcur = g.fact.p;
            g.nfcur = nf;
            drop_graph();
        }
    }
    drop_graph();
    if (!bicg && nij) launch_pcg_flush(jobs.p, itiles, nit, s0);
    if (chip) run_chip();
    bool capped = false;
    int64_t slice_iters = 0;
    double bytes = 0.0;
    for (int j = 0; j < nj; ++j)
        for (int c = 0; c < h[j].C; ++c) {
            const int* sp = &h_st[((size_t)j * kMaxSlices + c) * kStInts];
            slice_iters += sp[1];
            if (stats) {
                stats->steps += sp[1];
                stats->max_steps = std::max<int64_t>(stats->max_steps, sp[1]);
                stats->not_converged += sp[2];
            }
            if (sp[2]) capped = true;
            // algorithmic bytes of one harmonic's SpMV with R right-hand sides: A_c values
            // and column ids once, p read and q written once
            bytes += (double)sp[1] * (8.0 * h[j].nnz + 8.0 * h[j].n * h[j].R);
        }
    if (ctx->prof) ctx->prof_bytes += bytes;
    (void)slice_iters;
    return capped;
}

}  // namespace mpf
