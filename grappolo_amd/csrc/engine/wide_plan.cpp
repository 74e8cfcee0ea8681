// wide_plan.cpp -- the work items of the whole-GPU persistent sweep (see
// wide.hpp), built on the host once per phase from the (degree bin, color)
// grouping of the vertices.
#include <sched.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <new>

#include "host_workers.hpp"
#include "louvain.hpp"
#include "wide.hpp"

namespace glv {

// The items of one color class (giant indices local to the class; the
// giants' pair and count offsets relative to the class).
struct ClassPlan {
    std::vector<WideItem> wi;         // workgroup items, then per workgroup their bounds
    std::vector<i64> wstart, pstart;  // per workgroup, nb + 1 each
    std::vector<int2> pi;             // giant partitions
    std::vector<WideRow> extra;       // the mid vertices of bin 7
    std::vector<int32_t> rank;        // per workgroup
    std::vector<WideGiant> giants;
    int groups = 0;
    i64 items = 0;  // wavefront items
    i64 pairs = 0, counts = 0, parts = 1;
    bool ok = true;
};

// rows: the vertices of bins 7 .. 9, from position hlo on.  The dealing
// starts at another workgroup of the grid for each class (`turn`): the one that
// ends a step last, with the costliest item, is still reading ahead when the
// others leave the barrier, and must not be the one they wait for again.
static void plan_class(const PhaseSetup &P, const std::vector<WideRow> &rows, i64 hlo, int c, int nb,
                       ClassPlan &out) {
    std::vector<WideItem> cls;  // the workgroup items of the class: giants' chunks, heavy vertices
    std::vector<WideGiant> &giants = out.giants;
    i64 pairs = 0, counts = 0;
    for (int b = 8; b < kNumBins; b++)
        for (i64 q = P.lo(b, c); q < P.hi(b, c); q++) {
            const WideRow &r = rows[q - hlo];
            const i64 d = r.deg;
            if (d <= kWHeavyMaxDeg) continue;
            WideGiant G;
            G.v = r.v;
            G.nchunks = (int32_t)((d + kWChunk - 1) / kWChunk);
            if (G.nchunks > kWMaxChunks) {
                out.ok = false;
                return;
            }
            G.nparts = (int32_t)std::min<i64>(kWMaxParts, std::max<i64>(1, (d + kWPartKeys - 1) / kWPartKeys));
            G.pairs = pairs;
            G.cnt = counts;
            pairs += (i64)G.nchunks * kWChunk;
            counts += (i64)G.nchunks * (G.nparts + 1);
            out.parts = std::max<i64>(out.parts, G.nparts);
            const int32_t gi = (int32_t)giants.size();
            giants.push_back(G);
            for (int32_t j = 0; j < G.nchunks; j++)
                cls.push_back(WideItem{r.beg + j * kWChunk, r.v, (int32_t)std::min<i64>(kWChunk, d - j * kWChunk),
                                       gi, j});
        }
    out.pairs = pairs;
    out.counts = counts;
    for (int b = kNumBins - 1; b >= 7; b--)
        for (i64 q = P.lo(b, c); q < P.hi(b, c); q++) {
            const WideRow &r = rows[q - hlo];
            if (r.deg <= kWMidMaxDeg) out.extra.push_back(r);
            else if (r.deg <= kWHeavyMaxDeg) cls.push_back(WideItem{r.beg, r.v, r.deg, -1, 0});
        }
    // longest processing time first: each item, costliest first (equal costs
    // in list order), to the workgroup with the least work so far (lowest
    // index on a tie)
    std::vector<std::pair<double, int>> heap;  // max-heap of (-load, -workgroup)
    for (int w = 0; w < nb; w++) heap.push_back({-0.0, -w});
    std::make_heap(heap.begin(), heap.end());
    const int turn = (int)((i64)c * 37 % nb);
    auto at_grid = [&](int w) { return (w + turn) % nb; };
    auto give = [&](double cost) {
        std::pop_heap(heap.begin(), heap.end());
        auto &h = heap.back();
        const int w = -h.second;
        h.first -= cost;
        std::push_heap(heap.begin(), heap.end());
        return at_grid(w);
    };
    auto item_cost = [](const WideItem &it) { return it.g >= 0 ? kWCostChunk : kWCostHeavy + 3.0 * it.len / 1024.0; };
    std::vector<size_t> order(cls.size());
    for (size_t i = 0; i < cls.size(); i++) order[i] = i;
    std::stable_sort(order.begin(), order.end(),
                     [&](size_t a, size_t b) { return item_cost(cls[a]) > item_cost(cls[b]); });
    std::vector<int> to(cls.size());
    for (size_t i : order) to[i] = give(item_cost(cls[i]));
    // the wavefront items go, in turn, to the workgroups that the items level
    // off with: the `groups` least loaded ones
    i64 items = (i64)out.extra.size() + P.hi(6, c) - P.lo(6, c);
    double cost = items * kWCostMid;
    for (int b = 5; b >= 1; b--) {
        const i64 per_item = kWave / kBinGroup[b], n = (P.hi(b, c) - P.lo(b, c) + per_item - 1) / per_item;
        items += n;
        cost += n * kWCostLight;
    }
    out.items = items;
    std::vector<std::pair<double, int>> load;  // (load, workgroup)
    for (const auto &h : heap) load.push_back({-h.first, -h.second});
    std::sort(load.begin(), load.end());
    double level = cost / kWWavesPerGroup;
    int groups = 0;
    while (groups < nb && (groups == 0 || load[groups].first * groups < level)) level += load[groups++].first;
    groups = (int)std::min<i64>(groups, std::max<i64>(items, 1));
    out.groups = groups;
    out.rank.assign(nb, -1);
    for (int r = 0; r < groups; r++) out.rank[at_grid(load[r].second)] = r;
    // per workgroup: chunks before heavy vertices, the class's order otherwise
    out.wstart.assign(nb + 1, 0);
    for (size_t i = 0; i < cls.size(); i++) out.wstart[to[i] + 1]++;
    for (int w = 0; w < nb; w++) out.wstart[w + 1] += out.wstart[w];
    out.wi.resize(cls.size());
    {
        std::vector<i64> at(out.wstart.begin(), out.wstart.end() - 1);
        for (size_t i = 0; i < cls.size(); i++) out.wi[at[to[i]]++] = cls[i];
    }
    // the giants' partitions (scored once every chunk is in), to the least
    // loaded workgroups; they follow all other work of a step, so a partition
    // waits only on chunks, which never wait
    std::vector<std::pair<int, int2>> parts;
    for (size_t gi = 0; gi < giants.size(); gi++)
        for (int32_t j = 0; j < giants[gi].nparts; j++) parts.push_back({give(kWCostPart), int2{(int)gi, j}});
    out.pstart.assign(nb + 1, 0);
    for (const auto &p : parts) out.pstart[p.first + 1]++;
    for (int w = 0; w < nb; w++) out.pstart[w + 1] += out.pstart[w];
    out.pi.resize(parts.size());
    std::vector<i64> at(out.pstart.begin(), out.pstart.end() - 1);
    for (const auto &p : parts) out.pi[at[p.first]++] = p.second;
}

// host threads for the planning: the CPUs this process may run on, at most 16
static int host_threads() {
    cpu_set_t set;
    int n = 1;
    if (sched_getaffinity(0, sizeof(set), &set) == 0) n = CPU_COUNT(&set);
    return std::max(1, std::min(n, 16));
}

bool build_wide_plan(const DevGraph &g, const PhaseSetup &P, const double *selfw, int nb, WidePlan &L,
                     hipStream_t s) {
    const auto t0 = std::chrono::steady_clock::now();
    const int ncol = P.ncol;
    // the vertices in perm's order; those of bins 7..9 (heavy and giant) for the plan
    const i64 hlo = P.bin_lo(7), hhi = P.bin_hi(kNumBins - 1), extra0 = P.bin_hi(7);
    // (the extra rows of bin 7 may take the place of bins 8 and 9, which the kernel reads no rows of)
    L.rows.alloc(std::max<i64>(hhi + (P.bin_hi(7) - hlo), 1), s);
    launch_wide_rows(P.perm.p, g.off, P.k.p, selfw, P.bin_lo(1), hhi, L.rows.p, s);
    std::vector<WideRow> rows(hhi - hlo);
    if (hhi > hlo) {
        Readback rb(s);
        rb.add(rows.data(), L.rows.p + hlo, rows.size() * sizeof(WideRow));
        rb.run();
    }
    // the classes are planned independently, on host threads, then concatenated
    std::vector<ClassPlan> cp(ncol);
    // (a thread per 16384 vertices: starting one costs about what planning
    // that many does)
    const int nthreads = (int)std::min<i64>({(i64)ncol, (i64)host_threads(), 1 + g.nv / 16384});
    std::atomic<int> next{0};
    std::atomic<bool> no_memory{false};
    auto worker = [&]() {
        for (int c = next++; c < ncol; c = next++) {
            try {
                plan_class(P, rows, hlo, c, nb, cp[c]);
            } catch (const std::bad_alloc &) {
                no_memory = true;
            }
        }
    };
    run_workers(nthreads, worker);
    if (no_memory) throw std::bad_alloc();
    // the non-empty classes, and every workgroup's streams over them
    std::vector<WideClass> classes;
    std::vector<WideRow> extra;
    std::vector<int32_t> rank, used;  // used: the colors of `classes`
    std::vector<WideGiant> giants;
    std::vector<i64> gbase;
    i64 gpairs = 0, gcounts = 0, gparts = 1, nwi = 0, npi = 0, nvi = 0, vlo = 0;
    for (int c = 0; c < ncol; c++) {
        const ClassPlan &C = cp[c];
        if (!C.ok) {
            trace("  wide plan: a vertex of more than %ld entries", (long)(kWMaxChunks * kWChunk));
            return false;
        }
        WideClass K{};
        K.lo = (int32_t)vlo;
        for (int b = 0; b < kNumBins; b++) vlo += P.hi(b, c) - P.lo(b, c);
        K.hi = (int32_t)vlo;
        if (C.items == 0 && C.wi.empty()) continue;  // at most vertices without entries, which stay
        K.nextra = (int32_t)C.extra.size();
        K.extra0 = (int32_t)(extra0 + (i64)extra.size());
        for (int b = 0; b < 6; b++) {
            K.bin_lo[b] = (int32_t)P.lo(6 - b, c);
            K.bin_n[b] = (int32_t)(P.hi(6 - b, c) - P.lo(6 - b, c));
        }
        K.groups = C.groups;
        classes.push_back(K);
        used.push_back(c);
        extra.insert(extra.end(), C.extra.begin(), C.extra.end());
        rank.insert(rank.end(), C.rank.begin(), C.rank.end());
        gbase.push_back((i64)giants.size());
        giants.insert(giants.end(), C.giants.begin(), C.giants.end());
        gpairs = std::max(gpairs, C.pairs);
        gcounts = std::max(gcounts, C.counts);
        gparts = std::max(gparts, C.parts);
        nwi += (i64)C.wi.size();
        npi += (i64)C.pi.size();
        nvi += C.items;
    }
    const int ncls = (int)classes.size();
    std::vector<WideItem> wi;
    std::vector<int2> pi;
    wi.reserve(nwi + nb);
    pi.reserve(npi);
    std::vector<i64> wbeg(nb), pbeg(nb), wend((size_t)nb * ncls), pend((size_t)nb * ncls);
    for (int w = 0; w < nb; w++) {
        wbeg[w] = (i64)wi.size();
        pbeg[w] = (i64)pi.size();
        for (int k = 0; k < ncls; k++) {
            const ClassPlan &C = cp[used[k]];
            for (i64 i = C.wstart[w]; i < C.wstart[w + 1]; i++) {
                wi.push_back(C.wi[i]);
                if (C.wi[i].g >= 0) wi.back().g += (int32_t)gbase[k];
            }
            for (i64 i = C.pstart[w]; i < C.pstart[w + 1]; i++)
                pi.push_back(int2{C.pi[i].x + (int)gbase[k], C.pi[i].y});
            wend[(size_t)w * ncls + k] = (i64)wi.size();
            pend[(size_t)w * ncls + k] = (i64)pi.size();
        }
        wi.push_back(WideItem{0, 0, 0, -1, 0});  // the stream's end, read ahead and never run
    }
    L.ncls = ncls;
    L.nwitems = nwi;
    L.nvitems = nvi;
    L.ngiants = (i64)giants.size();
    L.gparts = gparts;
    L.gpairs = gpairs;
    L.gcounts = gcounts;
    // (everything is allocated before the first copy, which reads the host
    // vectors until the wait below)
    auto room = [&](auto &buf, size_t n) { buf.alloc(std::max<size_t>(n, 1), s); };
    room(L.classes, classes.size());
    room(L.over, ncls);
    room(L.rank, rank.size());
    room(L.witems, wi.size());
    room(L.wbeg, wbeg.size());
    room(L.wend, wend.size());
    room(L.pitems, pi.size());
    room(L.pbeg, pbeg.size());
    room(L.pend, pend.size());
    room(L.giants, giants.size());
    const i64 ng = std::max<i64>(L.ngiants, 1);
    room(L.gpk, gpairs);
    room(L.gpv, gpairs);
    room(L.gcnt, gcounts);
    room(L.gstate, 3 * ng);
    room(L.gsc, ng);
    room(L.gout, ng);
    room(L.gcand, 3 * ng * gparts);
    room(L.gcid, ng * gparts);
    auto upload = [&](auto *at, const auto &host) {
        if (!host.empty())
            GLV_HIP(hipMemcpyAsync(at, host.data(), host.size() * sizeof(host[0]), hipMemcpyHostToDevice, s));
    };
    upload(L.rows.p + extra0, extra);
    upload(L.classes.p, classes);
    upload(L.rank.p, rank);
    upload(L.witems.p, wi);
    upload(L.wbeg.p, wbeg);
    upload(L.wend.p, wend);
    upload(L.pitems.p, pi);
    upload(L.pbeg.p, pbeg);
    upload(L.pend.p, pend);
    upload(L.giants.p, giants);
    GLV_HIP(hipStreamSynchronize(s));  // the host vectors are pageable
    trace("  wide plan: %ld workgroup items, %ld wavefront items, %ld giants (%ld pairs, %ld partitions at most), "
          "%.1f ms on the host",
          (long)L.nwitems, (long)L.nvitems, (long)L.ngiants, (long)gpairs, (long)gparts,
          std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count());
    return true;
}

}  // namespace glv
