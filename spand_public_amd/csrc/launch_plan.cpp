// Host-side launch plans (launch_plan.hpp). No device is touched here.
#include "launch_plan.hpp"

#include <algorithm>
#include <numeric>

#include "kernels.hpp"

namespace spand {

std::vector<GetrfLaunch> plan_getrf(const std::vector<int>& n) {
    std::vector<GetrfLaunch> out;
    // tasks [0, longer(m)) have more than m rows
    auto longer = [&](int m) {
        return (int)(std::partition_point(n.begin(), n.end(), [&](int x) { return x > m; }) - n.begin());
    };
    // tasks [0, last) with per(rows) workgroups each, one launch at the largest one's unless more
    // than GETRF_IDLE of them would have nothing to do (a launch costs about as much as these)
    constexpr long long GETRF_IDLE = 1 << 15;
    auto add = [&](GetrfLaunch l, int last, auto&& per) {
        for (int first = 0; first < last; first += l.count) {
            l.first = first;
            l.per_task = per(n[first]);
            const int half = std::min(last, longer(n[first] / 2));
            int end = last;
            if (half < last && (long long)(last - half) * (l.per_task - per(n[half])) > GETRF_IDLE) end = half;
            l.count = (int)std::min<long long>(end - first, launch_blocks_max(l.threads) / l.per_task);
            out.push_back(l);
        }
    };
    const int nmax = n.empty() ? 0 : n[0];
    for (int kb = 0; kb < nmax;) {
        const int rows = nmax - kb;
        const int rpt = rows <= 1024 ? 1 : (rows <= 2048 ? 2 : 4), nb = GETRF_NB / rpt;
        const int threads = ((rows + rpt - 1) / rpt + 63) / 64 * 64;
        // a pivot no longer than kb is done; one inside the first panel has no other column
        add({GetrfLaunch::PANEL, kb, nb, 0, 0, 1, threads}, longer(kb), [](int) { return 1; });
        add({GetrfLaunch::TRAIL, kb, nb, 0, 0, 1, GETRF_NT}, longer(kb > 0 ? kb : nb), [](int m) { return (m + 7) / 8; });
        kb += nb;
    }
    add({GetrfLaunch::SPLIT, 0, 0, 0, 0, 1, GETRF_NT}, longer(0), [](int m) { return (m + 31) / 32 * ((m + 31) / 32); });
    return out;
}

SlabPlan place_slabs(const std::vector<int>& nsub, const std::vector<int>& steps, int cap) {
    constexpr int XCDS = 8;
    const int each = cap / XCDS;
    SlabPlan P;
    std::vector<int> order(nsub.size());
    std::iota(order.begin(), order.end(), 0);
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return nsub[a] > nsub[b]; });
    if (order.empty() || nsub[order[0]] > cap) return P;
    size_t x0 = 0;
    while (x0 < order.size() && nsub[order[x0]] > each) {  // too long for one XCD
        SlabChunk c{(int)P.place.size(), 0, 0, false};
        while (x0 < order.size() && nsub[order[x0]] > each && c.count + nsub[order[x0]] <= cap) {
            const int x = order[x0++];
            for (int k = 0; k < nsub[x]; k++) P.place.push_back({x, k});
            c.count += nsub[x];
            c.steps = std::max(c.steps, steps[x]);
            c.waits = c.waits || nsub[x] > 1;
        }
        P.chunk.push_back(c);
        P.spread++;
    }
    std::vector<int> rest(order.begin() + x0, order.end()), later;
    while (!rest.empty()) {
        std::vector<RrqrSlab> on[XCDS];
        SlabChunk c{(int)P.place.size(), 0, 0, false};
        size_t most = 0;
        later.clear();
        for (int x : rest) {
            auto* q = &on[0];
            for (auto& o : on)
                if (o.size() < q->size()) q = &o;
            if ((int)q->size() + nsub[x] > each) {
                later.push_back(x);
                continue;
            }
            for (int k = 0; k < nsub[x]; k++) q->push_back({x, k});
            most = std::max(most, q->size());
            c.steps = std::max(c.steps, steps[x]);
            c.waits = c.waits || nsub[x] > 1;
        }
        c.count = (int)(most * XCDS);
        P.place.resize(c.first + most * XCDS, {-1, 0});
        for (int o = 0; o < XCDS; o++)
            for (size_t k = 0; k < on[o].size(); k++) P.place[c.first + k * XCDS + o] = on[o][k];
        P.chunk.push_back(c);
        rest.swap(later);
    }
    return P;
}

}  // namespace spand

// For tests of the plans on the host: rows of (kind, kb, nb, first, count, per_task, threads),
// their number returned.
extern "C" int spand_plan_getrf(const int* n, int ntasks, int* out, int max_rows) {
    const auto v = spand::plan_getrf(std::vector<int>(n, n + ntasks));
    for (int i = 0; i < (int)v.size() && i < max_rows; i++) {
        const auto& l = v[i];
        const int row[7] = {l.kind, l.kb, l.nb, l.first, l.count, l.per_task, l.threads};
        std::copy(row, row + 7, out + 7 * i);
    }
    return (int)v.size();
}
// rows of (first, count, steps, waits) per chunk, their number returned; place: (cluster, slab) by
// workgroup, at most max_place of them, their number in n_place
extern "C" int spand_plan_slabs(const int* nsub, const int* steps, int n, int cap, int* chunks, int max_chunks,
                                int* place, int max_place, int* n_place) {
    const auto p = spand::place_slabs(std::vector<int>(nsub, nsub + n), std::vector<int>(steps, steps + n), cap);
    for (int i = 0; i < (int)p.chunk.size() && i < max_chunks; i++) {
        const int row[4] = {p.chunk[i].first, p.chunk[i].count, p.chunk[i].steps, p.chunk[i].waits};
        std::copy(row, row + 4, chunks + 4 * i);
    }
    *n_place = (int)p.place.size();
    for (int i = 0; i < *n_place && i < max_place; i++) {
        place[2 * i] = p.place[i].big;
        place[2 * i + 1] = p.place[i].slab;
    }
    return (int)p.chunk.size();
}
