// Host-side launch plans (launch_plan.hpp). No device is touched here.
#include "launch_plan.hpp"

#include <algorithm>

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
