// Lines of a strided array along one axis, and how far apart the lines of one workgroup lie.
// Plain C++, for the host and the device alike.
#pragma once

#include <algorithm>

namespace ifft {

constexpr int kLineDims = 9;   // dimensions of an array besides the axis, at most

// element offsets of the lines along one axis: the other dimensions, last fastest
struct LineMap {
    int nd;
    long long cnt[kLineDims];
    long long st[kLineDims];
};

// Bounds of the element offset of any line of a group from the group's first line, the groups being
// runs of `tb` lines from multiples of tb on.  Exact where the lines are evenly spaced; where a group
// may pass from one run of the faster dimensions into the next, from either end of the run.
inline void line_reach(const LineMap &m, long long tb, long long &lo, long long &hi)
{
    lo = hi = 0;
    long long inner = 1;   // lines per step of the dimension at hand
    for (int d = m.nd - 1; d >= 0;) {
        long long c = m.cnt[d];
        const long long st = m.st[d];
        for (--d; d >= 0 && (m.cnt[d] == 1 || m.st[d] == c * st); --d) c *= m.cnt[d];   // evenly spaced: one run
        if (inner % tb == 0) return;   // no group leaves a run of the faster dimensions
        const long long fwd = std::min(c - 1, (tb - 1 + inner - 1) / inner);
        const bool wraps = d >= 0 && inner * c % tb != 0;
        const long long a = fwd * st, b = wraps ? -(c - 1) * st : 0;
        lo += std::min(std::min(a, b), 0LL);
        hi += std::max(std::max(a, b), 0LL);
        if (!wraps) return;
        inner *= c;
    }
}

}  // namespace ifft
