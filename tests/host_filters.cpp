// The crossing pass's predicates for the host (test infrastructure): the double
// filters and the exact determinants of exact.hpp over given rational points.
// A point is 5 words: X low, X high, Y low, Y high, W.
#include <hip/hip_runtime.h>

#include "../gcdt_amd/csrc/exact.hpp"

using namespace gcdt;

static HPt point(const int64_t* w)
{
    HPt h;
    h.X.w[0] = (uint64_t)w[0];
    h.X.w[1] = (uint64_t)w[1];
    h.Y.w[0] = (uint64_t)w[2];
    h.Y.w[1] = (uint64_t)w[3];
    h.W = w[4];
    return h;
}

// n items of 4 points: out[4i..] = orient filter, exact, incircle filter, exact
extern "C" void host_filters(const int64_t* w, int n, int32_t* out)
{
    for (int i = 0; i < n; i++) {
        HPt p[4];
        for (int j = 0; j < 4; j++) p[j] = point(w + 20 * i + 5 * j);
        out[4 * i] = orient_filter(dpt(p[0]), dpt(p[1]), dpt(p[2]));
        out[4 * i + 1] = orient_h(p[0], p[1], p[2]);
        out[4 * i + 2] = incircle_filter(dpt(p[0]), dpt(p[1]), dpt(p[2]), dpt(p[3]));
        out[4 * i + 3] = incircle_h(p[0], p[1], p[2], p[3]);
    }
}
