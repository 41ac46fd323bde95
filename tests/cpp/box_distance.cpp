// calc_box_dist against the reference's six comparisons (ikd_Tree.cpp:1380-1391),
// bit for bit, over every combination of awkward values per axis.
#include <cstdio>
#include <cstring>
#include <limits>

#include "ikd_common.h"

static float reference(const float* b, const float* p) {
    float s = 0.0f;
    for (int a = 0; a < 3; ++a) {
        if (p[a] < b[a]) { float t = p[a] - b[a]; s = s + t * t; }
        if (p[a] > b[3 + a]) { float t = p[a] - b[3 + a]; s = s + t * t; }
    }
    return s;
}

int main() {
    const float inf = std::numeric_limits<float>::infinity(), nan = std::numeric_limits<float>::quiet_NaN();
    const float v[] = {0.0f, -0.0f, 1.0f, -1.5f, 0.1f, 1e-30f, -1e-40f, 3.3e7f, 2e19f, -3e38f, inf, -inf, nan};
    const int n = sizeof v / sizeof v[0];
    struct Axis { float lo, hi, p; };
    static Axis ax[n * n * n];
    int na = 0;
    for (int i = 0; i < n; ++i)
        for (int j = 0; j < n; ++j)
            for (int k = 0; k < n; ++k) {
                // ranges are ordered, empty (+inf, -inf) or hold a NaN
                if (v[i] > v[j] && !(v[i] == inf && v[j] == -inf)) continue;
                ax[na++] = Axis{v[i], v[j], v[k]};
            }
    long long bad = 0, all = 0;
    for (int x = 0; x < na; ++x)
        for (int y = 0; y < na; y += 7)
            for (int z = (x + y) % 11; z < na; z += 11) {
                const float b[6] = {ax[x].lo, ax[y].lo, ax[z].lo, ax[x].hi, ax[y].hi, ax[z].hi};
                const float p[3] = {ax[x].p, ax[y].p, ax[z].p};
                const float r = reference(b, p), g = ikd::calc_box_dist(b, p[0], p[1], p[2]);
                ++all;
                if (std::memcmp(&r, &g, 4) != 0) ++bad;
            }
    std::printf("%lld of %lld differ\n", bad, all);
    return bad != 0;
}
