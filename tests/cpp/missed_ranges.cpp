// Which kNN walk a tree takes after Add_Point_Boxes, from the kernels that the
// emulation build counts: one lane per query with exact distances while stored
// ranges may miss restored points, a team again once the whole tree is new.
#include <cstdio>
#include <cstring>
#include <vector>

#include "ikd_tree_amd.h"

extern "C" void emu_dispatch_reset();
extern "C" long long emu_dispatch_tally(char* buf, int len);

static char g_buf[1 << 16];

// 't': a team walked, 'e': one lane with exact distances, 'b': both, '?': neither
static char walked() {
    emu_dispatch_tally(g_buf, sizeof(g_buf));
    const bool team = std::strstr(g_buf, "k_knn_team") != nullptr, exact = std::strstr(g_buf, "STACK_EXACT") != nullptr;
    return team ? (exact ? 'b' : 't') : (exact ? 'e' : '?');
}
static char walk(ikd_tree_t t) {
    const float q[3] = {1, 2, 3};
    float xyz[15], d2[5];
    uint32_t ids[5];
    int32_t cnt;
    emu_dispatch_reset();
    if (ikd_nearest_search(t, q, 1, 5, 1e9, xyz, d2, ids, &cnt) != IKD_OK) return '?';
    return walked();
}
// the same of a launch over n trees
static char walk_batch(ikd_batch_t b, const ikd_tree_t* trees, int n) {
    static float q[30], xyz[150], d2[50];
    static uint32_t ids[50];
    static int32_t cnt[10], which[10];
    for (int i = 0; i < 10; ++i) which[i] = i % n;
    emu_dispatch_reset();
    if (ikd_batch_nearest_search_device(b, trees, n, which, q, 10, nullptr, 5, nullptr, 1e9, xyz, d2, ids, cnt) != IKD_OK)
        return 'x';
    return walked();
}

#define REQUIRE(x)                                      \
    do {                                                \
        if (!(x)) {                                     \
            std::printf("line %d: %s\n", __LINE__, #x); \
            return 1;                                   \
        }                                               \
    } while (0)

int main() {
    unsigned x = 1;
    auto rnd = [&] {
        x = x * 1664525u + 1013904223u;
        return (float)(x >> 8) / (1 << 24);
    };
    std::vector<float> p(3 * 600), far(3 * 3000);
    for (float& v : p) v = 10 * rnd();
    for (float& v : far) v = 30 + 10 * rnd();
    ikd_tree_t t;
    REQUIRE(ikd_create(0.5f, 0.6f, 0.2f, &t) == IKD_OK && ikd_build(t, p.data(), nullptr, 600) == IKD_OK);
    REQUIRE(walk(t) == 't');
    const float del[6] = {2, 2, 2, 6, 6, 6}, back[6] = {1, 1, 1, 5, 5, 5}, away[6] = {50, 50, 50, 60, 60, 60};
    int32_t n = 0;
    REQUIRE(ikd_delete_point_boxes(t, del, 1, &n) == IKD_OK && n > 0);
    REQUIRE(walk(t) == 't');
    REQUIRE(ikd_add_point_boxes(t, away, 1) == IKD_OK && walk(t) == 't');  // restores nothing
    REQUIRE(ikd_add_point_boxes(t, back, 1) == IKD_OK && walk(t) == 'e');
    REQUIRE(ikd_add_points(t, p.data(), nullptr, 1, 0, &n) == IKD_OK && walk(t) == 'e');
    // a launch over several trees with one such
    ikd_tree_t other;
    ikd_batch_t b;
    REQUIRE(ikd_create(0.5f, 0.6f, 0.2f, &other) == IKD_OK && ikd_build(other, p.data(), nullptr, 600) == IKD_OK);
    REQUIRE(ikd_batch_create(&b) == IKD_OK);
    const ikd_tree_t both[2] = {other, t};
    REQUIRE(walk_batch(b, both, 1) == 't' && walk_batch(b, both + 1, 1) == 'e' && walk_batch(b, both, 2) == 'e');
    REQUIRE(ikd_batch_destroy(b) == IKD_OK && ikd_destroy(other) == IKD_OK);
    // far more points on one side: the root is rebuilt
    REQUIRE(ikd_add_points(t, far.data(), nullptr, 3000, 0, &n) == IKD_OK && walk(t) == 't');
    REQUIRE(ikd_delete_point_boxes(t, del, 1, &n) == IKD_OK && ikd_add_point_boxes(t, back, 1) == IKD_OK && walk(t) == 'e');
    REQUIRE(ikd_build(t, p.data(), nullptr, 600) == IKD_OK && walk(t) == 't');
    REQUIRE(ikd_destroy(t) == IKD_OK);
    std::printf("ok\n");
    return 0;
}
