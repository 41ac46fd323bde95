// The order between trees and batches, followed through the events the library
// records and waits for.  Linked against the emulation build, whose event calls
// this program replaces: every stream carries a clock of what it is behind.
//   batch_events <scenario>; prints "ok" or what is out of order.
#include <cstdio>
#include <cstring>
#include <map>
#include <vector>

#include "hip_emu.h"
#include "ikd_tree_amd.h"

using Clock = std::map<hipStream_t, long>;  // records of a stream that are behind us
static std::map<hipStream_t, Clock> g_now;
static std::map<hipEvent_t, Clock> g_at;
static long g_live_events = 0, g_waits = 0;

hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new char);
    ++g_live_events;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<char*>(e);
    g_at.erase(e);
    --g_live_events;
    return hipSuccess;
}
static bool captured(hipStream_t s) {
    hipStreamCaptureStatus st;
    hipStreamIsCapturing(s, &st);
    return st != hipStreamCaptureStatusNone;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (captured(s)) {  // part of the graph: orders nothing outside
        g_at[e].clear();
        return hipSuccess;
    }
    ++g_now[s][s];
    g_at[e] = g_now[s];
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    ++g_waits;
    if (captured(s)) return hipSuccess;
    for (auto& kv : g_at[e]) g_now[s][kv.first] = std::max(g_now[s][kv.first], kv.second);
    return hipSuccess;
}

#define REQUIRE(x)                                         \
    do {                                                   \
        if (!(x)) {                                        \
            std::printf("line %d: %s\n", __LINE__, #x);    \
            return 1;                                      \
        }                                                  \
    } while (0)

constexpr int N = 300, NQ = 20, K = 3;
static float g_pts[3 * N], g_q[3 * NQ], g_xyz[3 * NQ * K], g_d2[NQ * K], g_r[NQ];
static uint32_t g_ids[NQ * K];
static int32_t g_cnt[NQ], g_tree[NQ];
static int64_t g_off[NQ + 1];

static ikd_tree_t make_tree() {
    ikd_tree_t t = nullptr;
    if (ikd_create(0.5f, 0.6f, 0.2f, &t) != IKD_OK || ikd_build(t, g_pts, nullptr, N) != IKD_OK) return nullptr;
    return t;
}
static hipStream_t stream_of(ikd_batch_t b) {
    void* s = nullptr;
    ikd_batch_stream(b, &s);
    return (hipStream_t)s;
}
static int launch(ikd_batch_t b, const ikd_tree_t* t, int n) {
    return ikd_batch_nearest_search_device(b, t, n, g_tree, g_q, NQ, nullptr, K, nullptr, 5.0, g_xyz, g_d2, g_ids, g_cnt);
}
static int launch_noalloc(ikd_batch_t b, const ikd_tree_t* t, int n) {
    return ikd_batch_nearest_search_noalloc(b, t, n, g_tree, g_q, NQ, nullptr, K, nullptr, 5.0, g_xyz, g_d2, g_ids,
                                            g_cnt);
}
static int launch_radius(ikd_batch_t b, const ikd_tree_t* t, int n) {
    int64_t total;
    return ikd_batch_radius_search_device(b, t, n, g_tree, g_q, g_r, NQ, g_off, nullptr, nullptr, 0, &total);
}
// stream s is behind the last launch of batch b
static bool behind(hipStream_t s, ikd_batch_t b) {
    const hipStream_t bs = stream_of(b);
    return g_now[s][bs] >= g_now[bs][bs] && g_now[bs][bs] > 0;
}

// launches of two batches with a tree in common, nothing called on the trees between
static int two_batches() {
    ikd_tree_t t[3] = {make_tree(), make_tree(), make_tree()};
    ikd_batch_t a, b;
    REQUIRE(t[0] && t[1] && t[2]);
    REQUIRE(ikd_batch_create(&a) == IKD_OK && ikd_batch_create(&b) == IKD_OK);
    ikd_knn_graph_t g;
    REQUIRE(ikd_batch_knn_graph_create(b, t + 1, 2, g_tree, g_q, NQ, nullptr, K, nullptr, 5.0, g_xyz, g_d2, g_ids, g_cnt,
                                       &g) == IKD_OK);
    int (*const form[])(ikd_batch_t, const ikd_tree_t*, int) = {launch, launch_noalloc, launch_radius};
    for (int i = 0; i < 3; ++i) {
        for (int j = 0; j < 3; ++j) {
            REQUIRE(form[i](a, t, 2) == IKD_OK);
            REQUIRE(form[j](b, t + 1, 2) == IKD_OK);
            REQUIRE(behind(stream_of(b), a));
            REQUIRE(form[i](a, t, 2) == IKD_OK);
            REQUIRE(behind(stream_of(a), b));
        }
        REQUIRE(ikd_batch_knn_graph_launch(g) == IKD_OK);
        REQUIRE(behind(stream_of(b), a));
    }
    // and the trees' later work is behind both
    int32_t n = 0;
    REQUIRE(ikd_add_points(t[1], g_q, nullptr, 3, 0, &n) == IKD_OK);
    void* s = nullptr;
    REQUIRE(ikd_stream(t[1], &s) == IKD_OK);
    REQUIRE(behind((hipStream_t)s, a) && behind((hipStream_t)s, b));
    return 0;
}

// a launch that the caller captures from the batch's stream runs when the caller
// replays it: the order of what runs now does not change
static int captured_launch() {
    ikd_tree_t t = make_tree();
    ikd_batch_t b;
    REQUIRE(t && ikd_batch_create(&b) == IKD_OK);
    const hipStream_t bs = stream_of(b);
    for (int round = 0; round < 2; ++round) {
        REQUIRE(launch(b, &t, 1) == IKD_OK);
        const long first = g_now[bs][bs];
        hipGraph_t g = nullptr;
        REQUIRE(hipStreamBeginCapture(bs, hipStreamCaptureModeThreadLocal) == hipSuccess);
        REQUIRE(launch_noalloc(b, &t, 1) == IKD_OK);
        REQUIRE(hipStreamEndCapture(bs, &g) == hipSuccess);
        REQUIRE(hipGraphDestroy(g) == hipSuccess);
        // the tree's next work is behind the launch before the capture
        int32_t n = 0;
        REQUIRE(ikd_add_points(t, g_q, nullptr, 3, 0, &n) == IKD_OK);
        long most = 0;
        for (auto& kv : g_now)
            if (kv.first != bs) most = std::max(most, kv.second[bs]);
        REQUIRE(most >= first);
        // a launch after a captured one is behind the tree's work
        REQUIRE(hipStreamBeginCapture(bs, hipStreamCaptureModeThreadLocal) == hipSuccess);
        REQUIRE(launch_noalloc(b, &t, 1) == IKD_OK);
        REQUIRE(hipStreamEndCapture(bs, &g) == hipSuccess);
        REQUIRE(hipGraphDestroy(g) == hipSuccess);
        const Clock before = g_now[bs];
        REQUIRE(launch(b, &t, 1) == IKD_OK);
        bool waited = false;
        for (auto& kv : g_now[bs])
            if (kv.first != bs) waited = waited || !before.count(kv.first) || kv.second > before.at(kv.first);
        REQUIRE(waited);
    }
    return 0;
}

// a batch per request over a tree that is only searched: a closed batch leaves
// nothing behind
static int closed_batches() {
    ikd_tree_t t = make_tree();
    ikd_batch_t keep;
    REQUIRE(t && ikd_batch_create(&keep) == IKD_OK && launch(keep, &t, 1) == IKD_OK);
    const long events = g_live_events;
    for (int i = 0; i < 50; ++i) {
        ikd_batch_t b;
        REQUIRE(ikd_batch_create(&b) == IKD_OK);
        REQUIRE(launch(b, &t, 1) == IKD_OK && launch(keep, &t, 1) == IKD_OK);
        REQUIRE(ikd_batch_destroy(b) == IKD_OK);
        REQUIRE(g_live_events <= events + 1);
    }
    const long waits = g_waits;
    int32_t n = 0;
    REQUIRE(ikd_add_points(t, g_q, nullptr, 3, 0, &n) == IKD_OK);
    REQUIRE(g_waits - waits <= 2);
    REQUIRE(ikd_batch_destroy(keep) == IKD_OK && ikd_destroy(t) == IKD_OK);
    REQUIRE(g_live_events == 0);
    return 0;
}

int main(int argc, char** argv) {
    unsigned x = 1;
    auto rnd = [&] {
        x = x * 1664525u + 1013904223u;
        return (float)(x >> 8) / (1 << 24);
    };
    for (float& v : g_pts) v = 20 * rnd();
    for (float& v : g_q) v = 20 * rnd();
    for (float& v : g_r) v = 1 + rnd();
    const char* what = argc > 1 ? argv[1] : "";
    int rc = 2;
    if (!std::strcmp(what, "two_batches")) rc = two_batches();
    if (!std::strcmp(what, "captured_launch")) rc = captured_launch();
    if (!std::strcmp(what, "closed_batches")) rc = closed_batches();
    if (rc == 0) std::printf("ok\n");
    return rc;
}
