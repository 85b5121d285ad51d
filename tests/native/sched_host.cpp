// sched_host.cpp -- the chunk scheduler (mccl_amd/csrc/mcclx_sched.cpp) over the host stand-in of
// the kernel layer (null_mcclx.cpp): launches per list, results of fp32 sums, workspace sizes.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "mcclx.h"

extern "C" std::atomic<long> null_memory_questions;

// The calling thread's allocation number `g_fail_at` fails, once.
thread_local long g_fail_at = -1;
void* operator new(size_t n) {
    if (g_fail_at >= 0 && g_fail_at-- == 0) throw std::bad_alloc();
    if (void* p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

namespace {
int g_bad = 0;

// A call whose k-th allocation fails, for every k it has: an error code and no exception, and the
// call goes through as soon as nothing fails any more.
template <class F>
void without_memory(mcclx_ctx* ctx, const char* what, F&& call) {
    int refused = 0;
    for (long k = 0;; ++k) {
        int rc = MCCLX_OK;
        bool threw = false;
        g_fail_at = k;
        try {
            rc = call();
        } catch (...) {
            threw = true;
        }
        const bool met = g_fail_at < 0;
        g_fail_at = -1;
        mcclx_queue_drain(ctx);
        if (threw || (met && rc != MCCLX_ERR_NOMEM) || (!met && rc != MCCLX_OK)) {
            printf("FAILED: %s, allocation %ld: %s, code %d\n", what, k, threw ? "an exception" : "returned", rc);
            ++g_bad;
            return;
        }
        if (!met) break;
        ++refused;
    }
    if (!refused) {
        printf("FAILED: %s allocates nothing\n", what);
        ++g_bad;
    }
}

mcclx_replay replay(int world, int algo, int op, int wire, int mode, uint64_t numel, void* const* tensors) {
    mcclx_replay r;
    memset(&r, 0, sizeof r);
    r.world = world;
    r.algo = algo;
    r.op = op;
    r.dtype = MCCLX_F32;
    r.wire_bf16 = wire;
    r.mode = mode;
    r.acc = MCCLX_ACC_STEP;
    r.numel = numel;
    r.tensors = const_cast<void**>(tensors);
    return r;
}

// A list of `entries` allreduces whose sizes alternate; returns the launches it took.
unsigned long long list(mcclx_ctx* ctx, const char* what, int world, int algo, int op, int wire, int mode,
                        uint64_t small, uint64_t large, int entries, unsigned long long want) {
    std::vector<std::vector<float>> data;
    std::vector<std::vector<void*>> ptrs(static_cast<size_t>(entries));
    std::vector<std::vector<char>> ws;
    std::vector<mcclx_replay> reps;
    for (int e = 0; e < entries; ++e) {
        const uint64_t n = e % 2 ? large : small;
        for (int r = 0; r < world; ++r) data.emplace_back(n, static_cast<float>(r + 1 + e));
    }
    for (int e = 0; e < entries; ++e) {
        const uint64_t n = e % 2 ? large : small;
        for (int r = 0; r < world; ++r) ptrs[size_t(e)].push_back(data[size_t(e * world + r)].data());
        mcclx_replay rp = replay(world, algo, op, wire, mode, n, ptrs[size_t(e)].data());
        ws.emplace_back(mcclx_replay_workspace_bytes(&rp) + 1);
        rp.workspace = ws.back().data();
        rp.workspace_bytes = ws.back().size() - 1;
        reps.push_back(rp);
    }
    const unsigned long long before = mcclx_launch_count(ctx);
    if (mcclx_allreduce_replay_many(ctx, reps.data(), static_cast<uint32_t>(entries)) != MCCLX_OK) {
        printf("FAILED: %s: %s\n", what, mcclx_last_error());
        ++g_bad;
    }
    const unsigned long long launches = mcclx_launch_count(ctx) - before;
    mcclx_queue_drain(ctx);
    if (launches != want) {
        printf("FAILED: %s: %llu launches, expected %llu\n", what, launches, want);
        ++g_bad;
    }
    if (!wire && op == MCCLX_SUM)  // what the stand-in computes
        for (int e = 0; e < entries; ++e)
            for (int r = 0; r < world; ++r)
                for (float v : data[size_t(e * world + r)])
                    if (v != static_cast<float>(world * (world + 1) / 2 + world * e)) {
                        printf("FAILED: %s: entry %d rank %d holds %g\n", what, e, r, static_cast<double>(v));
                        ++g_bad;
                        return launches;
                    }
    return launches;
}
}  // namespace

int main() {
    mcclx_ctx* ctx = nullptr;
    if (mcclx_init(0, &ctx) != MCCLX_OK) return 1;
    // one plan for the whole list, however its entries' sizes alternate: one launch
    list(ctx, "8 ranks, AVG, tree", 8, MCCLX_ALGO_TREE, MCCLX_AVG, 0, MCCLX_REPLAY_FUSED, 1024, 65536, 100, 1);
    list(ctx, "8 ranks, AVG over the codec, ring", 8, MCCLX_ALGO_RING, MCCLX_AVG, 1, MCCLX_REPLAY_DIRECT, 1024, 65536, 100, 1);
    list(ctx, "3 ranks, MAX, ring", 3, MCCLX_ALGO_RING, MCCLX_MAX, 0, MCCLX_REPLAY_FUSED, 1024, 200000, 100, 1);
    list(ctx, "3 ranks, MAX over the codec, tree", 3, MCCLX_ALGO_TREE, MCCLX_MAX, 1, MCCLX_REPLAY_DIRECT, 1024, 200000, 10, 1);
    list(ctx, "5 ranks, SUM over the codec through copies", 5, MCCLX_ALGO_RING, MCCLX_SUM, 1, MCCLX_REPLAY_FUSED, 1024, 65536, 10, 3);
    for (int world = 2; world <= 8; ++world)
        for (int algo : {MCCLX_ALGO_RING, MCCLX_ALGO_TREE, MCCLX_ALGO_BUTTERFLY})
            list(ctx, "SUM", world, algo, MCCLX_SUM, 0, MCCLX_REPLAY_FUSED, 37, 70001, 6, 1);
    // where a workspace lies is asked of runs that are long enough to be cut into pieces only
    null_memory_questions = 0;
    list(ctx, "3 ranks, AVG over the codec through copies", 3, MCCLX_ALGO_RING, MCCLX_AVG, 1, MCCLX_REPLAY_FUSED, 1024, 8192, 40, 2);
    const long asked = null_memory_questions;
    list(ctx, "the same, large", 3, MCCLX_ALGO_RING, MCCLX_AVG, 1, MCCLX_REPLAY_FUSED, 4000000, 4000000, 2, 2);
    if (asked || !null_memory_questions) {
        printf("FAILED: %ld questions about small workspaces, %ld in all\n", asked, null_memory_questions.load());
        ++g_bad;
    }
    {   // a list long enough for three pieces with one bad entry is refused whole, wherever that entry is
        const int entries = 5000;
        std::vector<float> a(size_t(entries) * 4100, 1.f), b(a.size(), 1.f);
        for (int wrong : {0, 2047, 2048, 3000, 4999}) {
            std::vector<void*> p;
            std::vector<mcclx_replay> reps;
            for (int e = 0; e < entries; ++e) {
                p.push_back(&a[size_t(e) * 4100]);
                p.push_back(e == wrong ? nullptr : &b[size_t(e) * 4100]);
            }
            for (int e = 0; e < entries; ++e) reps.push_back(replay(2, MCCLX_ALGO_TREE, MCCLX_SUM, 0, MCCLX_REPLAY_FUSED, e % 3 ? 4100 : 4096, &p[size_t(2 * e)]));
            const unsigned long long before = mcclx_launch_count(ctx);
            const int rc = mcclx_allreduce_replay_many(ctx, reps.data(), uint32_t(entries));
            mcclx_queue_drain(ctx);
            if (rc != MCCLX_ERR_INVALID || mcclx_launch_count(ctx) != before || a[0] != 1.f) {
                printf("FAILED: a bad entry at %d: code %d, %llu launches\n", wrong, rc, static_cast<unsigned long long>(mcclx_launch_count(ctx) - before));
                ++g_bad;
            }
        }
    }
    {
        std::vector<std::vector<float>> data(12, std::vector<float>(4096, 1.f));
        std::vector<void*> p;
        for (auto& d : data) p.push_back(d.data());
        std::vector<mcclx_replay> reps;
        for (int e = 0; e < 4; ++e) reps.push_back(replay(3, MCCLX_ALGO_TREE, MCCLX_AVG, 0, MCCLX_REPLAY_FUSED, 4096, &p[size_t(3 * e)]));
        without_memory(ctx, "a list", [&] { return mcclx_allreduce_replay_many(ctx, reps.data(), 4); });
        without_memory(ctx, "one allreduce", [&] { return mcclx_allreduce_replay(ctx, &reps[1]); });
        without_memory(ctx, "reduce_scatter", [&] {
            return mcclx_reduce_scatter_replay(ctx, 3, &p[0], &p[3], MCCLX_F32, 1024, MCCLX_AVG, MCCLX_REPLAY_FUSED, MCCLX_ACC_STEP);
        });
        without_memory(ctx, "allgather", [&] { return mcclx_allgather_replay(ctx, 3, &p[0], &p[3], 4 * 1024); });
    }
    // what a replay needs does not fall as it grows: sized once for the largest, enough for all
    for (int world = 2; world <= 20; ++world)
        for (int algo : {MCCLX_ALGO_RING, MCCLX_ALGO_TREE, MCCLX_ALGO_BUTTERFLY})
            for (int op : {MCCLX_SUM, MCCLX_MAX})
                for (int wire : {0, 1})
                    for (int mode : {MCCLX_REPLAY_STEPWISE, MCCLX_REPLAY_FUSED, MCCLX_REPLAY_DIRECT}) {
                        uint64_t last = 0;
                        for (uint64_t n = 32; n < (1u << 24); n = n * 5 / 4) {
                            mcclx_replay r = replay(world, algo, op, wire, mode, n, nullptr);
                            const uint64_t need = mcclx_replay_workspace_bytes(&r);
                            if (need < last || (mode == MCCLX_REPLAY_DIRECT && world <= 8 && need)) {
                                printf("FAILED: workspace of world %d algo %d op %d wire %d mode %d numel %llu\n", world, algo,
                                       op, wire, mode, static_cast<unsigned long long>(n));
                                ++g_bad;
                                break;
                            }
                            last = need;
                        }
                    }
    mcclx_destroy(ctx);
    if (!g_bad) printf("ok\n");
    return g_bad ? 1 : 0;
}
