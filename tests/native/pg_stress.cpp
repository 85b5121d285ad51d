// pg_stress.cpp -- the ownership side of the c10d backend under a sanitizer, without a GPU: the real
// ProcessGroupMCCL, WorkMCCL, Progress, LocalMesh, HostWire and chunk scheduler, compiled with
// -DMCCL_NULL_DEVICE (backend/Device.hpp) over a host stand-in of the kernel layer
// (null_mcclx.cpp).  Groups of 2-5 rank threads come and go; every second group completes its
// allreduces event-based (completer thread, two queues, parked buckets).  What the test is after
// is who lets go of what, where:
//   * the registry of meshes and shared contexts while ranks join and leave at different times;
//   * Works and Futures settled on the engine and completer threads;
//   * the LAST reference to a process group dropped by a Future callback on the group's own
//     engine thread, and on the mesh's completer thread -- the group, its engine, the shared
//     context and the completer are then destroyed from inside one of their own tasks.
// Results of the fp32 sums are checked, so that a buffer freed or reused too early shows up as
// a wrong value as well as a sanitizer report.  WAIT_MS = 0 makes every wait untimed (a timed
// wait is pthread_cond_clockwait, which ThreadSanitizer builds of this toolchain do not model).
#include <torch/csrc/distributed/c10d/HashStore.hpp>

#include <ATen/ATen.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
#include <vector>

#include "backend/ProcessGroupMCCL.hpp"

#ifndef WAIT_MS
#define WAIT_MS 0
#endif

using namespace mccl;

namespace {
std::atomic<long> g_bad{0}, g_checked{0};

void expect(const at::Tensor& t, float want) {
    const float* p = t.data_ptr<float>();
    for (int64_t i = 0; i < t.numel(); ++i)
        if (p[i] != want) {
            ++g_bad;
            return;
        }
    ++g_checked;
}

void settled(const c10::intrusive_ptr<c10d::Work>& w) { w->getFuture()->wait(); }  // untimed, and the Work has settled after it
// Lists whose entries depend on each other run entry by entry, in the order of the list, as
// separate calls would: an entry that reads what an earlier one writes sees it, and of several
// copies into one tensor the last one stays.
void lists(ProcessGroupMCCL& pg, int rank, int world) {
    auto full = [](float v) { return at::full({19}, v); };
    auto outputs = [&] {
        std::vector<at::Tensor> t;
        for (int p = 0; p < world; ++p) t.push_back(full(-1.0f));
        return t;
    };
    // entry 1's input is entry 0's first output: everybody ends with rank 0's value
    std::vector<std::vector<at::Tensor>> chain = {outputs(), outputs()};
    std::vector<at::Tensor> in = {full(float(rank + 10)), chain[0][0]};
    pg.allgather(chain, in)->wait();
    for (int p = 0; p < world; ++p) {
        expect(chain[0][size_t(p)], float(p + 10));
        expect(chain[1][size_t(p)], 10.0f);
    }
    // one tensor in the place of every output: the last rank's value
    at::Tensor one = full(-1.0f);
    std::vector<std::vector<at::Tensor>> same = {std::vector<at::Tensor>(size_t(world), one)};
    std::vector<at::Tensor> mine = {full(float(rank + 20))};
    pg.allgather(same, mine)->wait();
    expect(one, float(world + 19));
    // in place: an output is the input itself, twice in the list
    std::vector<std::vector<at::Tensor>> own = {outputs(), outputs()};
    std::vector<at::Tensor> ins;
    for (int e = 0; e < 2; ++e) {
        own[size_t(e)][size_t(rank)].fill_(float(rank + 30 + 100 * e));
        ins.push_back(own[size_t(e)][size_t(rank)]);
    }
    pg.allgather(own, ins)->wait();
    for (int e = 0; e < 2; ++e)
        for (int p = 0; p < world; ++p) expect(own[size_t(e)][size_t(p)], float(p + 30 + 100 * e));
    // a tensor named twice where the root has two
    at::Tensor a = full(float(rank)), b = full(float(rank + 40));
    std::vector<at::Tensor> list = {a, rank == 0 ? b : a};
    c10d::BroadcastOptions root;
    root.rootRank = 0;
    pg.broadcast(list, root)->wait();
    expect(a, rank == 0 ? 0.0f : 40.0f);
}
}  // namespace

int main(int argc, char** argv) {
    const int groups = argc > 1 ? atoi(argv[1]) : 60;
    for (int g = 0; g < groups; ++g) {
        const int world = g % 10 == 9 ? 5 : 2 + g % 3;  // (five: sums go back into every operand)
        const bool async = (g & 1) != 0;
        if (async)
            setenv("MCCL_ALLREDUCE_ASYNC", "1", 1);
        else
            unsetenv("MCCL_ALLREDUCE_ASYNC");
        if (g % 4 == 3)
            setenv("MCCL_ASYNC_QUEUES", "1", 1);
        else
            unsetenv("MCCL_ASYNC_QUEUES");
        auto store = c10::make_intrusive<c10d::HashStore>();
        const float total = world * (world + 1) / 2.0f;
        std::vector<std::thread> ts;
        for (int r = 0; r < world; ++r)
            ts.emplace_back([&, r] {
                ProcessGroupMCCL::Options opts;
                opts.timeout = std::chrono::milliseconds(WAIT_MS);
                auto pg = c10::make_intrusive<ProcessGroupMCCL>(store, r, world, opts);
                c10d::AllreduceOptions sum;
                // a few buckets back to back (in the event-based mode they park and coalesce)
                std::vector<std::vector<at::Tensor>> buckets;
                std::vector<c10::intrusive_ptr<c10d::Work>> works;
                for (int b = 0; b < 5; ++b) {
                    buckets.push_back({at::full({1000 + 37 * b}, float(r + 1))});
                    works.push_back(pg->allreduce(buckets.back(), sum));
                }
                for (int b = 4; b >= 0; --b) {
                    works[size_t(b)]->wait();
                    settled(works[size_t(b)]);
                    expect(buckets[size_t(b)][0], total);
                }
                works.clear();
                // engine-thread collectives
                at::Tensor mine = at::full({33}, float(r)), all = at::empty({33 * world});
                auto wg = pg->_allgather_base(all, mine);
                auto wb = pg->barrier();
                wg->wait();
                wb->wait();
                for (int p = 0; p < world; ++p)
                    if (all.data_ptr<float>()[33 * p] != float(p)) ++g_bad;
                lists(*pg, r, world);
                // the last reference to the group goes with a Future callback: on the completer
                // thread (event-based allreduce) or on the group's own engine thread (barrier)
                std::vector<at::Tensor> last = {at::full({257}, float(r + 1))};
                c10::intrusive_ptr<c10d::Work> w = (g % 3 == 0) ? pg->barrier() : pg->allreduce(last, sum);
                auto fut = w->getFuture();
                fut->addCallback([keep = pg](c10::ivalue::Future&) {});
                pg.reset();   // this thread lets go first
                w.reset();
                fut->wait();
                if (g % 3 != 0) expect(last[0], total);
                fut.reset();  // whoever held the callback last has destroyed the group by now, or does so here
            });
        for (auto& t : ts) t.join();
    }
    if (g_bad.load()) {
        printf("FAILED: %ld wrong results\n", g_bad.load());
        return 1;
    }
    printf("ok: %d groups, %ld results checked\n", groups, g_checked.load());
    return 0;
}
