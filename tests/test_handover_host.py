"""The hand-over of query counts (csrc/handover.h) compiled for the host, a thread a lane: places, and what is left for the caller
where a workgroup gives up waiting, whenever it does so.  A word that comes late is one the test holds back; the wait is cut short by
its own limit."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vtpack_amd", "csrc")
PROGRAM = r"""
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <atomic>
#include <functional>
#include <thread>
#include <vector>
#define __device__
#define __forceinline__ inline
#define __HIP_MEMORY_SCOPE_AGENT 0
constexpr int WAVE = 64;
struct Wave {
    std::atomic<int> here{0}, turn{0};
    unsigned long long bits[64];
    float values[64];
    void meet()
    {
        const int t = turn;
        if (++here == 64) { here = 0; turn++; }
        else while (turn == t) std::this_thread::yield();
    }
};
struct Lane { unsigned x; };
static thread_local Lane threadIdx;
static thread_local Wave *wave;
static std::function<void(void *, bool)> on_access;      // before a load or store of lane 0
static void seen(const void *p, bool store) { if (threadIdx.x == 0 && on_access) on_access((void *)p, store); }
template <typename T> T load(const T *p) { seen(p, false); return __atomic_load_n(p, __ATOMIC_SEQ_CST); }
template <typename T, typename V> void store(T *p, V v) { seen(p, true); __atomic_store_n(p, (T)v, __ATOMIC_SEQ_CST); }
template <typename T> T exchange(T *p, T v) { seen(p, true); return __atomic_exchange_n(p, v, __ATOMIC_SEQ_CST); }
#define __hip_atomic_load(p, order, scope) load(p)
#define __hip_atomic_store(p, v, order, scope) store(p, v)
#define __hip_atomic_exchange(p, v, order, scope) exchange(p, v)
static unsigned long long __builtin_amdgcn_ballot_w64(bool b)
{
    wave->bits[threadIdx.x] = b;
    wave->meet();
    unsigned long long r = 0;
    for (int i = 0; i < 64; i++) r |= wave->bits[i] << i;
    wave->meet();
    return r;
}
static float wave_sum(float v)
{
    wave->values[threadIdx.x] = v;
    wave->meet();
    float r = 0.f;
    for (int i = 0; i < 64; i++) r += wave->values[i];
    wave->meet();
    return r;
}
static void __builtin_amdgcn_s_sleep(int) {}
template <int N> void wait_vmcnt() {}
#include "handover.h"
using namespace vtdge;

constexpr int WGS = 150, CAPACITY = 16 * WGS;
static unsigned long long status[1 + WGS];
static int64_t total;
static int queries(int wg) { return 1 + 5 * wg % 16; }
static int before(int wg)
{
    int n = 0;
    for (int i = 0; i < wg; i++) n += queries(i);
    return n;
}
static void lanes(std::function<void()> f)
{
    Wave w;
    std::vector<std::thread> all;
    for (unsigned i = 0; i < 64; i++) all.emplace_back([&, i] { threadIdx.x = i; wave = &w; f(); });
    for (auto &t : all) t.join();
}
static void publish(int wg) { threadIdx.x = 0; chain_publish(status + 1, wg, queries(wg)); }
static long long run(int wg)
{
    std::vector<long long> got(64);
    lanes([&] {
        const unsigned i = threadIdx.x;
        got[i] = chain_rows_before(status, wg, queries(wg), CAPACITY, &total, 20);
        if (wg == WGS - 1 && i == 0) chain_total(status, &total, got[i] + queries(wg), CAPACITY);
    });
    for (long long v : got) if (v != got[0]) { printf("lanes differ\n"); exit(1); }
    return got[0];
}
#define CHECK(x) do { if (!(x)) { printf("line %d: %s (total %lld)\n", __LINE__, #x, (long long)total); exit(1); } } while (0)
// workgroup `late` gives up: a word it needs is there for the others only
static void give_up(int late)
{
    const int held = late % 64 ? late - 1 : late - 64 + 63;      // its neighbour's count, or the sum of the group before
    const unsigned long long word = status[1 + held];
    status[1 + held] = 0;
    auto hook = on_access;
    on_access = nullptr;
    CHECK(run(late) == CAPACITY);
    on_access = hook;
    status[1 + held] = word;
}
int main(int argc, char **argv)
{
    const int when = atoi(argv[1]), late = atoi(argv[2]), last = WGS - 1;
    memset(status, 0, sizeof(status));
    total = -7;                                                  // not cleared by anybody
    for (int i = 0; i < WGS; i++) publish(i);
    if (when == 0) {                                             // nobody gives up, whatever lay in the total's place
        if (late) total = CAPACITY + 1;
        for (int i : {0, 1, 2, 62, 63, 64, 65, 126, 127, 128, 148, 149}) CHECK(run(i) == before(i));
        CHECK(status[0] == 0 && total == before(WGS));
        return 0;
    }
    for (int i = 0; i < last; i++) {
        if (i == late && when == 1) give_up(late);               // long before the last workgroup
        else if (i % 64 == 63) run(i);                           // (says the sum of its group)
    }
    int times = 0;
    auto once = [&](void *p, bool st, void *at, bool want) { return p == at && st == want && times++ == 0; };
    if (when == 1) run(last);
    if (when == 2) { run(last); give_up(late); }                 // after it
    if (when == 3) {                                             // another before it, this one between its total and its look at the flag
        give_up(late == 40 ? 41 : 40);
        on_access = [&](void *p, bool st) { if (once(p, st, status, false)) give_up(late); };
        run(last);
        CHECK(times > 0);
    }
    if (when == 4) {                                             // before its total
        on_access = [&](void *p, bool st) { if (once(p, st, &total, true)) give_up(late); };
        run(last);
        CHECK(times > 0);
    }
    if (when == 5) {                                             // the last between the flag of the other and its total
        const int held = late % 64 ? late - 1 : late - 64 + 63;
        const unsigned long long word = status[1 + held];
        status[1 + held] = 0;
        on_access = [&](void *p, bool st) {
            if (!once(p, st, &total, true)) return;
            status[1 + held] = word;
            std::thread(run, last).join();
        };
        CHECK(run(late) == CAPACITY);
        CHECK(times > 0);
    }
    CHECK(status[0] == 1 && total > CAPACITY);
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("needs g++")
    folder = tmp_path_factory.mktemp("handover")
    (folder / "main.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-I", CSRC, str(folder / "main.cpp"), "-o", str(folder / "main"), "-lpthread"],
                   check=True, capture_output=True)
    return str(folder / "main")


def _go(program, when, late):
    r = subprocess.run([program, str(when), str(late)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.parametrize("past", [0, 1])
def test_places(program, past):
    _go(program, 0, past)


@pytest.mark.parametrize("when", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("late", [1, 40, 62, 63, 64, 100, 127, 148])
def test_a_workgroup_that_gives_up_shows_in_the_total(program, when, late):
    _go(program, when, late)
