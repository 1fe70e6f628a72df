"""The meeting of a DEM step's workgroups (hybird_amd/csrc/dem_barrier.h), run on the host.

One thread stands for each workgroup, the words are atomics and the clock is the host's, so that workgroups can be made
late without a GPU.
"""
import os
import shutil
import subprocess

import pytest

from helpers import ROOT

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")

HEAD = r"""
#include <atomic>
#include <chrono>
#include <cstddef>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <thread>
#include <vector>
#define __host__
#define __device__
#define __forceinline__ inline
#include "dem_barrier.h"
using namespace hyb;

struct HostWords {  // 1 tick: 1 us
    static u64 load(u64* w) { return __atomic_load_n(w, __ATOMIC_SEQ_CST); }
    static void store(u64* w, u64 v) { __atomic_store_n(w, v, __ATOMIC_SEQ_CST); }
    static u64 swap(u64* w, u64 from, u64 to) {
        __atomic_compare_exchange_n(w, &from, to, false, __ATOMIC_SEQ_CST, __ATOMIC_SEQ_CST);
        return from;
    }
    static unsigned add(unsigned* w, unsigned v) { return __atomic_fetch_add(w, v, __ATOMIC_SEQ_CST); }
    static u64 now() {
        return (u64)std::chrono::duration_cast<std::chrono::microseconds>(
            std::chrono::steady_clock::now().time_since_epoch()).count();
    }
    static void pause() { std::this_thread::yield(); }
};
constexpr u64 LONG = 60000000;

void check(bool ok, const char* what) {
    if (ok) return;
    std::printf("failed: %s\n", what);
    std::exit(1);
}
void late(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }
template <class F>
void launch(int nwg, F&& f) {
    std::vector<std::thread> t;
    for (int wg = 0; wg < nwg; ++wg) t.emplace_back([&f, wg] { f(wg); });
    for (std::thread& x : t) x.join();
}
"""


def _run(tmp_path, body):
    src, exe = tmp_path / "meet.cpp", tmp_path / "meet"
    src.write_text(HEAD + body)
    subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-I", os.path.join(ROOT, "hybird_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr


def test_every_meeting_gives_every_workgroup_the_maximum(tmp_path):
    """Several launches, each with another number of meetings: the sets of words rotate on over the launches."""
    _run(tmp_path, r"""
int main() {
    for (int nwg : {2, 3, 7}) {
        std::vector<u64> words(4 * nwg, SLOT_EMPTY);
        unsigned kept = 0;
        for (int l = 0; l < 40; ++l) {
            const int meetings = 1 + l % 5;
            const unsigned from = kept;
            launch(nwg, [&](int wg) {
                std::mt19937 rng(1000 * l + wg);
                Meeting<HostWords> m{words.data(), from, nwg};
                for (int k = 0; k < meetings; ++k) {
                    if (rng() % 8 == 0) late(1);
                    m.arrive(wg, (u64)(100 * k + wg));
                    const u64 v = m.wait_all(0, 1, LONG);
                    check(v == (u64)(100 * k + nwg - 1), "maximum");
                    m.free_last(wg);
                    ++m.n;
                }
                if (leaving(wg, 0) == LEAVE_STATE) kept = m.n % 3u + 3u;
            });
        }
    }
    return 0;
}
""")


def test_a_wait_that_ends_without_the_others_is_reported(tmp_path):
    """At the last meeting workgroup 1 gives up on the late workgroup 2; the first one comes later still and finds
    everybody's word. The launch must not count as done."""
    _run(tmp_path, r"""
int main() {
    const int nwg = 3;
    std::vector<u64> words(4 * nwg, SLOT_EMPTY);
    std::atomic<int> error{0}, gone{0};
    launch(nwg, [&](int wg) {
        Meeting<HostWords> m{words.data(), 0, nwg};
        if (wg == 2) while (!gone.load()) late(1);
        if (wg == 0) while (HostWords::load(&m.set(0)[2]) == SLOT_EMPTY) late(1);
        m.arrive(wg, 5);
        const u64 v = m.wait_all(0, 1, wg == 1 ? 2000 : LONG);
        if (wg == 1) { check(v == SLOT_TIMEOUT, "workgroup 1 gives up"); gone = 1; }
        if (wg == 0) check(v == 5, "workgroup 0 finds all words");
        if (leaving(wg, v == SLOT_TIMEOUT ? 7 : 0) == LEAVE_ERROR) error = 7;
    });
    check(error == 7, "the launch is reported as failed");
    return 0;
}
""")


def test_a_roll_call_has_one_verdict(tmp_path):
    """Workgroups that are late at random, against a short wait: all come to the same verdict; a refused launch is done
    once, by the last to leave; the launches after it meet as ever."""
    _run(tmp_path, r"""
int main() {
    int together = 0, apart = 0;
    for (int nwg : {2, 5}) {
        std::vector<u64> words(4 * nwg, SLOT_EMPTY);
        for (int wg = 0; wg < nwg; ++wg) words[3 * nwg + wg] = 0;
        unsigned kept = 0, left = 0;
        for (int l = 0; l < 150; ++l) {
            const unsigned from = kept;
            std::atomic<int> present{0}, refused{0}, done{0};
            const u64 wait = l % 10 == 0 ? 0 : 1500;
            launch(nwg, [&](int wg) {
                std::mt19937 rng(1000 * l + wg);
                if (rng() % 4 == 0) late((int)(rng() % 4));
                Meeting<HostWords> m{words.data(), from, nwg};
                const u64 checked = m.check_in(wg, l, wait);
                if (rng() % 4 == 0) late((int)(rng() % 3));
                m.arrive(wg, checked);
                const u64 verdict = m.call(0, 1, l, wait, LONG);
                if (verdict == SLOT_REFUSED) {
                    ++refused;
                    if (m.last_out(&left)) {
                        check(refused == nwg, "everybody has left");
                        m.clear_all(0, 1, l);
                        left = 0;
                        ++done;
                    }
                    return;
                }
                check(verdict == SLOT_PRESENT, "present or refused");
                m.free_last(wg);
                ++m.n;
                ++present;
                for (int k = 0; k < 1 + l % 4; ++k) {
                    m.arrive(wg, (u64)(10 * k + wg));
                    check(m.wait_all(0, 1, LONG) == (u64)(10 * k + nwg - 1), "maximum after the roll call");
                    m.free_last(wg);
                    ++m.n;
                }
                if (leaving(wg, 0) == LEAVE_STATE) {
                    kept = m.n % 3u + 3u;
                    ++done;
                }
            });
            check((present == nwg && refused == 0) || (present == 0 && refused == nwg), "one verdict");
            check(done == 1, "the step is done once");
            check(wait || refused == nwg, "no wait, nobody present");
            (refused ? apart : together) += 1;
        }
    }
    check(together > 10 && apart > 10, "both verdicts occur");
    return 0;
}
""")
