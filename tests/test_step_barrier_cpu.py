"""The order of things at the barrier between two steps of a single launch (csrc/step_barrier.h), as it is in the kernel, on every
interleaving of a few workgroups: one that is late by any amount, at any step, whoever gives up its wait meanwhile."""
import os
import subprocess

import pytest

from dldt_amd import build

SOURCE = r"""
#include <array>
#include <cstdio>
#include <set>
#include <vector>

#include "step_barrier.h"

using namespace hipie;

constexpr int kWorkgroups = WORKGROUPS, kSteps = STEPS;

struct Launch {
    struct Place { int8_t step = 0, phase = 0, flag = 1, ended = 0; };      // phase 0: in front of a step's wait, 1: behind its work
    std::array<Place, kWorkgroups> at;
    int8_t count = 0, word = 0, spoiled = 0, gave_up = 0;                   // spoiled: a step ran without what it waited for
    bool operator<(const Launch& o) const { return key() < o.key(); }
    std::array<int8_t, 4 * kWorkgroups + 4> key() const {
        std::array<int8_t, 4 * kWorkgroups + 4> k{};
        for (int i = 0; i < kWorkgroups; ++i) {
            k[4 * i] = at[i].step; k[4 * i + 1] = at[i].phase; k[4 * i + 2] = at[i].flag; k[4 * i + 3] = at[i].ended;
        }
        k[4 * kWorkgroups] = count; k[4 * kWorkgroups + 1] = word; k[4 * kWorkgroups + 2] = spoiled; k[4 * kWorkgroups + 3] = gave_up;
        return k;
    }
};

struct Workgroup {
    Launch& l;
    Launch::Place& p;
    bool dead = false;
    int32_t verdict() const { return p.flag; }
    bool lost(int32_t held) const { return held == 0; }
    void lose() { p.flag = 0; }
    void settle() {}
    void count(bool held) { l.count += held; }
    void tell(uint32_t what) { l.word = static_cast<int8_t>(what); }
};

std::set<Launch> seen;
long ends[2] = {0, 0}, wrong = 0, taken_back = 0, silent = 0, hasty = 0;

void arrive(Workgroup& w) {
#ifdef ADDS_BEFORE_IT_LOOKS
    w.count(true);
    w.dead = w.p.flag == 0;
#else
    arrive_at(w);
#endif
}

void explore(const Launch& now);
void go(const Launch& before, const Launch& next) {
    if (before.word == kReportLost && next.word == kReportDone) ++taken_back;
    if (before.word != kReportDone && next.word == kReportDone)             // the host goes on the moment it sees the word
        for (const auto& p : next.at) hasty += p.step < kSteps;
    explore(next);
}

void explore(const Launch& now) {
    if (!seen.insert(now).second) return;
    bool moved = false;
    for (int i = 0; i < kWorkgroups; ++i) {
        if (now.at[i].ended) continue;
        moved = true;
        Launch next = now;
        Launch::Place& p = next.at[i];
        Workgroup w{next, p};
        if (p.phase == 1) {                                                 // the step's work is done
            arrive(w);
            p.phase = 0;
            ++p.step;
            p.ended = w.dead || (p.step == kSteps && i != 0);
            go(now, next);
            continue;
        }
        const bool waits = p.step != 0, complete = !waits || next.count >= p.step * kWorkgroups;
        if (!complete) {                                                    // its time may be up now (or later: another one moves first)
            give_up(w);
            next.gave_up = 1;
        }
        if (p.step == kSteps) {
            report(w);
            p.ended = 1;
        } else {
            next.spoiled |= !complete;
            p.phase = 1;
        }
        go(now, next);
    }
    if (moved) return;
    ++ends[now.gave_up];
    wrong += now.word == kReportDone && now.spoiled;
    silent += now.word == 0 || (!now.gave_up && now.word != kReportDone);
}

int main() {
    explore(Launch());
    std::printf("%zu %ld %ld %ld %ld %ld %ld\n", seen.size(), ends[0], ends[1], wrong, taken_back, silent, hasty);
    return 0;
}
"""


def _explore(tmp_path, workgroups, steps, *flags):
    source, program = tmp_path / "barrier.cpp", tmp_path / "barrier"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-I", build.CSRC, "-DWORKGROUPS=%d" % workgroups, "-DSTEPS=%d" % steps, *flags,
                    str(source), "-o", str(program)], check=True)
    states, whole, given_up, wrong, taken_back, silent, hasty = map(int, subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.split())
    assert states > 10 and whole >= 1 and given_up >= 1
    return wrong, taken_back, silent, hasty


@pytest.mark.parametrize("workgroups,steps", [(2, 1), (2, 2), (2, 4), (3, 1), (3, 3), (4, 2)])
def test_a_launch_that_was_given_up_anywhere_is_never_reported_as_done(tmp_path, workgroups, steps):
    """and one that nobody gave up always is, when every workgroup has done its last step's work"""
    assert _explore(tmp_path, workgroups, steps) == (0, 0, 0, 0)


@pytest.mark.parametrize("workgroups,steps", [(2, 2), (3, 3)])
def test_the_search_finds_what_an_addition_in_front_of_the_verdict_gets_wrong(tmp_path, workgroups, steps):
    wrong, taken_back, silent, _ = _explore(tmp_path, workgroups, steps, "-DADDS_BEFORE_IT_LOOKS")
    assert wrong > 0 and taken_back > 0 and silent == 0


def test_the_kernel_goes_by_this_order():
    text = open(os.path.join(build.CSRC, "program.hip")).read()
    assert text.count("arrive_at(*this)") == 1 and text.count("report(*this)") == 1 and text.count("give_up(*this)") == 1
    assert text.count("tell(") == 2                              # its definition, and a roll call that was cancelled
