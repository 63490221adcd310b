"""The helper threads and the slot ring of the result copies (copy_team.hpp), on the host with a stand-in
for the device: every piece arrives once and unchanged with any number of helpers, also with those that
the system refuses to start, from several callers at once, and a failure in any piece ends the copy with
its error."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from .conftest import ROOT

CXX = shutil.which("g++") or shutil.which("c++")

PROGRAM = r"""
#include "copy_team.hpp"

#include <dlfcn.h>
#include <pthread.h>

#include <cerrno>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

static int allowed = 1 << 30; // threads that may still be started

extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) {
    static auto* real = reinterpret_cast<decltype(&pthread_create)>(dlsym(RTLD_NEXT, "pthread_create"));
    return allowed-- > 0 ? real(t, a, f, arg) : EAGAIN;
}

// Pieces of 64 KiB; a queued piece is in its slot at once and reported at the third question.
struct Fake {
    static constexpr std::size_t bytes = 1 << 16;
    static constexpr int ring = 8;
    std::vector<char> dev, host, slots;
    std::vector<int> copied, asked;
    int fail_queue = -1, fail_arrive = -1;
    explicit Fake(int n) : dev(n * bytes), host(n * bytes), slots(ring * bytes), copied(n), asked(ring) {
        for (std::size_t i = 0; i < dev.size(); ++i) {
            dev[i] = static_cast<char>(i * 7 + i / 251);
        }
    }
    int enter() { return 0; }
    int queue(int i, int slot) {
        if (i == fail_queue) {
            return 11;
        }
        std::memcpy(&slots[slot * bytes], &dev[i * bytes], bytes);
        asked[slot] = 0;
        return 0;
    }
    int arrived(int slot, bool& yes) {
        yes = ++asked[slot] >= 3;
        return slot == fail_arrive ? 22 : 0;
    }
    void copy_out(int i, int slot) {
        std::memcpy(&host[i * bytes], &slots[slot * bytes], bytes);
        ++copied[i];
    }
};

static int copy(Fake& f, cfdg::CopyTeam* team) {
    return cfdg::RingCopy<Fake::ring, Fake>(f, static_cast<int>(f.copied.size())).run(team);
}

static int whole(int n, cfdg::CopyTeam* team) {
    Fake f(n);
    int bad = copy(f, team) != 0;
    bad += f.host != f.dev;
    for (int c : f.copied) {
        bad += c != 1;
    }
    return bad;
}

int main(int argc, char** argv) {
    const int starts = argc > 1 ? std::atoi(argv[1]) : 1 << 30;
    allowed = starts;
    cfdg::CopyTeam* team = &cfdg::CopyTeam::get();
    int bad = team->helpers() != std::min(starts, static_cast<int>(cfdg::CopyTeam::k_helpers));
    allowed = 1 << 30;
    for (cfdg::CopyTeam* t : {team, static_cast<cfdg::CopyTeam*>(nullptr)}) {
        for (int n : {0, 1, 7, 8, 9, 16, 100}) {
            for (int rep = 0; rep < 5; ++rep) {
                bad += whole(n, t);
            }
        }
        for (int piece : {0, 7, 8, 50}) {
            Fake q(60), a(60);
            q.fail_queue = piece;
            bad += copy(q, t) != 11;
            a.fail_arrive = piece % Fake::ring;
            bad += copy(a, t) != 22;
        }
    }
    std::vector<std::thread> callers;
    std::atomic<int> wrong{0};
    for (int k = 0; k < 6; ++k) {
        callers.emplace_back([&, k] {
            for (int rep = 0; rep < 12; ++rep) {
                wrong += whole(5 + 13 * k, team);
            }
        });
    }
    for (std::thread& t : callers) {
        t.join();
    }
    bad += wrong;
    std::printf("%d\n", bad);
    return bad != 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if CXX is None:
        pytest.skip("no C++ compiler")
    d = tmp_path_factory.mktemp("copy_team")
    (d / "copy.cpp").write_text(PROGRAM)
    subprocess.run([CXX, "-O1", "-g", "-std=c++17", "-fsanitize=address", "-pthread", "-rdynamic", "-I", str(ROOT / "cfd_amd" / "csrc"),
                    str(d / "copy.cpp"), "-o", str(d / "copy"), "-ldl"], check=True, timeout=300)
    return d / "copy"


@pytest.mark.parametrize("starts", [0, 1, 2, 3])
def test_copies_with_as_many_helpers_as_start(program, starts):
    out = subprocess.run([str(program), str(starts)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
