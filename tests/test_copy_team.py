"""The helper threads and the slot ring of the result copies (copy_team.hpp), on the host with a stand-in
for the device: every piece arrives once and unchanged with any number of helpers, also with those that
the system refuses to start, from several callers at once; a failure in any piece ends the copy with its
error; the device is only called by the caller, and the caller waits for a helper only while that one
copies a piece."""
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

#include <algorithm>
#include <cerrno>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

using cfdg::CopyTeam;

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
    std::thread::id caller = std::this_thread::get_id();
    int fail_queue = -1, fail_arrive = -1, strangers = 0, drained = 0;
    std::atomic<int> left{0};
    static inline std::atomic<int> helpers{0};
    explicit Fake(int n) : dev(n * bytes), host(n * bytes), slots(ring * bytes), copied(n), asked(ring) {
        for (std::size_t i = 0; i < dev.size(); ++i) {
            dev[i] = static_cast<char>(i * 7 + i / 251);
        }
    }
};

struct Device {
    Fake* f;
    int queue(int i, int slot) const {
        f->strangers += std::this_thread::get_id() != f->caller;
        if (i == f->fail_queue) {
            return 11;
        }
        std::memcpy(&f->slots[slot * f->bytes], &f->dev[i * f->bytes], f->bytes);
        f->asked[slot] = 0;
        return 0;
    }
    int arrived(int slot, bool& yes) const {
        f->strangers += std::this_thread::get_id() != f->caller;
        yes = ++f->asked[slot] >= 3;
        return slot == f->fail_arrive ? 22 : 0;
    }
    bool copy_out(int i, int slot, int part) const {
        const std::size_t o = part * f->bytes / 4;
        std::memcpy(&f->host[i * f->bytes + o], &f->slots[slot * f->bytes + o], f->bytes / 4);
        ++f->copied[i];
        return part < 3;
    }
    void drain() const { ++f->drained; }
    void leave() const { f->left.fetch_add(1); }
};

// The copy's error, negative if the device was used wrongly.
static int copy(Fake& f, CopyTeam* team) {
    auto ring = std::make_unique<cfdg::RingCopy<Fake::ring, Device>>(Device{&f}, static_cast<int>(f.copied.size()));
    const int e = ring->run(team, 1 + f.helpers++ % CopyTeam::k_helpers);
    const std::vector<char> host = f.host;
    while (f.left.load() == 0) {
    }
    return f.strangers != 0 || host != f.host || f.left != 1 || f.drained != (e != 0) ? -1 : e;
}

static int whole(int n, CopyTeam* team) {
    Fake f(n);
    int bad = copy(f, team) != 0;
    bad += f.host != f.dev;
    for (int c : f.copied) {
        bad += c != 4; // parts
    }
    return bad;
}

// A helper that is kept from leaving a job (as one whose CPU another thread has taken) keeps no caller.
struct Held : CopyTeam::Job {
    std::atomic<int> in{0}, go{0}, out{0};
};

static int late_helper(CopyTeam& team) {
    Held h;
    h.help = [](CopyTeam::Job& j) {
        auto& s = static_cast<Held&>(j);
        s.in.fetch_add(1);
        while (s.go.load() == 0) {
        }
    };
    h.leave = [](CopyTeam::Job& j) { static_cast<Held&>(j).out.fetch_add(1); };
    team.open(h, CopyTeam::k_helpers);
    while (h.in.load() < team.helpers()) {
    }
    team.close(h);
    int bad = h.out.load() != (team.helpers() == 0);
    bad += whole(20, &team); // alone: every helper is in the other job
    h.go.store(1);
    while (h.out.load() == 0) {
    }
    return bad;
}

int main(int argc, char** argv) {
    const int starts = argc > 1 ? std::atoi(argv[1]) : 1 << 30;
    allowed = starts;
    CopyTeam* team = &CopyTeam::get();
    const int wanted = CopyTeam::k_helpers;
    int bad = team->helpers() != std::min(starts, wanted);
    allowed = 1 << 30;
    for (CopyTeam* t : {team, static_cast<CopyTeam*>(nullptr)}) {
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
    bad += late_helper(*team);
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
