"""A level-0 kernel's own rows are read and written at their places in arrays of any length: the
kernels' row functions, compiled for the host, on a sparse mapping of more than 2^30 values (an offset
of 32 bits wraps to the array's beginning from 2^29 FP64 values on)."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from .conftest import ROOT

HIPCC = shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")

PROGRAM = r"""
#include "kernels.hpp"
#include <sys/mman.h>
#include <cstdio>

using namespace cfdg;

long long place(unsigned r) { return r; }
long long place(const LaneRow& r) { return r.start + r.lane; }

template <int Form, class T>
int wrong(int n) {
    const std::size_t bytes = static_cast<std::size_t>(n) * sizeof(T);
    void* m = mmap(nullptr, bytes, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
    if (m == MAP_FAILED) {
        return -1;
    }
    T* a = static_cast<T*>(m);
    gmem_t<T>* g = (gmem_t<T>*)a;
    int bad = 0;
    const int last = (n - 1) / k_wave;
    const int ds = 5;
    for (long long first : {0LL, 1LL, (1LL << 22) - 3, 1LL << 23, (1LL << 23) + 1, 1LL << 24, (long long)last - ds, (long long)last}) {
        if (first < 0 || first > last) {
            continue;
        }
        const int slice = static_cast<int>(first);
        for (int lane = 0; lane < k_wave; ++lane) {
            long long want[2];
            for (int h = 0; h < 2; ++h) {
                want[h] = (slice + static_cast<long long>(h) * ds) * k_wave + lane;
                if (want[h] < n) {
                    a[want[h]] = static_cast<T>(h + 1 + lane);
                }
            }
            T got[2] = {};
            RowOf<Form> row[2];
            own_rows<2>(slice, ds, lane, n, row, [&](int h, const auto& r) {
                bad += place(r) < 0 || place(r) >= n; // also for a row past the end
                got[h] = load_at<T>((const gmem_t<const T>*)g, r);
            });
            for (int h = 0; h < 2; ++h) {
                bad += inside(row[h], n) != (want[h] < n);
                if (want[h] < n) {
                    bad += got[h] != static_cast<T>(h + 1 + lane);
                    store_at<T>(g, row[h], static_cast<T>(-7));
                    bad += a[want[h]] != static_cast<T>(-7);
                    a[want[h]] = T(0);
                }
            }
        }
    }
    munmap(m, bytes);
    return bad;
}

int main() {
    int bad = 0;
    for (int n : {1, 63, 64, 65, 700, (1 << 29) - 1}) {
        bad += wrong<L0_SYM7, double>(n) != 0; // symmetric storage ends here
    }
    for (int n : {1, 63, 64, 65, 700, (1 << 29) - 1, 1 << 29, (1 << 29) + 1, (1 << 30) + 77}) {
        bad += wrong<L0_ANY, double>(n) != 0;
        bad += wrong<L0_ANY, float>(n) != 0;
        bad += wrong<L0_CSR, double>(n) != 0;
    }
    std::printf("%d\n", bad);
    return bad != 0;
}
"""


@pytest.mark.skipif(HIPCC is None, reason="hipcc not present")
def test_own_rows_of_arrays_past_32_bit_offsets(tmp_path):
    src = tmp_path / "rows.hip"
    src.write_text(PROGRAM)
    exe = tmp_path / "rows"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-x", "hip", "--offload-arch=gfx950", "-w", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I", str(ROOT / "cfd_amd" / "csrc"), "-I", str(ROOT / "include"), str(src),
                    "-o", str(exe)], check=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
