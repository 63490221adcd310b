// Device kernels of the AMG-PCG / Krylov backend for gfx950 (CDNA4, wave64).
//
// Layout. Every matrix is sliced ELL with a slice height of 64 rows, one wavefront per slice:
// entry k of row (64 s + lane) sits at sp[s] + 64 k + lane, so each load instruction of a wave
// reads 64 consecutive column indices / values. Rows keep the CSR (ascending column) order of
// the reference and padding entries (value 0) come last, so an FP64 row sum equals the
// reference's serial sum (src/gpu/src/krylov_kernels.inc:12-25) bit for bit. A workgroup is
// four wavefronts = four slices = 256 rows.
//
// Work mapping. A launch covers the rows of one level for a set of systems: block b processes
// the 256-row block blocks[b].y of system blocks[b].x. A single solve is a set of one system.
//
// Reductions. Dot products never use atomics: each group of rows (at most k_max_groups a system)
// gets one partial sum (wave butterfly, then the four wave sums in order), and the kernel that needs
// the dot product adds the partials in a fixed order in its prologue (take_step). Results are
// reproducible run to run and do not depend on which other systems share the launch.
//
// Control. Each system carries a SolveState; kernels of a system whose status is non-zero
// return at once, so the host may enqueue iterations ahead of the convergence test.
#pragma once

#include "layout.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

namespace cfdg {

// ------------------------------------------------------------------------------------------
// Arithmetic helpers. The library is compiled with -ffp-contract=off; FP32 kernels use
// explicit fused multiply-adds, FP64 kernels keep the reference's separate multiply and add.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ double madd(double a, double b, double c) { return c + a * b; }
__device__ __forceinline__ float madd(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

template <class T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_xor(v, off, k_wave);
    }
    return v;
}

// Sums one value per thread over the block; thread 0 receives the result.
template <int N>
__device__ __forceinline__ void block_sums(double (&v)[N], double (&out)[N]) {
    __shared__ double red[N][k_slices_per_block];
    const int wave = threadIdx.x / k_wave;
    const int lane = threadIdx.x % k_wave;
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const double w = wave_sum(v[q]);
        if (lane == 0) {
            red[q][wave] = w;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < N; ++q) {
            double s = red[q][0];
#pragma unroll
            for (int w = 1; w < k_slices_per_block; ++w) {
                s += red[q][w];
            }
            out[q] = s;
        }
    }
}

__device__ __forceinline__ float bf16_to_float(unsigned short h) {
    return __uint_as_float(static_cast<unsigned>(h) << 16);
}

// Device buffers seen in the global address space: loads through such pointers compile to
// global_load with a scalar base instead of flat loads (which also count against the LDS
// counter and need a full 64-bit address per lane). Descriptor pointers are generic.
template <class T>
using gmem_t = __attribute__((address_space(1))) T;

template <class T>
__device__ __forceinline__ gmem_t<T>* gm(T* p) {
    return (gmem_t<T>*)p;
}

// Element i of an array whose base is the same for the whole wavefront: the base stays in scalar
// registers and the address is one 32-bit byte offset per lane (i sizeof(T) < 2^32), which all the
// loads of a row share.
template <class T>
__host__ __device__ __forceinline__ T load_at(const gmem_t<const T>* __restrict__ base, unsigned i) {
    return *(const gmem_t<const T>*)((const gmem_t<const char>*)base + i * static_cast<unsigned>(sizeof(T)));
}

template <class T>
__host__ __device__ __forceinline__ void store_at(gmem_t<T>* __restrict__ base, unsigned i, T v) {
    *(gmem_t<T>*)((gmem_t<char>*)base + i * static_cast<unsigned>(sizeof(T))) = v;
}

// A lane's row in a slice of 64, for arrays of any length: the slice's first row, the same for the
// whole wavefront, moves the scalar base, and only the lane's place in the slice is a vector offset.
struct LaneRow {
    long long start;
    unsigned lane;
    int left; // rows from start to the end of the matrix; at most 0 past it
};

template <class T>
__host__ __device__ __forceinline__ T load_at(const gmem_t<const T>* __restrict__ base, const LaneRow& r) {
    return load_at<T>(base + r.start, r.lane);
}

template <class T>
__host__ __device__ __forceinline__ void store_at(gmem_t<T>* __restrict__ base, const LaneRow& r, T v) {
    store_at<T>(base + r.start, r.lane, v);
}

// Column index of the lane's entry in the 64 slots from k on (uniform over the wavefront): 32-bit
// columns (ColAbs), row + 16-bit offset (ColOff, square matrices), the slice's base column + unsigned
// 16-bit offset (ColBase, transfer operators) or row + the slice's stencil offset of round k
// (ColStencil, square matrices, one lane per row). The format is chosen once per matrix (a uniform
// branch), never per slot: a per-lane pointer test would turn every column load into a divergent
// branch with its own wait.
struct ColAbs {
    const gmem_t<const int>* __restrict__ col;
    unsigned lane;
    __device__ __forceinline__ int operator()(int k) const { return load_at<int>(col + k, lane); }
};

struct ColOff {
    const gmem_t<const short>* __restrict__ dcol;
    unsigned lane;
    int row;
    __device__ __forceinline__ int operator()(int k) const { return row + static_cast<int>(load_at<short>(dcol + k, lane)); }
};

struct ColBase {
    const gmem_t<const unsigned short>* __restrict__ dcol;
    unsigned lane;
    int base;
    __device__ __forceinline__ int operator()(int k) const {
        return base + static_cast<int>(load_at<unsigned short>(dcol + k, lane));
    }
};

// Stencil column: the slice's offset table (uniform over the wavefront) added to the row,
// clamped to [0, last] for the value-0 slots of rows that lack an offset.
struct ColStencil {
    const gmem_t<const int>* __restrict__ off;
    int row;
    int last;
    __device__ __forceinline__ int operator()(int k) const { return min(max(row + off[k / k_wave], 0), last); }
};

template <class T, class V>
__device__ __forceinline__ T value_at(const gmem_t<const V>* __restrict__ val, unsigned lane) {
    if constexpr (sizeof(V) == 2) {
        return bf16_to_float(load_at<V>(val, lane));
    } else {
        return load_at<V>(val, lane);
    }
}

// Entries of a sliced-ELL row whose loads are issued together. FP32: 6 (level 1 of a 16-system batch,
// 4 / 6 / 8 entries: sweep 16.3 / 14.6 / 17.3 us, level-0 prolongation 13.5 / 12.1 / 15.6; 128^3 within
// 4%, 4 and 6 alike). FP64: 4 (128^3: level-1 sweep 20.8 / 21.7 / 24.7, restriction 33.8 / 34.9 / 36.3).
template <class T>
constexpr int ell_group() {
    return sizeof(T) == 4 ? 6 : 4;
}

// Storage-order row sum of sliced-ELL slots with values val (type V) converted to T. Loads are
// issued ell_group entries at a time, the tail (w mod ell_group, uniform over the slice's
// wavefront) as one more group with its unused loads repeating a valid slot; only real entries
// are summed.
template <class T, class V, class C, class F>
__device__ __forceinline__ T ell_sum(const C& ci, const gmem_t<const V>* __restrict__ val, unsigned lane, int w, F load) {
    constexpr int G = ell_group<T>();
    T s = T(0);
    int k = 0;
    for (; k + G <= w; k += G) {
        int c[G];
        T a[G];
        T x[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            c[g] = ci((k + g) * k_wave);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            a[g] = value_at<T, V>(val + (k + g) * k_wave, lane);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            x[g] = load(c[g]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            s = madd(a[g], x[g], s);
        }
    }
    const int rem = w - k;
    if (rem > 0) {
        int c[G - 1];
        T a[G - 1];
        T x[G - 1];
#pragma unroll
        for (int g = 0; g < G - 1; ++g) {
            c[g] = ci((g < rem ? k + g : k) * k_wave);
        }
#pragma unroll
        for (int g = 0; g < G - 1; ++g) {
            a[g] = value_at<T, V>(val + (g < rem ? k + g : k) * k_wave, lane);
        }
#pragma unroll
        for (int g = 0; g < G - 1; ++g) {
            x[g] = load(c[g]);
        }
        s = madd(a[0], x[0], s);
#pragma unroll
        for (int g = 1; g < G - 1; ++g) {
            if (g < rem) {
                s = madd(a[g], x[g], s);
            }
        }
    }
    return s;
}

// Sum over the CSR entries k, k + step, ... < end of one lane, in that order, four loads at a
// time (the lane's share of a row read by step lanes).
template <class T, class F>
__device__ __forceinline__ T csr_lane_sum(const gmem_t<const int>* __restrict__ col,
                                          const gmem_t<const T>* __restrict__ val, int k, int end, int step,
                                          F load) {
    T s = T(0);
    for (; k + 3 * step < end; k += 4 * step) {
        const int c0 = col[k];
        const int c1 = col[k + step];
        const int c2 = col[k + 2 * step];
        const int c3 = col[k + 3 * step];
        const T a0 = val[k];
        const T a1 = val[k + step];
        const T a2 = val[k + 2 * step];
        const T a3 = val[k + 3 * step];
        const T x0 = load(c0);
        const T x1 = load(c1);
        const T x2 = load(c2);
        const T x3 = load(c3);
        s = madd(a0, x0, s);
        s = madd(a1, x1, s);
        s = madd(a2, x2, s);
        s = madd(a3, x3, s);
    }
    if (k < end) {
        const bool has1 = k + step < end;
        const bool has2 = k + 2 * step < end;
        const int k1 = has1 ? k + step : k;
        const int k2 = has2 ? k + 2 * step : k;
        const int c0 = col[k];
        const int c1 = col[k1];
        const int c2 = col[k2];
        const T a0 = val[k];
        const T a1 = val[k1];
        const T a2 = val[k2];
        const T x0 = load(c0);
        const T x1 = load(c1);
        const T x2 = load(c2);
        s = madd(a0, x0, s);
        if (has1) {
            s = madd(a1, x1, s);
        }
        if (has2) {
            s = madd(a2, x2, s);
        }
    }
    return s;
}

constexpr int k_sym_group = 8; // entries whose loads are issued together

// What a row product multiplies a column with: (c) for any column; at(near, k, row) for column
// row + o[k] of a stencil, near = near<N>(o) being the arrays' addresses moved by the stencil's
// offsets (they stay in scalar registers; added to the row in the loop, they became a 64-bit vector
// address per load).
template <int N, class T>
struct Moved {
    const gmem_t<const T>* p[N];
    __device__ __forceinline__ Moved(const gmem_t<const T>* base, const int (&o)[N]) {
#pragma unroll
        for (int k = 0; k < N; ++k) {
            p[k] = base + o[k];
        }
    }
};

template <class T>
struct GatherX { // x_c
    const gmem_t<const T>* x;
    __device__ __forceinline__ T operator()(int c) const { return x[c]; }
    template <int N>
    struct Near {
        Moved<N, T> x;
    };
    template <int N>
    __device__ __forceinline__ Near<N> near(const int (&o)[N]) const {
        return {Moved<N, T>(x, o)};
    }
    template <int N>
    __device__ __forceinline__ T at(const Near<N>& a, int k, unsigned row) const {
        return load_at<T>(a.x.p[k], row);
    }
};

template <class T>
struct GatherX1 { // (f wd_c) b_c: the first Jacobi iterate from zero, formed on the fly
    const gmem_t<const T>* wd;
    const gmem_t<const T>* b;
    T f;
    __device__ __forceinline__ T operator()(int c) const { return (f * wd[c]) * b[c]; }
    template <int N>
    struct Near {
        Moved<N, T> wd;
        Moved<N, T> b;
    };
    template <int N>
    __device__ __forceinline__ Near<N> near(const int (&o)[N]) const {
        return {Moved<N, T>(wd, o), Moved<N, T>(b, o)};
    }
    template <int N>
    __device__ __forceinline__ T at(const Near<N>& a, int k, unsigned row) const {
        return (f * load_at<T>(a.wd.p[k], row)) * load_at<T>(a.b.p[k], row);
    }
};

template <class TZ>
struct GatherPz { // z_c + beta p_c: the new search direction
    const gmem_t<const TZ>* z;
    const gmem_t<const double>* p;
    double beta;
    __device__ __forceinline__ double operator()(int c) const { return static_cast<double>(z[c]) + beta * p[c]; }
    template <int N>
    struct Near {
        Moved<N, TZ> z;
        Moved<N, double> p;
    };
    template <int N>
    __device__ __forceinline__ Near<N> near(const int (&o)[N]) const {
        return {Moved<N, TZ>(z, o), Moved<N, double>(p, o)};
    }
    template <int N>
    __device__ __forceinline__ double at(const Near<N>& a, int k, unsigned row) const {
        return static_cast<double>(load_at<TZ>(a.z.p[k], row)) + beta * load_at<double>(a.p.p[k], row);
    }
};

struct GatherOne { // row sums of the matrix
    __device__ __forceinline__ double operator()(int) const { return 1.0; }
    template <int N>
    struct Near {};
    template <int N>
    __device__ __forceinline__ Near<N> near(const int (&)[N]) const {
        return {};
    }
    template <int N>
    __device__ __forceinline__ double at(const Near<N>&, int, unsigned) const {
        return 1.0;
    }
};

// Entry of offset o of a row in symmetric stencil storage (stored slot j of |o|) where the row may
// lie within the stencil's reach of the matrix's ends: the column is clamped to the matrix, as in
// the per-slice stencil layout (whose missing offsets hold zeros), and the value is zero where
// row + o < 0.
template <class T, class F>
__device__ __forceinline__ void sym_entry(const gmem_t<const T>* __restrict__ val, int pad, int last, int row, int o,
                                          int j, F load, T& a, T& x) {
    const int r = o < 0 ? row + o : row;
    const T v = load_at<T>(val + static_cast<long long>(j) * pad, static_cast<unsigned>(max(r, 0)));
    a = r < 0 ? T(0) : v;
    x = load(min(max(row + o, 0), last));
}

// A symmetric stencil of N offsets, in scalar registers for a whole kernel (read from the table
// inside a loop that stores, it came back by vector loads and a wait each time).
template <int N, class T>
struct SymStencil {
    int o[N];                      // offsets, ascending and symmetric
    const gmem_t<const T>* val[N]; // value of offset o[k] of row r at val[k][r]
    int reach;
    int last;
    __device__ __forceinline__ explicit SymStencil(const EllView& m) {
        const auto tab = gm(m.soff); // offsets [0, N), stored slots [N, 2 N)
        const long long pad = static_cast<long long>(m.n_slices) * k_wave;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            o[k] = __builtin_amdgcn_readfirstlane(tab[k]);
            const int j = __builtin_amdgcn_readfirstlane(tab[N + k]);
            val[k] = gm(static_cast<const T*>(m.val)) + (j * pad + min(o[k], 0));
        }
        reach = o[N - 1];
        last = m.n_rows - 1;
    }
};

// Row sums of Rows slices (s, s + ds) of a symmetric stencil: every entry's loads are issued before
// the sums, which run in offset order. Away from the matrix's ends an entry is one value load and
// the gather's loads, all from scalar bases with the lane's row as the only vector address; in the
// first and last few slices, within the stencil's reach of the ends, every entry has clamped
// addresses of its own. Rows past the end give the last row's sum.
template <int Rows, int N, class T, class F, class Near>
__device__ __forceinline__ void sym_rows_fixed(const SymStencil<N, T>& m, int s, int ds, int lane, const F& load,
                                               const Near& near, T (&y)[2]) {
    const int lo = s * k_wave;
    const int hi = (s + (Rows - 1) * ds) * k_wave + k_wave - 1;
    T a[Rows][N];
    T x[Rows][N];
    if (lo >= m.reach && hi + m.reach <= m.last) { // uniform over the wavefront
#pragma unroll
        for (int k = 0; k < N; ++k) {
#pragma unroll
            for (int h = 0; h < Rows; ++h) {
                const unsigned row = static_cast<unsigned>((s + h * ds) * k_wave + lane);
                a[h][k] = load_at<T>(m.val[k], row);
                x[h][k] = load.at(near, k, row);
            }
        }
        asm volatile("; stencil inside"); // keeps the compiler from merging the two branches' loads
    } else {
#pragma unroll
        for (int k = 0; k < N; ++k) {
#pragma unroll
            for (int h = 0; h < Rows; ++h) {
                // Both arrays are read at the row whose column row + o[k] is clamped to the matrix,
                // as in the per-slice stencil layout (whose missing offsets hold zeros). The value of
                // an offset past the end is the row's own slot, a stored zero.
                const int row = min((s + h * ds) * k_wave + lane, m.last);
                const int c = min(max(row + m.o[k], 0), m.last);
                const T v = load_at<T>(m.val[k], static_cast<unsigned>(m.o[k] < 0 ? c - m.o[k] : row));
                a[h][k] = row + m.o[k] < 0 ? T(0) : v;
                x[h][k] = load.at(near, k, static_cast<unsigned>(c - m.o[k]));
            }
        }
        asm volatile("; stencil at an end");
    }
#pragma unroll
    for (int h = 0; h < Rows; ++h) {
        T t = T(0);
#pragma unroll
        for (int k = 0; k < N; ++k) {
            t = madd(a[h][k], x[h][k], t);
        }
        asm volatile("" : "+v"(t)); // summed here: not moved, loads and all, under the row's store
        y[h] = t;
    }
}

// Any stencil size: the table read per entry, loads issued k_sym_group entries at a time.
template <int Rows, class T, class F>
__device__ __forceinline__ void sym_rows_any(const EllView& m, int s, int ds, int lane, F load, T (&y)[2]) {
    const int n = m.sym_n;
    const auto tab = gm(m.soff);
    const auto val = gm(static_cast<const T*>(m.val));
    const int pad = m.n_slices * k_wave;
    const int last = m.n_rows - 1;
    T t[Rows];
#pragma unroll
    for (int h = 0; h < Rows; ++h) {
        t[h] = T(0);
    }
    for (int k = 0; k < n; k += k_sym_group) {
        T a[Rows][k_sym_group];
        T x[Rows][k_sym_group];
#pragma unroll
        for (int g = 0; g < k_sym_group; ++g) {
            const int kk = min(k + g, n - 1); // past the stencil: repeats its last entry, not added
            const int o = tab[kk];
            const int j = tab[n + kk];
#pragma unroll
            for (int h = 0; h < Rows; ++h) {
                sym_entry<T>(val, pad, last, min((s + h * ds) * k_wave + lane, last), o, j, load, a[h][g], x[h][g]);
            }
        }
#pragma unroll
        for (int g = 0; g < k_sym_group; ++g) {
            if (k + g < n) {
#pragma unroll
                for (int h = 0; h < Rows; ++h) {
                    t[h] = madd(a[h][g], x[h][g], t[h]);
                }
            }
        }
    }
#pragma unroll
    for (int h = 0; h < Rows; ++h) {
        y[h] = t[h];
    }
}

// Row sums of slices s and (Rows == 2) s + ds in symmetric stencil storage (EllView::sym_w > 0),
// entries in offset order; their loads are issued together. Rows past the end give the sums of the
// last row.
template <int Rows, class T, class F>
__device__ __forceinline__ void sym_rows(const EllView& m, int s, int ds, int lane, F load, T (&y)[2]) {
    s = __builtin_amdgcn_readfirstlane(s); // one slice per wavefront
    switch (m.sym_n) { // uniform: the stencils of 3-D, 2-D and 1-D box meshes unrolled
    case 7: {
        const SymStencil<7, T> st(m);
        sym_rows_fixed<Rows>(st, s, ds, lane, load, load.near(st.o), y);
        return;
    }
    case 5: {
        const SymStencil<5, T> st(m);
        sym_rows_fixed<Rows>(st, s, ds, lane, load, load.near(st.o), y);
        return;
    }
    case 3: {
        const SymStencil<3, T> st(m);
        sym_rows_fixed<Rows>(st, s, ds, lane, load, load.near(st.o), y);
        return;
    }
    default:
        sym_rows_any<Rows, T>(m, s, ds, lane, load, y);
    }
}

// Row sum of an ELL row with the x entry of column c produced by load(c), in storage order.
// BF16 rows (fmt 1, FP32 kernels only) give diag_i x_i + rscale_i sum_k bf16_k x_ck.
template <class T, class F>
__device__ __forceinline__ T ell_row_f(const EllView& m, int slice, int lane, F load) {
    if (m.sym_w > 0) {
        T y[2];
        sym_rows<1, T>(m, slice, 0, lane, load, y);
        return y[0];
    }
    slice = __builtin_amdgcn_readfirstlane(slice); // one slice per wavefront: its streams have scalar bases
    const unsigned ul = static_cast<unsigned>(lane);
    const auto sp = gm(m.sp);
    const int base = __builtin_amdgcn_readfirstlane(sp[slice]);
    const int w = (__builtin_amdgcn_readfirstlane(sp[slice + 1]) - base) / k_wave;
    const int lg = __builtin_ctz(m.tpr); // lanes per row = 2^lg
    const int row = slice * (k_wave >> lg) + (lane >> lg);
    auto sum = [&](const auto& ci) -> T {
        if constexpr (sizeof(T) == 4) {
            if (m.fmt == 1) {
                const auto val = gm(static_cast<const unsigned short*>(m.val)) + base;
                const T s = ell_sum<T, unsigned short>(ci, val, ul, w, load);
                const T dx = row < m.n_rows ? gm(m.diag)[row] * load(row) : T(0);
                return madd(gm(m.rscale)[row], s, dx);
            }
        }
        return ell_sum<T, T>(ci, gm(static_cast<const T*>(m.val)) + base, ul, w, load);
    };
    if (m.soff != nullptr) {
        return sum(ColStencil{gm(m.soff) + base / k_wave, row, m.n_rows - 1});
    }
    if (m.cbase != nullptr) {
        return sum(ColBase{gm(reinterpret_cast<const unsigned short*>(m.dcol)) + base, ul, gm(m.cbase)[slice]});
    }
    if (m.dcol != nullptr) {
        return sum(ColOff{gm(m.dcol) + base, ul, row});
    }
    return sum(ColAbs{gm(m.col) + base, ul});
}

// Row sum of an ELL row: sum_k val_k * x[col_k] in storage order (any column / value format).
template <class T>
__device__ __forceinline__ T ell_row(const EllView& m, int slice, int lane, const T* __restrict__ x) {
    return ell_row_f<T>(m, slice, lane, GatherX<T>{gm(x)});
}

// Row sum with the first Jacobi iterate x1_j = wd_j * b_j formed on the fly (the reference's
// first sweep multiplies A by x = 0, so x1 = (w dinv) b exactly).
template <class T>
__device__ __forceinline__ T ell_row_x1(const EllView& m, int slice, int lane, const gmem_t<const T>* __restrict__ wd,
                                        const gmem_t<const T>* __restrict__ b, T f) {
    return ell_row_f<T>(m, slice, lane, GatherX1<T>{wd, b, f});
}

// Row sums of two slices with equal widths and one column format, their loads issued together
// (ell_group entries of each slice, then the sums in storage order per row): twice the loads in
// flight per wavefront, the same arithmetic as two ell_sum calls.
template <class T, class V, class C, class F>
__device__ __forceinline__ void ell_sum2(const C& ca, const C& cb, const gmem_t<const V>* __restrict__ va,
                                         const gmem_t<const V>* __restrict__ vb, unsigned lane, int w, F load, T& sa,
                                         T& sb) {
    constexpr int G = ell_group<T>();
    sa = T(0);
    sb = T(0);
    int k = 0;
    for (; k + G <= w; k += G) {
        int c0[G];
        int c1[G];
        T a0[G];
        T a1[G];
        T x0[G];
        T x1[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            c0[g] = ca((k + g) * k_wave);
            c1[g] = cb((k + g) * k_wave);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            a0[g] = value_at<T, V>(va + (k + g) * k_wave, lane);
            a1[g] = value_at<T, V>(vb + (k + g) * k_wave, lane);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            x0[g] = load(c0[g]);
            x1[g] = load(c1[g]);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            sa = madd(a0[g], x0[g], sa);
            sb = madd(a1[g], x1[g], sb);
        }
    }
    const int rem = w - k;
    if (rem > 0) {
        int c0[G - 1];
        int c1[G - 1];
        T a0[G - 1];
        T a1[G - 1];
        T x0[G - 1];
        T x1[G - 1];
#pragma unroll
        for (int g = 0; g < G - 1; ++g) {
            const int kk = g < rem ? k + g : k;
            c0[g] = ca(kk * k_wave);
            c1[g] = cb(kk * k_wave);
        }
#pragma unroll
        for (int g = 0; g < G - 1; ++g) {
            const int kk = g < rem ? k + g : k;
            a0[g] = value_at<T, V>(va + kk * k_wave, lane);
            a1[g] = value_at<T, V>(vb + kk * k_wave, lane);
        }
#pragma unroll
        for (int g = 0; g < G - 1; ++g) {
            x0[g] = load(c0[g]);
            x1[g] = load(c1[g]);
        }
        sa = madd(a0[0], x0[0], sa);
        sb = madd(a1[0], x1[0], sb);
#pragma unroll
        for (int g = 1; g < G - 1; ++g) {
            if (g < rem) {
                sa = madd(a0[g], x0[g], sa);
                sb = madd(a1[g], x1[g], sb);
            }
        }
    }
}

// The lane's share of its rows in slices s0 and s1 = s0 + ds of a sliced-ELL matrix (a slice past
// the end gives 0; with tpr > 1 the caller adds the row groups): equal to ell_row_f on each slice,
// bit for bit. Slices of different widths are summed one after the other. Stencil columns and
// BF16 rows occur with one lane per row only.
template <class T, class F>
__device__ __forceinline__ void ell_row_pair(const EllView& m, int s0, int ds, int lane, F load, T& ya, T& yb) {
    const int s1 = s0 + ds;
    ya = T(0);
    yb = T(0);
    if (s0 >= m.n_slices) {
        return;
    }
    if (s1 >= m.n_slices) {
        ya = ell_row_f<T>(m, s0, lane, load);
        return;
    }
    if (m.sym_w > 0) {
        T y[2];
        sym_rows<2, T>(m, s0, ds, lane, load, y);
        ya = y[0];
        yb = y[1];
        return;
    }
    s0 = __builtin_amdgcn_readfirstlane(s0);
    const unsigned ul = static_cast<unsigned>(lane);
    const auto sp = gm(m.sp);
    const int b0 = __builtin_amdgcn_readfirstlane(sp[s0]);
    const int b1 = __builtin_amdgcn_readfirstlane(sp[s0 + ds]);
    const int w = (__builtin_amdgcn_readfirstlane(sp[s0 + 1]) - b0) / k_wave;
    if (w != (__builtin_amdgcn_readfirstlane(sp[s0 + ds + 1]) - b1) / k_wave) {
        ya = ell_row_f<T>(m, s0, lane, load);
        yb = ell_row_f<T>(m, s1, lane, load);
        return;
    }
    const int lg = __builtin_ctz(m.tpr);
    const int r0 = s0 * (k_wave >> lg) + (lane >> lg);
    const int r1 = s1 * (k_wave >> lg) + (lane >> lg);
    auto pair = [&](const auto& c0, const auto& c1) {
        if constexpr (sizeof(T) == 4) {
            if (m.fmt == 1) {
                const auto val = gm(static_cast<const unsigned short*>(m.val));
                T sa;
                T sb;
                ell_sum2<T, unsigned short>(c0, c1, val + b0, val + b1, ul, w, load, sa, sb);
                const T dxa = r0 < m.n_rows ? gm(m.diag)[r0] * load(r0) : T(0);
                const T dxb = r1 < m.n_rows ? gm(m.diag)[r1] * load(r1) : T(0);
                ya = madd(gm(m.rscale)[r0], sa, dxa);
                yb = madd(gm(m.rscale)[r1], sb, dxb);
                return;
            }
        }
        const auto val = gm(static_cast<const T*>(m.val));
        ell_sum2<T, T>(c0, c1, val + b0, val + b1, ul, w, load, ya, yb);
    };
    if (m.soff != nullptr) {
        pair(ColStencil{gm(m.soff) + b0 / k_wave, r0, m.n_rows - 1}, ColStencil{gm(m.soff) + b1 / k_wave, r1, m.n_rows - 1});
    } else if (m.cbase != nullptr) {
        const auto dc = gm(reinterpret_cast<const unsigned short*>(m.dcol));
        pair(ColBase{dc + b0, ul, gm(m.cbase)[s0]}, ColBase{dc + b1, ul, gm(m.cbase)[s0 + ds]});
    } else if (m.dcol != nullptr) {
        pair(ColOff{gm(m.dcol) + b0, ul, r0}, ColOff{gm(m.dcol) + b1, ul, r1});
    } else {
        pair(ColAbs{gm(m.col) + b0, ul}, ColAbs{gm(m.col) + b1, ul});
    }
}

// Sum over groups of tpr consecutive lanes (tpr a power of two <= 64); every lane of the
// wavefront must take part.
template <class T>
__device__ __forceinline__ T group_sum(T v, int tpr) {
    for (int off = tpr >> 1; off > 0; off >>= 1) {
        v += __shfl_xor(v, off, k_wave);
    }
    return v;
}

// Row product of a matrix in either layout for the row / sub-lane of the calling thread; the
// result is complete in every lane of the row's group. Rows past the end give 0.
template <class T>
__device__ __forceinline__ T mat_row(const EllView& m, int row, int sub, const T* __restrict__ x) {
    if (m.csr == 0) {
        const int lg = __builtin_ctz(m.tpr);
        const int slice = row >> (6 - lg); // 64 / tpr rows per slice
        const T s = slice < m.n_slices ? ell_row<T>(m, slice, static_cast<int>(threadIdx.x) & (k_wave - 1), x)
                                       : T(0);
        return m.tpr > 1 ? group_sum(s, m.tpr) : s;
    }
    T s = T(0);
    if (row < m.n_rows) {
        const auto gx = gm(x);
        s = csr_lane_sum<T>(gm(m.col), gm(static_cast<const T*>(m.val)), m.sp[row] + sub, m.sp[row + 1],
                            m.tpr, [&](int c) { return gx[c]; });
    }
    return group_sum(s, m.tpr);
}

template <class T>
__device__ __forceinline__ T mat_row_x1(const EllView& m, int row, int sub, const gmem_t<const T>* __restrict__ wd,
                                        const gmem_t<const T>* __restrict__ b, T f) {
    if (m.csr == 0) {
        const int lg = __builtin_ctz(m.tpr);
        const int slice = row >> (6 - lg);
        const T s = slice < m.n_slices
                        ? ell_row_x1<T>(m, slice, static_cast<int>(threadIdx.x) & (k_wave - 1), wd, b, f)
                        : T(0);
        return m.tpr > 1 ? group_sum(s, m.tpr) : s;
    }
    T s = T(0);
    if (row < m.n_rows) {
        s = csr_lane_sum<T>(gm(m.col), gm(static_cast<const T*>(m.val)), m.sp[row] + sub, m.sp[row + 1],
                            m.tpr, [&](int c) { return (f * wd[c]) * b[c]; });
    }
    return group_sum(s, m.tpr);
}

// Workgroups are dispatched to the 8 XCDs round-robin (workgroup i runs on XCD i mod 8) and
// every XCD has its own L2. This bijection hands each XCD a contiguous range of logical blocks,
// so rows that share neighbours (and their x entries) meet in the same L2.
__device__ __forceinline__ int xcd_block() {
    const int g = static_cast<int>(gridDim.x);
    const int b = static_cast<int>(blockIdx.x);
    const int q = g / k_xcds;
    const int r = g % k_xcds;
    const int xcd = b % k_xcds;
    const int k = b / k_xcds;
    return xcd < r ? xcd * (q + 1) + k : r * (q + 1) + (xcd - r) * q + k;
}

// The launch table's (system, block) entry of this workgroup, read as one 8-byte load: both
// halves arrive with one wait (the block half is otherwise fetched again after the status test).
__device__ __forceinline__ int2 block_entry(const int2* __restrict__ blocks) {
    const auto e = gm(reinterpret_cast<const unsigned long long*>(blocks))[xcd_block()];
    return make_int2(static_cast<int>(static_cast<unsigned>(e)), static_cast<int>(static_cast<unsigned>(e >> 32)));
}

// Forms of the level-0 operator that a kernel is built for. L0_ANY: the library's layouts, told
// apart at run time. L0_SYM7: symmetric stencil storage of 7 offsets (every 3-D box's pressure
// matrix), for launches whose systems all have it: the kernel holds that one path, in fewer
// registers. L0_CSR: a caller's CSR arrays read in place (a64.sp = row offsets, a64.col, a64.val;
// one lane per row, entries in CSR order), which gives the same sums: the sliced-ELL padding and
// stencil gaps add exact zeros after or between the same products in the same order.
enum L0Form : int { L0_ANY = 0, L0_SYM7 = 1, L0_CSR = 2 };

// The level-0 operator and what it is multiplied with, as a kernel of that form keeps them.
template <int Form, class T, class F>
struct L0Op {
    EllView m;
    F load;
    __device__ __forceinline__ L0Op(const EllView& v, const F& f) : m(v), load(f) {}
};

template <class T, class F>
struct L0Op<L0_SYM7, T, F> {
    SymStencil<7, T> m;
    F load;
    typename F::template Near<7> near;
    __device__ __forceinline__ L0Op(const EllView& v, const F& f) : m(v), load(f), near(f.near(m.o)) {}
};

// Row sums of the lane's rows of slices s and (Rows == 2) s + ds, their loads issued together. Rows
// past the end give some row's sum, or 0.
template <int Rows, int Form, class T, class F>
__device__ __forceinline__ void l0_rows(const L0Op<Form, T, F>& op, int s, int ds, int lane, T (&y)[2]) {
    const auto& m = op.m;
    if constexpr (Form == L0_CSR) {
        const auto sp = gm(m.sp);
#pragma unroll
        for (int h = 0; h < Rows; ++h) {
            const int row = (s + h * ds) * k_wave + lane;
            y[h] = row < m.n_rows ? csr_lane_sum<double>(gm(m.col), gm(static_cast<const double*>(m.val)), sp[row],
                                                         sp[row + 1], 1, op.load)
                                  : 0.0;
        }
    } else if constexpr (Form == L0_SYM7) {
        sym_rows_fixed<Rows>(m, __builtin_amdgcn_readfirstlane(s), ds, lane, op.load, op.near, y);
    } else if constexpr (Rows == 2) {
        ell_row_pair<T>(m, s, ds, lane, op.load, y[0], y[1]);
    } else {
        y[0] = s < m.n_slices ? ell_row_f<T>(m, s, lane, op.load) : T(0);
    }
}

#define CFDG_BLOCK_PROLOGUE(sysarr, blocks)                                                     \
    const int2 bk_ = block_entry(blocks);                                                         \
    const SysDev& S = (sysarr)[bk_.x];                                                            \
    const int wave_ = threadIdx.x / k_wave;                                                       \
    const int lane = threadIdx.x % k_wave;                                                        \
    const int slice = bk_.y * k_slices_per_block + wave_;                                         \
    const int row = slice * k_wave + lane;                                                        \
    (void)row;

// ------------------------------------------------------------------------------------------
// Scalar steps of the Krylov recurrences
// ------------------------------------------------------------------------------------------

// Steps between two kernels of an iteration. Each needs the sum of one or two partials of the
// kernel before it. The kernel after it makes the step itself: every workgroup adds the at most
// k_max_groups partials (a few kilobytes, L2-resident) in the same order and computes the same
// scalars, and the system's first workgroup stores the new state. A launch of its own for the step
// cost 4.6 to 8.9 us an iteration at 128^3 and 2.3 us in the smallest systems; in the kernel's
// prologue it costs about 0.7 us. The state is kept in k_states copies, so that no workgroup reads
// the copy that the first one writes: step Op reads copy state_in and writes state_out, and the
// state goes round them once an iteration.
enum FinOp : int {
    FIN_RES = 0,          // AMG-PCG: |r|; converged?
    FIN_BETA = 1,         // rz_new; beta = rz_new / rz (0 first); it++ / limit
    FIN_BETA_FLEX = 2,    // rz_new, zq; beta = -zq / pq (0 first); it++ / limit
    FIN_ALPHA = 3,        // pq; breakdown if 0; alpha = rz / pq
    FIN_CG_RES_BETA = 4,  // Jacobi CG: residual test, then beta (0 first)
    FIN_BICG_RES = 5,     // residual test, then rho and beta
    FIN_BICG_ALPHA = 6,
    FIN_BICG_S = 7,       // |s|: early exit?
    FIN_BICG_OMEGA = 8,
    FIN_TRUE = 9          // true residual (after the solve, copy 0 in place)
};

// Copies: AMG-PCG and Jacobi CG 2 -> (residual step) -> 0 -> (beta) -> 1 -> (alpha) -> 2, Jacobi CG
// taking residual and beta in one step 2 -> 1 and reporting through copy 0; BiCGStab 3 ->
// (residual, rho) -> 0 -> (alpha) -> 1 -> (s) -> 2 -> (omega) -> 3. Copy 0 is the solve's public state.
__host__ __device__ constexpr int state_in(int op) {
    return op == FIN_BETA || op == FIN_BETA_FLEX || op == FIN_BICG_ALPHA || op == FIN_TRUE ? 0
           : op == FIN_ALPHA || op == FIN_BICG_S                                           ? 1
           : op == FIN_BICG_RES                                                            ? 3
                                                                                           : 2;
}

__host__ __device__ constexpr int state_out(int op) {
    return op == FIN_BETA || op == FIN_BETA_FLEX || op == FIN_BICG_ALPHA || op == FIN_CG_RES_BETA ? 1
           : op == FIN_ALPHA || op == FIN_BICG_S                                                  ? 2
           : op == FIN_BICG_OMEGA                                                                 ? 3
                                                                                                  : 0;
}

template <int Op>
__host__ __device__ constexpr int step_slots() { // partials a step adds
    return Op == FIN_BETA_FLEX || Op == FIN_CG_RES_BETA || Op == FIN_BICG_RES || Op == FIN_BICG_OMEGA ? 2 : 1;
}

template <int Op>
__host__ __device__ constexpr int step_slot(int q) {
    switch (Op) {
    case FIN_RES: return SLOT_RR;
    case FIN_BETA: return SLOT_RZ;
    case FIN_BETA_FLEX: return q == 0 ? SLOT_RZ : SLOT_ZQ;
    case FIN_ALPHA: return SLOT_PQ;
    case FIN_CG_RES_BETA: return q == 0 ? SLOT_RR : SLOT_RZ;
    case FIN_BICG_RES: return q == 0 ? SLOT_RR : SLOT_R0R;
    case FIN_BICG_ALPHA: return SLOT_R0V;
    case FIN_BICG_S: return SLOT_SS;
    case FIN_BICG_OMEGA: return q == 0 ? SLOT_TT : SLOT_TS;
    default: return SLOT_TRUE;
    }
}

// Sums of the system's partials in slots slot(0) .. slot(N - 1), complete in every thread of a
// k_block workgroup: thread t adds entries t, t + 256, ..., then the wavefront butterfly and the
// four wavefronts in order. Every workgroup gets the same bits.
template <int N, class Slot>
__device__ __forceinline__ void reduce_slots(const SysDev& S, Slot slot, double (&out)[N]) {
    __shared__ double red[N][k_slices_per_block];
    const int n = S.n_groups;
    double v[N][k_max_groups / k_block];
#pragma unroll
    for (int q = 0; q < N; ++q) {
        const auto p = gm(static_cast<const double*>(S.partials)) + slot(q) * n;
#pragma unroll
        for (int k = 0; k < k_max_groups / k_block; ++k) { // every load before the first sum
            const int i = static_cast<int>(threadIdx.x) + k * k_block;
            v[q][k] = i < n ? p[i] : 0.0;
        }
    }
#pragma unroll
    for (int q = 0; q < N; ++q) {
        double s = v[q][0];
#pragma unroll
        for (int k = 1; k < k_max_groups / k_block; ++k) {
            s += v[q][k];
        }
        s = wave_sum(s);
        if (threadIdx.x % k_wave == 0) {
            red[q][threadIdx.x / k_wave] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; ++q) {
        double t = red[q][0];
#pragma unroll
        for (int w = 1; w < k_slices_per_block; ++w) {
            t += red[q][w];
        }
        out[q] = t;
    }
}

// A state in registers, loaded and stored field by field: copied as a SolveState, the compiler
// keeps it in scratch memory (16 us a kernel).
struct Scalars {
    double tol, rz, pq, alpha, beta, res, bnorm, rho, omega;
    int it, max_it, status;
};

__device__ __forceinline__ Scalars load_state(const SolveState* p) {
    const auto g = gm(p);
    Scalars s;
    s.tol = g->tol;
    s.rz = g->rz;
    s.pq = g->pq;
    s.alpha = g->alpha;
    s.beta = g->beta;
    s.res = g->res;
    s.bnorm = g->bnorm;
    s.rho = g->rho;
    s.omega = g->omega;
    s.it = g->it;
    s.max_it = g->max_it;
    s.status = g->status;
    return s;
}

__device__ __forceinline__ void store_state(SolveState* p, const Scalars& s) {
    const auto g = gm(p);
    g->tol = s.tol;
    g->rz = s.rz;
    g->pq = s.pq;
    g->alpha = s.alpha;
    g->beta = s.beta;
    g->res = s.res;
    g->bnorm = s.bnorm;
    g->rho = s.rho;
    g->omega = s.omega;
    g->it = s.it;
    g->max_it = s.max_it;
    g->status = s.status;
}

// The arithmetic of a step (krylov_kernels.inc:44-169, 240-301) on the sums v0, v1. A system that
// ended keeps its state; an early exit of BiCGStab is complete after its x update.
template <int Op>
__device__ __forceinline__ void state_step(Scalars& st, double v0, double v1) {
    if (Op == FIN_BICG_OMEGA && st.status == ST_CONVERGED_PENDING) {
        st.status = ST_CONVERGED;
    } else if (st.status == ST_RUNNING) {
        if (Op == FIN_RES || Op == FIN_CG_RES_BETA || Op == FIN_BICG_RES) {
            st.res = sqrt(v0);
            st.status = st.res <= st.tol ? ST_CONVERGED : ST_RUNNING;
        }
        if (Op == FIN_BETA || Op == FIN_BETA_FLEX || (Op == FIN_CG_RES_BETA && st.status == ST_RUNNING)) {
            const double rz_new = Op == FIN_CG_RES_BETA ? v1 : v0;
            const double ratio = Op == FIN_BETA_FLEX ? -v1 / st.pq : rz_new / st.rz;
            st.beta = st.it == 0 ? 0.0 : ratio;
            st.rz = rz_new;
            st.it += 1;
            st.status = st.it > st.max_it ? ST_MAXIT : ST_RUNNING;
        }
        if (Op == FIN_ALPHA) {
            st.pq = v0;
            if (v0 == 0.0) {
                st.status = ST_BREAKDOWN;
            } else {
                st.alpha = st.rz / v0;
            }
        }
        if (Op == FIN_BICG_RES && st.status == ST_RUNNING) {
            // rho_new = r0.r, the limit, the guards rho_new == 0 and omega == 0, beta
            st.it += 1;
            if (st.it > st.max_it) {
                st.status = ST_MAXIT;
            } else if (v1 == 0.0 || st.omega == 0.0) {
                st.status = ST_BREAKDOWN;
            } else {
                st.beta = (v1 / st.rho) * (st.alpha / st.omega);
                st.rho = v1;
            }
        }
        if (Op == FIN_BICG_ALPHA) {
            if (v0 == 0.0) {
                st.status = ST_BREAKDOWN;
            } else {
                st.alpha = st.rho / v0;
            }
        }
        if (Op == FIN_BICG_S) {
            const double s_norm = sqrt(v0);
            if (s_norm <= st.tol) {
                st.res = s_norm;
                st.status = ST_CONVERGED_PENDING;
            }
        }
        if (Op == FIN_BICG_OMEGA) {
            st.omega = v0 > 0.0 ? v1 / v0 : 0.0;
        }
    }
}

// A system's progress as one 64-bit word, so that a host that polls it never sees half a report:
// the residual (FP32 bits) above, the number of finished iterations and the status below. The word
// goes to host-mapped memory at every residual step; the host reads it while later iterations are
// queued, without an event (an event record between two graph launches costs 4 us).
__device__ __forceinline__ unsigned long long report_word(const Scalars& st, int done) {
    const unsigned low = (static_cast<unsigned>(done) << k_report_status_bits) | static_cast<unsigned>(st.status);
    return (static_cast<unsigned long long>(__float_as_uint(static_cast<float>(st.res))) << 32) | low;
}

// Iterations finished when residual step Op has run (Jacobi CG and BiCGStab count the next one
// in the step when the solve goes on).
template <int Op>
__device__ __forceinline__ int iterations_done(const Scalars& st) {
    return Op != FIN_RES && (st.status == ST_RUNNING || st.status == ST_BREAKDOWN) ? st.it - 1 : st.it;
}

template <int Op>
__device__ __forceinline__ void store_report(const Scalars& st, unsigned long long* report, int id) {
    if (report != nullptr) {
        __hip_atomic_store(report + id, report_word(st, iterations_done<Op>(st)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// Step Op in the prologue of a k_block kernel: the state after it in every thread, stored (and
// reported, report may be null) by the system's first workgroup. Workgroups of a system that ended
// skip the sums.
template <int Op>
__device__ __forceinline__ Scalars take_step(const SysDev& S, bool first, unsigned long long* report, int id) {
    Scalars st = load_state(S.st + state_in(Op));
    double v0 = 0.0;
    double v1 = 0.0;
    if (st.status == ST_RUNNING) { // uniform over the workgroup
        double o[step_slots<Op>()];
        reduce_slots<step_slots<Op>()>(S, [](int q) { return step_slot<Op>(q); }, o);
        v0 = o[0];
        v1 = o[step_slots<Op>() - 1];
    }
    state_step<Op>(st, v0, v1);
    if (first && threadIdx.x == 0) {
        store_state(S.st + state_out(Op), st);
        store_report<Op>(st, report, id);
    }
    return st;
}

// Residual step Op (its result in the public copy 0), or the true residual, as a launch of its
// own, one workgroup per system (ids: descriptor indices): at the end of a graph, where no kernel
// of the next iteration makes the step yet, and in cycles whose first kernel cannot make it. The
// step is the same one, bit for bit, so making it twice changes nothing.
template <int Op>
__global__ void __launch_bounds__(k_block) k_step(const SysDev* __restrict__ sys, const int* __restrict__ ids,
                                                  unsigned long long* __restrict__ report) {
    const int id = ids[blockIdx.x];
    const SysDev& S = sys[id];
    if (Op == FIN_TRUE) {
        double t[1];
        reduce_slots<1>(S, [](int) { return static_cast<int>(SLOT_TRUE); }, t);
        if (threadIdx.x == 0) {
            S.st[0].true_res = sqrt(t[0]);
        }
        return;
    }
    Scalars st = load_state(S.st + state_in(Op));
    double o[step_slots<Op>()];
    reduce_slots<step_slots<Op>()>(S, [](int q) { return step_slot<Op>(q); }, o);
    if (threadIdx.x == 0) {
        state_step<Op>(st, o[0], o[step_slots<Op>() - 1]);
        store_state(S.st, st);
        store_report<Op>(st, report, id);
    }
}

// The start of a solve after its initial residual: |b| and BiCGStab's rho = alpha = omega = 1 into
// the state that residual step Op reads, then that step.
template <int Op>
__global__ void __launch_bounds__(k_block) k_start(const SysDev* __restrict__ sys, const int* __restrict__ ids,
                                                   unsigned long long* __restrict__ report) {
    const int id = ids[blockIdx.x];
    const SysDev& S = sys[id];
    constexpr int n = step_slots<Op>() + 1;
    double o[n];
    reduce_slots<n>(S, [](int q) { return q + 1 == n ? static_cast<int>(SLOT_BB) : step_slot<Op>(q); }, o);
    if (threadIdx.x == 0) {
        Scalars st = load_state(S.st + state_in(Op));
        st.bnorm = sqrt(o[n - 1]);
        st.rho = 1.0;
        st.alpha = 1.0;
        st.omega = 1.0;
        store_state(S.st + state_in(Op), st);
        state_step<Op>(st, o[0], o[n - 2]);
        store_state(S.st, st);
        store_report<Op>(st, report, id);
    }
}

// ------------------------------------------------------------------------------------------
// Level-0 kernels: groups of rows
// ------------------------------------------------------------------------------------------

// A level-0 kernel's workgroup serves the row groups [bk_.y, bk_.y + gpb) of its system, one after
// the other. A group is S.chunks chunks of 256 rows and has one partial sum per dot product, so
// that a step adds at most k_max_groups partials whatever the system's size (one chunk up to
// 262,144 rows, 8 at 128^3); the grouping depends on the system's size only, so its sums do not
// depend on which systems share the launch. gpb > 1 in large batches keeps the number of
// workgroups, each of which makes the step, near 16384.
//
// A group's chunks are not neighbours: the groups fall into k_xcds segments (one XCD's workgroups of
// a single system), a segment owns a contiguous range of chunks, and its groups take the chunks of
// the range in turn. The workgroups of an XCD thus move through the rows as one window, as if every
// chunk were a workgroup of its own. With a group's chunks side by side the workgroups read at a
// distance of 2048 rows from each other, which keeps a few memory channels busy and the others idle:
// 41.7 against 39.0 us for the outer product at 128^3 (two chunks of its rows at a time).
#define CFDG_L0_PROLOGUE(sysarr, blocks)                                                          \
    const int2 bk_ = block_entry(blocks);                                                         \
    const SysDev& S = (sysarr)[bk_.x];                                                            \
    const int wave_ = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / k_wave);     \
    const int lane = static_cast<int>(threadIdx.x) % k_wave;                                      \
    const bool first_ = bk_.y == 0;                                                               \
    (void)first_;                                                                                 \
    (void)lane;

// The chunks of a workgroup's groups in the order in which its wavefronts serve them: a group at a time,
// or, where groups are single chunks and the kernel takes two chunks at a time (Pair: two rows' loads in
// flight in each lane), two groups at a time. slice: the wavefront's in the first chunk, ds slices before
// the next one's.
struct Chunks {
    int groups; // served together, 1 or 2
    int count;
    int slice;
    int ds;
};

template <bool Pair>
__device__ __forceinline__ Chunks chunks_of(const SysDev& S, int g, int end, int wave) {
    const int chunks = S.chunks;
    if (Pair && chunks == 1 && g + 1 < end) {
        return {2, 2, g * k_slices_per_block + wave, k_slices_per_block};
    }
    const int seg = S.segment;
    const int s = g / seg;
    const int ds = min(seg, S.n_groups - s * seg) * k_slices_per_block; // a group's chunks are this far apart
    return {1, chunks, (s * seg * chunks + (g - s * seg)) * k_slices_per_block + wave, ds};
}

// How a level-0 kernel names a lane's row. Symmetric storage has fewer than 2^29 rows (System builds
// it for no more), so that its row number alone is the offset that a row's own loads and its stencil's
// share; the other forms take systems of any size.
template <int Form>
using RowOf = std::conditional_t<Form == L0_SYM7, unsigned, LaneRow>;

__host__ __device__ __forceinline__ void set_row(unsigned& r, int slice, int lane, int) {
    r = static_cast<unsigned>(slice) * k_wave + static_cast<unsigned>(lane);
}
__host__ __device__ __forceinline__ void set_row(LaneRow& r, int slice, int lane, int n) {
    r.start = static_cast<long long>(slice) * k_wave;
    r.lane = static_cast<unsigned>(lane);
    r.left = static_cast<int>(n - r.start);
}
__host__ __device__ __forceinline__ bool inside(unsigned r, int n) { return r < static_cast<unsigned>(n); }
__host__ __device__ __forceinline__ bool inside(const LaneRow& r, int) { return static_cast<int>(r.lane) < r.left; }

// The row, or some row of the matrix for one past its end.
__host__ __device__ __forceinline__ unsigned in_matrix(unsigned r, int n) {
    const unsigned last = static_cast<unsigned>(n) - 1;
    return r < last ? r : last;
}
__host__ __device__ __forceinline__ LaneRow in_matrix(const LaneRow& r, int) {
    LaneRow c = r;
    c.start = r.left > 0 ? r.start : 0;
    c.lane = static_cast<int>(r.lane) < r.left ? r.lane : 0;
    return c;
}

// The lane's rows of slices slice and (Rows == 2) slice + ds; load(h, r) requests what a row's result
// needs of its own entries, before the row sums' loads (rows past the end: of some other row).
template <int Rows, class Row, class F>
__host__ __device__ __forceinline__ void own_rows(int slice, int ds, int lane, int n, Row (&row)[2], F load) {
#pragma unroll
    for (int h = 0; h < Rows; ++h) {
        set_row(row[h], slice + h * ds, lane, n);
        load(h, in_matrix(row[h], n));
    }
}

// Runs rows(H, slice, ds, t) over the workgroup's groups: slice and, where the constant H is 2, slice +
// ds; rows past the end are included. The rows' terms t[h][q] are added, first row first, and the sums of
// each group go to partials slots slot(0) .. slot(N - 1). The wavefronts meet once, after the last group:
// with two barriers a group and single chunks one at a time a batch of 256 systems at 14 groups a
// workgroup took 43.7 ms in mixed and 48.5 in BF16, so 43.5 and 47.4.
template <int N, bool Pair, class R, class Slot>
__device__ __forceinline__ void for_groups(const SysDev& S, int first, int gpb, int wave, R rows, Slot slot) {
    __shared__ double red[k_max_gpb][N][k_slices_per_block];
    const int n = S.n_groups;
    const int end = min(first + gpb, n);
    for (int g = first; g < end;) {
        const Chunks ch = chunks_of<Pair>(S, g, end, wave);
        double v[2][N] = {};
        int slice = ch.slice;
        int c = 0;
        if constexpr (Pair) {
            for (; c + 1 < ch.count; c += 2, slice += 2 * ch.ds) {
                double t[2][N] = {};
                rows(std::integral_constant<int, 2>{}, slice, ch.ds, t);
#pragma unroll
                for (int q = 0; q < N; ++q) {
                    v[0][q] += t[0][q];
                    if (ch.groups == 2) {
                        v[1][q] += t[1][q];
                    } else {
                        v[0][q] += t[1][q];
                    }
                }
            }
        }
        for (; c < ch.count; ++c, slice += ch.ds) {
            double t[2][N] = {};
            rows(std::integral_constant<int, 1>{}, slice, ch.ds, t);
#pragma unroll
            for (int q = 0; q < N; ++q) {
                v[0][q] += t[0][q];
            }
        }
#pragma unroll
        for (int h = 0; h < (Pair ? 2 : 1); ++h) {
            if (h < ch.groups) {
#pragma unroll
                for (int q = 0; q < N; ++q) {
                    const double w = wave_sum(v[h][q]);
                    if (threadIdx.x % k_wave == 0) {
                        red[g + h - first][q][wave] = w;
                    }
                }
            }
        }
        g += ch.groups;
    }
    __syncthreads();
    const int i = static_cast<int>(threadIdx.x) / N; // group and slot of this thread
    const int q = static_cast<int>(threadIdx.x) % N;
    if (i < end - first) {
        double s = red[i][q][0];
#pragma unroll
        for (int w = 1; w < k_slices_per_block; ++w) {
            s += red[i][q][w];
        }
        S.partials[slot(q) * n + first + i] = s;
    }
}

// The same without dot products: rows(H, slice, ds).
template <bool Pair, class R>
__device__ __forceinline__ void for_group_rows(const SysDev& S, int first, int gpb, int wave, R rows) {
    const int end = min(first + gpb, S.n_groups);
    for (int g = first; g < end;) {
        const Chunks ch = chunks_of<Pair>(S, g, end, wave);
        int slice = ch.slice;
        int c = 0;
        if constexpr (Pair) {
            for (; c + 1 < ch.count; c += 2, slice += 2 * ch.ds) {
                rows(std::integral_constant<int, 2>{}, slice, ch.ds);
            }
        }
        for (; c < ch.count; ++c, slice += ch.ds) {
            rows(std::integral_constant<int, 1>{}, slice, ch.ds);
        }
        g += ch.groups;
    }
}

// ------------------------------------------------------------------------------------------
// Outer Krylov kernels (level 0, FP64)
// ------------------------------------------------------------------------------------------

// r = b - A x, partials r.r and b.b; p = q = 0. For mixed precision also r32 = (float) r.
template <bool Mixed, int Form>
__global__ void __launch_bounds__(k_block) k_residual0(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const L0Op<Form, double, GatherX<double>> A0(S.a64, {gm(static_cast<const double*>(S.x))});
    for_groups<2, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][2]) {
        const int row = slice * k_wave + lane;
        double y[2];
        l0_rows<1>(A0, slice, 0, lane, y);
        if (row < S.n) {
            const double bi = gm(S.b)[row];
            const double ri = bi - y[0];
            gm(S.r)[row] = ri;
            gm(S.p)[row] = 0.0;
            gm(S.q)[row] = 0.0;
            if (Mixed) {
                gm(S.r32)[row] = static_cast<float>(ri);
            }
            v[0][0] = ri * ri;
            v[0][1] = bi * bi;
        }
    }, [](int q) { return q == 0 ? SLOT_RR : SLOT_BB; });
}

// Jacobi CG start: r = b - A x, z = dinv r, p = 0; partials r.r, r.z, b.b.
template <int Form>
__global__ void __launch_bounds__(k_block) k_cg_init(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const L0Op<Form, double, GatherX<double>> A0(S.a64, {gm(static_cast<const double*>(S.x))});
    for_groups<3, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][3]) {
        const int row = slice * k_wave + lane;
        double y[2];
        l0_rows<1>(A0, slice, 0, lane, y);
        if (row < S.n) {
            const double bi = gm(S.b)[row];
            const double ri = bi - y[0];
            const double zi = ri * gm(S.dinv)[row];
            gm(S.r)[row] = ri;
            gm(S.z)[row] = zi;
            gm(S.p)[row] = 0.0;
            v[0][0] = ri * ri;
            v[0][1] = ri * zi;
            v[0][2] = bi * bi;
        }
    }, [](int q) { return q == 0 ? SLOT_RR : q == 1 ? SLOT_RZ : SLOT_BB; });
}

// Search directions alternate between two buffers: iteration k reads p_old = parity ? p : p2
// and writes p_new = parity ? p2 : p (parity = k mod 2, iterations counted from 1).
__device__ __forceinline__ double* p_old_of(const SysDev& S, int parity) { return (parity ^ S.flip) ? S.p : S.p2; }
__device__ __forceinline__ double* p_new_of(const SysDev& S, int parity) { return (parity ^ S.flip) ? S.p2 : S.p; }

// Step Op (beta), then q = A p_new with p_new = z + beta p_old formed per gathered column (the
// reference's separate p update, krylov_kernels.inc:293-296, folded into the next product;
// identical arithmetic), p_new written for the own rows, and the partial p_new.q. z is the level-0
// V-cycle output v[z_buf] (which = 1, FP64 or FP32) or the Jacobi-preconditioned residual S.z
// (which = 0).
// At 128^3 (170 MB from memory in the mixed solve, whose matrix has left the Infinity Cache since the
// last product) one chunk at a time takes 37.2 us and two 40.8: three arrays of loads a row fill the
// wavefront's queue already. Before, with the step as a launch of its own: 36.4 + 8.9 us and 130 MB:
// the groups of an XCD drift apart, and the plane below has left its L2 when it is read again (24
// bytes a row). Non-temporal stores of p and q don't bring it back (a mixed solve 3.21 -> 3.24 ms, FP64 6.33
// -> 6.40 ms).
template <class TZ, int Form, int Op>
__global__ void __launch_bounds__(k_block) k_spmv_pz(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb, int parity,
                          int which, int z_buf, unsigned long long* __restrict__ report) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto z = gm(which == 0 ? reinterpret_cast<const TZ*>(S.z) : static_cast<const TZ*>(S.lv[0].v[z_buf]));
    const auto po = gm(static_cast<const double*>(p_old_of(S, parity)));
    const auto pn = gm(p_new_of(S, parity));
    const auto qv = gm(S.q);
    const int n = S.n;
    L0Op<Form, double, GatherPz<TZ>> A0(S.a64, {z, po, 0.0});
    const Scalars st = take_step<Op>(S, first_, report, bk_.x);
    if (st.status != ST_RUNNING) {
        return;
    }
    A0.load.beta = st.beta;
    for_groups<1, false>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds, double (&v)[2][1]) {
        double y[2];
        double pi[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& r) { pi[h] = static_cast<double>(load_at<TZ>(z, r)) + st.beta * load_at<double>(po, r); });
        l0_rows<H.value>(A0, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                store_at<double>(pn, row[h], pi[h]);
                store_at<double>(qv, row[h], y[h]);
                v[h][0] = pi[h] * y[h];
            }
        }
    }, [](int) { return SLOT_PQ; });
}

// x = 0 for every system of a launch table (one launch for a whole batch).
__global__ void __launch_bounds__(k_block) k_zero_x(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    for_group_rows<false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int) {
        const int row = slice * k_wave + lane;
        if (row < S.n) {
            gm(S.x)[row] = 0.0;
        }
    });
}

// Step FIN_ALPHA, then x += alpha p; r -= alpha q; partial r.r. Jacobi CG also forms z = dinv r and
// r.z; the mixed solver writes r32 = (float) r for the FP32 V-cycle.
template <int Mode> // 0 AMG FP64, 1 Jacobi CG, 2 mixed AMG
__global__ void __launch_bounds__(k_block) k_update_xr(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb, int parity) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto x = gm(S.x);
    const auto r = gm(S.r);
    const auto p = gm(static_cast<const double*>(p_new_of(S, parity)));
    const auto qv = gm(static_cast<const double*>(S.q));
    const auto z = gm(S.z);
    const auto dinv = gm(S.dinv);
    const auto r32 = gm(S.r32);
    const int n = S.n;
    const Scalars st = take_step<FIN_ALPHA>(S, first_, nullptr, 0);
    if (st.status != ST_RUNNING) {
        return;
    }
    const double alpha = st.alpha;
    constexpr int n_dots = Mode == 1 ? 2 : 1;
    for_groups<n_dots, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][n_dots]) {
        const int row = slice * k_wave + lane;
        if (row < n) {
            x[row] = x[row] + alpha * p[row];
            const double ri = r[row] - alpha * qv[row];
            r[row] = ri;
            v[0][0] = ri * ri;
            if constexpr (Mode == 1) {
                const double zi = ri * dinv[row];
                z[row] = zi;
                v[0][1] = ri * zi;
            }
            if (Mode == 2) {
                r32[row] = static_cast<float>(ri);
            }
        }
    }, [](int q) { return q == 0 ? SLOT_RR : SLOT_RZ; });
}

// True residual |b - A x|^2 partials (always runs, after the solve).
template <int Form>
__global__ void __launch_bounds__(k_block) k_true_residual(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto b = gm(S.b);
    const L0Op<Form, double, GatherX<double>> A0(S.a64, {gm(static_cast<const double*>(S.x))});
    const int n = S.n;
    for_groups<1, true>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds, double (&v)[2][1]) {
        double y[2];
        double bi[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& r) { bi[h] = load_at<double>(b, r); });
        l0_rows<H.value>(A0, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                const double ri = bi[h] - y[h];
                v[h][0] = ri * ri;
            }
        }
    }, [](int) { return SLOT_TRUE; });
}

// ------------------------------------------------------------------------------------------
// BiCGStab kernels (krylov_kernels.inc:96-169): five launches an iteration
// ------------------------------------------------------------------------------------------

// r = b - A x; r0 = r; p = v = 0; partials r.r, b.b and r0.r.
template <int Form>
__global__ void __launch_bounds__(k_block) k_bicg_init(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const L0Op<Form, double, GatherX<double>> A0(S.a64, {gm(static_cast<const double*>(S.x))});
    for_groups<3, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][3]) {
        const int row = slice * k_wave + lane;
        double y[2];
        l0_rows<1>(A0, slice, 0, lane, y);
        if (row < S.n) {
            const double bi = gm(S.b)[row];
            const double ri = bi - y[0];
            gm(S.r)[row] = ri;
            gm(S.r0)[row] = ri;
            gm(S.p)[row] = 0.0;
            gm(S.v)[row] = 0.0;
            v[0][0] = ri * ri;
            v[0][1] = ri * ri;
            v[0][2] = bi * bi;
        }
    }, [](int q) { return q == 0 ? SLOT_RR : q == 1 ? SLOT_R0R : SLOT_BB; });
}

// Step FIN_BICG_RES (residual test, rho, beta), then p = r + beta (p - omega v); ph = dinv p.
__global__ void __launch_bounds__(k_block) k_bicg_p(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb,
                                                    unsigned long long* __restrict__ report) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto r = gm(static_cast<const double*>(S.r));
    const auto vv = gm(static_cast<const double*>(S.v));
    const auto dinv = gm(S.dinv);
    const auto p = gm(S.p);
    const auto ph = gm(S.ph);
    const int n = S.n;
    const Scalars st = take_step<FIN_BICG_RES>(S, first_, report, bk_.x);
    if (st.status != ST_RUNNING) {
        return;
    }
    const double beta = st.beta;
    const double omega = st.omega;
    for_group_rows<false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int) {
        const int row = slice * k_wave + lane;
        if (row < n) {
            const double pi = r[row] + beta * (p[row] - omega * vv[row]);
            p[row] = pi;
            ph[row] = pi * dinv[row];
        }
    });
}

// v = A ph, partial r0.v.
template <int Form>
__global__ void __launch_bounds__(k_block) k_bicg_v(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto vv = gm(S.v);
    const auto r0 = gm(static_cast<const double*>(S.r0));
    const L0Op<Form, double, GatherX<double>> A0(S.a64, {gm(static_cast<const double*>(S.ph))});
    const int n = S.n;
    if (S.st->status != ST_RUNNING) {
        return;
    }
    for_groups<1, true>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds, double (&v)[2][1]) {
        double y[2];
        double ri[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& r) { ri[h] = load_at<double>(r0, r); });
        l0_rows<H.value>(A0, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                store_at<double>(vv, row[h], y[h]);
                v[h][0] = ri[h] * y[h];
            }
        }
    }, [](int) { return SLOT_R0V; });
}

// Step FIN_BICG_ALPHA, then s = r - alpha v; sh = dinv s; partial s.s.
__global__ void __launch_bounds__(k_block) k_bicg_s(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto r = gm(static_cast<const double*>(S.r));
    const auto vv = gm(static_cast<const double*>(S.v));
    const auto dinv = gm(S.dinv);
    const auto sv = gm(S.s);
    const auto sh = gm(S.sh);
    const int n = S.n;
    const Scalars st = take_step<FIN_BICG_ALPHA>(S, first_, nullptr, 0);
    if (st.status != ST_RUNNING) {
        return;
    }
    const double alpha = st.alpha;
    for_groups<1, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][1]) {
        const int row = slice * k_wave + lane;
        if (row < n) {
            const double si = r[row] - alpha * vv[row];
            sv[row] = si;
            sh[row] = si * dinv[row];
            v[0][0] = si * si;
        }
    }, [](int) { return SLOT_SS; });
}

// Step FIN_BICG_S, then t = A sh with the partials t.t and t.s, or on the early exit x += alpha ph.
template <int Form>
__global__ void __launch_bounds__(k_block) k_bicg_t(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto tv = gm(S.t);
    const auto sv = gm(static_cast<const double*>(S.s));
    const auto x = gm(S.x);
    const auto ph = gm(static_cast<const double*>(S.ph));
    const L0Op<Form, double, GatherX<double>> A0(S.a64, {gm(static_cast<const double*>(S.sh))});
    const int n = S.n;
    const Scalars st = take_step<FIN_BICG_S>(S, first_, nullptr, 0);
    if (st.status == ST_CONVERGED_PENDING) {
        for_group_rows<false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int) {
            const int row = slice * k_wave + lane;
            if (row < n) {
                x[row] = x[row] + st.alpha * ph[row];
            }
        });
        return;
    }
    if (st.status != ST_RUNNING) {
        return;
    }
    for_groups<2, true>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds, double (&v)[2][2]) {
        double y[2];
        double si[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& r) { si[h] = load_at<double>(sv, r); });
        l0_rows<H.value>(A0, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                store_at<double>(tv, row[h], y[h]);
                v[h][0] = y[h] * y[h];
                v[h][1] = y[h] * si[h];
            }
        }
    }, [](int q) { return q == 0 ? SLOT_TT : SLOT_TS; });
}

// Step FIN_BICG_OMEGA, then x += alpha ph + omega sh; r = s - omega t; partials r.r and r0.r.
__global__ void __launch_bounds__(k_block) k_bicg_xr(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const auto x = gm(S.x);
    const auto r = gm(S.r);
    const auto ph = gm(static_cast<const double*>(S.ph));
    const auto sh = gm(static_cast<const double*>(S.sh));
    const auto sv = gm(static_cast<const double*>(S.s));
    const auto tv = gm(static_cast<const double*>(S.t));
    const auto r0 = gm(static_cast<const double*>(S.r0));
    const int n = S.n;
    const Scalars st = take_step<FIN_BICG_OMEGA>(S, first_, nullptr, 0);
    if (st.status != ST_RUNNING) {
        return;
    }
    const double alpha = st.alpha;
    const double omega = st.omega;
    for_groups<2, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][2]) {
        const int row = slice * k_wave + lane;
        if (row < n) {
            x[row] = x[row] + (alpha * ph[row] + omega * sh[row]);
            const double ri = sv[row] - omega * tv[row];
            r[row] = ri;
            v[0][0] = ri * ri;
            v[0][1] = r0[row] * ri;
        }
    }, [](int q) { return q == 0 ? SLOT_RR : SLOT_R0R; });
}

// ------------------------------------------------------------------------------------------
// V-cycle kernels (krylov_kernels.inc:182-238), element type T (double or float)
// ------------------------------------------------------------------------------------------

// Row mapping of a V-cycle kernel over matrix M: 256 / tpr rows per workgroup, tpr lanes per
// row. Early returns here are uniform over the workgroup.
// The system's status and the level's descriptor fields are requested before either is tested
// (one wait instead of a chain of dependent loads: the small levels' kernels are latency-bound).
#define CFDG_LEVEL_PROLOGUE(sysarr, blocks, level, MAT)                                            \
    const int2 bk_ = block_entry(blocks);                                                         \
    const SysDev& S = (sysarr)[bk_.x];                                                            \
    const LevelDev& L = S.lv[level];                                                              \
    const EllView M = L.MAT;                                                                      \
    const int tpr = M.tpr;                                                                        \
    if ((S.st->status != ST_RUNNING) | (L.coarsest != 0) | (tpr <= 0)) {                          \
        return;                                                                                   \
    }                                                                                             \
    const int row = bk_.y * (k_block / tpr) + static_cast<int>(threadIdx.x) / tpr;                \
    const int sub = static_cast<int>(threadIdx.x) & (tpr - 1);                                    \
    (void)sub;

// ------------------------------------------------------------------------------------------
// V-cycle operations on one row (or one lane of a row's group), used by the level kernels below.
// ------------------------------------------------------------------------------------------

// v[out] = (f wd) b.
template <class T>
__device__ __forceinline__ void op_jacobi_zero(const LevelDev& L, int row, int out, T f) {
    gm(static_cast<T*>(L.v[out]))[row] = (f * gm(static_cast<const T*>(L.wd))[row]) * gm(static_cast<const T*>(L.b))[row];
}

// v[out] = v[in] + (f wd) (b - A v[in]); returns the new entry (0 for rows past the end /
// sub > 0).
template <class T>
__device__ __forceinline__ T op_jacobi(const LevelDev& L, const EllView& M, int row, int sub, int in, int out, T f) {
    const T* x = static_cast<const T*>(L.v[in]);
    const auto b = gm(static_cast<const T*>(L.b));
    const auto wd = gm(static_cast<const T*>(L.wd));
    const T ax = mat_row<T>(M, row, sub, x);
    T z = T(0);
    if (sub == 0 && row < L.n) {
        z = x[row] + (f * wd[row]) * (b[row] - ax);
        gm(static_cast<T*>(L.v[out]))[row] = z;
    }
    return z;
}

// v[out] = b - A v[in].
template <class T>
__device__ __forceinline__ void op_residual(const LevelDev& L, const EllView& M, int row, int sub, int in, int out) {
    const T ax = mat_row<T>(M, row, sub, static_cast<const T*>(L.v[in]));
    if (sub == 0 && row < L.n) {
        gm(static_cast<T*>(L.v[out]))[row] = gm(static_cast<const T*>(L.b))[row] - ax;
    }
}

// v[out] = b - A x1 with x1 = (f wd) b formed per gathered column.
template <class T>
__device__ __forceinline__ void op_residual_x1(const LevelDev& L, const EllView& M, int row, int sub, int out, T f) {
    const auto b = gm(static_cast<const T*>(L.b));
    const auto wd = gm(static_cast<const T*>(L.wd));
    const T ax = mat_row_x1<T>(M, row, sub, wd, b, f);
    if (sub == 0 && row < L.n) {
        gm(static_cast<T*>(L.v[out]))[row] = b[row] - ax;
    }
}

// b_{l+1} = M x for a row of level l + 1 (M = R_l on a level vector, or the fused restriction
// on b_l); with x1_out >= 0 also v_{l+1}[x1_out] = (f wd) b unless level l + 1 is the coarsest.
template <class T>
__device__ __forceinline__ void op_restrict(const LevelDev& L, const LevelDev& N, const EllView& M, int row, int sub,
                                            const T* x, int x1_out, T f) {
    const T y = mat_row<T>(M, row, sub, x);
    if (sub == 0 && row < L.n_next) {
        gm(static_cast<T*>(N.b))[row] = y;
        if (x1_out >= 0 && !N.coarsest) {
            gm(static_cast<T*>(N.v[x1_out]))[row] = (f * gm(static_cast<const T*>(N.wd))[row]) * y;
        }
    }
}

// v_l[io] += P_l v_{l+1}[coarse_buf]; X1: v_l[io] = (f wd) b + P_l v_{l+1}[coarse_buf] (the
// level's single pre-sweep from zero was not stored).
template <class T, bool X1>
__device__ __forceinline__ void op_prolong(const LevelDev& L, const LevelDev& N, const EllView& M, int row, int sub,
                                           int io, int coarse_buf, T f) {
    const T t = mat_row<T>(M, row, sub, static_cast<const T*>(N.v[coarse_buf]));
    if (sub == 0 && row < L.n) {
        const auto x = gm(static_cast<T*>(L.v[io]));
        if constexpr (X1) {
            x[row] = (f * gm(static_cast<const T*>(L.wd))[row]) * gm(static_cast<const T*>(L.b))[row] + t;
        } else {
            x[row] = x[row] + t;
        }
    }
}

// Coarsest level, row i: v[out]_i = sum_j Cinv_ij b_j in FP64 by one wavefront (lane-strided
// partial sums, then the wavefront butterfly). A row's time is its loads' latency: 8 entries a lane
// are requested before the first is added (all of a row of 512). Order 507 (128^3's tail): 6.6 us one
// entry at a time, 4.6 so; 2.1 MB.
template <class T>
__device__ __forceinline__ void op_coarse_row(const LevelDev& L, int i, int lane, int out) {
    constexpr int G = 8;
    const int n = L.n;
    const auto m = gm(L.cinv) + static_cast<long long>(i) * L.n;
    const auto b = gm(static_cast<const T*>(L.b));
    double s = 0.0;
    for (unsigned j0 = static_cast<unsigned>(lane); j0 < n; j0 += G * k_wave) {
        double a[G];
        T x[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const unsigned j = j0 + static_cast<unsigned>(g * k_wave);
            const unsigned c = min(j, n - 1);
            a[g] = load_at<double>(m, c);
            x[g] = load_at<T>(b, c);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            if (j0 + static_cast<unsigned>(g * k_wave) < n) {
                s += a[g] * static_cast<double>(x[g]);
            }
        }
    }
    s = wave_sum(s);
    if (lane == 0) {
        gm(static_cast<T*>(L.v[out]))[i] = static_cast<T>(s);
    }
}

// One Jacobi sweep from x = 0: v[out] = (f wd) b (row-wise, 256 rows per workgroup).
template <class T>
__global__ void __launch_bounds__(k_block) k_jacobi_zero(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int out,
                                                         T f) {
    CFDG_BLOCK_PROLOGUE(sys, blocks)
    const LevelDev& L = S.lv[level]; // fields requested with the status (one wait)
    if ((S.st->status != ST_RUNNING) | (L.coarsest != 0) | (row >= L.n)) {
        return;
    }
    op_jacobi_zero<T>(L, row, out, f);
}

// v[out] = 0 (smoothing-free V-cycles; row-wise).
template <class T>
__global__ void __launch_bounds__(k_block) k_zero_level(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int out) {
    CFDG_BLOCK_PROLOGUE(sys, blocks)
    if (S.st->status != ST_RUNNING) {
        return;
    }
    const LevelDev& L = S.lv[level];
    if (L.coarsest || row >= L.n) {
        return;
    }
    gm(static_cast<T*>(L.v[out]))[row] = T(0);
}

// Jacobi sweep v[out] = v[in] + (f wd) (b - A v[in]).
template <class T>
__global__ void __launch_bounds__(k_block) k_jacobi(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int in, int out,
                                                    T f) {
    CFDG_LEVEL_PROLOGUE(sys, blocks, level, a)
    (void)op_jacobi<T>(L, M, row, sub, in, out, f);
}

// ------------------------------------------------------------------------------------------
// Level-0 V-cycle kernels over row groups (the finest operator is sliced ELL, one lane per row)
// ------------------------------------------------------------------------------------------

// State of the cycle's first kernel: step FIN_RES made here (Step), or made by a launch before it.
template <bool Step>
__device__ __forceinline__ bool cycle_runs(const SysDev& S, bool first, unsigned long long* report, int id) {
    if constexpr (Step) {
        return take_step<FIN_RES>(S, first, report, id).status == ST_RUNNING;
    } else {
        return S.st->status == ST_RUNNING;
    }
}

// v[out] = b - A x1 with x1 = (f wd) b, the single Jacobi sweep from zero, formed per gathered
// column instead of stored (one pre-sweep per side).
// 16.0 us at 128^3 in FP32 with the step (before: 17.4 and 5.2 for the step's launch).
template <class T, int Form, bool Step>
__global__ void __launch_bounds__(k_block) k_l0_residual_x1(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb, int out,
                                                            T f, unsigned long long* __restrict__ report) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const LevelDev& L = S.lv[0];
    const auto b = gm(static_cast<const T*>(L.b));
    const auto t = gm(static_cast<T*>(L.v[out]));
    const L0Op<Form, T, GatherX1<T>> M(L.a, {gm(static_cast<const T*>(L.wd)), b, f});
    const int n = L.n;
    if (!cycle_runs<Step>(S, first_, report, bk_.x) | (L.coarsest != 0)) {
        return;
    }
    for_group_rows<true>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds) {
        T y[2];
        T bi[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& r) { bi[h] = load_at<T>(b, r); });
        l0_rows<H.value>(M, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                store_at<T>(t, row[h], bi[h] - y[h]);
            }
        }
    });
}

// First two Jacobi sweeps from x = 0: v[out] = x1 + (f2 wd) (b - A x1), x1 = (f1 wd) b (the gathers
// of wd and b stay cache-resident for short rows). f1, f2: the sweeps' factors on the level's
// damping (Chebyshev weights; 1 for plain damped Jacobi, which leaves the arithmetic unchanged).
template <class T, int Form, bool Step>
__global__ void __launch_bounds__(k_block) k_l0_presmooth2(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb, int out,
                                                           T f1, T f2, unsigned long long* __restrict__ report) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const LevelDev& L = S.lv[0];
    const auto b = gm(static_cast<const T*>(L.b));
    const auto wd = gm(static_cast<const T*>(L.wd));
    const auto x = gm(static_cast<T*>(L.v[out]));
    const L0Op<Form, T, GatherX1<T>> M(L.a, {wd, b, f1});
    const int n = L.n;
    if (!cycle_runs<Step>(S, first_, report, bk_.x) | (L.coarsest != 0)) {
        return;
    }
    for_group_rows<true>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds) {
        T y[2];
        T bi[2];
        T wi[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& r) {
            bi[h] = load_at<T>(b, r);
            wi[h] = load_at<T>(wd, r);
        });
        l0_rows<H.value>(M, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                const T x1 = (f1 * wi[h]) * bi[h];
                store_at<T>(x, row[h], x1 + (f2 * wi[h]) * (bi[h] - y[h]));
            }
        }
    });
}

// k_residual and k_jacobi of level 0 for launches whose systems all have the operator in L0_SYM7 form: 256
// rows a workgroup, the stencil in scalar registers and the row as the only vector address. FP64 at 128^3
// 24.0 -> 21.4 us and 35.3 -> 34.3 (as row groups 23.5 and 35.2: neither has a step or a dot product to
// share among a group's rows).
#define CFDG_SYM7_PROLOGUE(sysarr, blocks, in)                                                    \
    const int2 bk_ = block_entry(blocks);                                                         \
    const SysDev& S = (sysarr)[bk_.x];                                                            \
    const LevelDev& L = S.lv[0];                                                                  \
    const int wave_ = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / k_wave);     \
    const int lane = static_cast<int>(threadIdx.x) % k_wave;                                      \
    const int slice = bk_.y * k_slices_per_block + wave_;                                         \
    const unsigned row = static_cast<unsigned>(slice * k_wave + lane);                            \
    const unsigned r = in_matrix(row, L.n);                                                       \
    const auto x = gm(static_cast<const T*>(L.v[in]));                                            \
    const T bi = load_at<T>(gm(static_cast<const T*>(L.b)), r);

template <class T>
__global__ void __launch_bounds__(k_block) k_sym7_residual(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int in, int out) {
    CFDG_SYM7_PROLOGUE(sys, blocks, in)
    const L0Op<L0_SYM7, T, GatherX<T>> M(L.a, {x});
    if ((S.st->status != ST_RUNNING) | (L.coarsest != 0)) {
        return;
    }
    T y[2];
    l0_rows<1>(M, slice, 0, lane, y);
    if (inside(row, L.n)) {
        store_at<T>(gm(static_cast<T*>(L.v[out])), row, bi - y[0]);
    }
}

template <class T>
__global__ void __launch_bounds__(k_block) k_sym7_jacobi(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int in, int out, T f) {
    CFDG_SYM7_PROLOGUE(sys, blocks, in)
    const T wi = load_at<T>(gm(static_cast<const T*>(L.wd)), r);
    const T xi = load_at<T>(x, r);
    const L0Op<L0_SYM7, T, GatherX<T>> M(L.a, {x});
    if ((S.st->status != ST_RUNNING) | (L.coarsest != 0)) {
        return;
    }
    T y[2];
    l0_rows<1>(M, slice, 0, lane, y);
    if (inside(row, L.n)) {
        store_at<T>(gm(static_cast<T*>(L.v[out])), row, xi + (f * wi) * (bi - y[0]));
    }
}

// The last post-sweep v[out] = v[in] + (f wd) (b - A v[in]) with the dot products of its result:
// Dots 1 partial r.z with r = b (FP64 level 0, where b aliases r); 2 partials r.z and z.q with r, q
// the FP64 outer vectors (mixed level 0). Pair: two chunks' rows at a time (the same results bit
// for bit; slower on BF16 rows).
template <class T, int Form, int Dots, bool Pair>
__global__ void __launch_bounds__(k_block) k_l0_jacobi(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb, int in, int out,
                                                       T f) {
    CFDG_L0_PROLOGUE(sys, blocks)
    const LevelDev& L = S.lv[0];
    const auto x = gm(static_cast<const T*>(L.v[in]));
    const auto b = gm(static_cast<const T*>(L.b));
    const auto wd = gm(static_cast<const T*>(L.wd));
    const auto o = gm(static_cast<T*>(L.v[out]));
    const auto r = gm(static_cast<const double*>(S.r));
    const auto qv = gm(static_cast<const double*>(S.q));
    const L0Op<Form, T, GatherX<T>> M(L.a, {x});
    const int n = L.n;
    if ((S.st->status != ST_RUNNING) | (L.coarsest != 0)) {
        return;
    }
    for_groups<Dots, Pair>(S, bk_.y, gpb, wave_, [&](auto H, int slice, int ds, double (&v)[2][Dots]) {
        T y[2];
        T bi[2];
        T wi[2];
        T xi[2];
        double ri[2];
        double qi[2];
        RowOf<Form> row[2];
        own_rows<H.value>(slice, ds, lane, n, row, [&](int h, const auto& i) {
            bi[h] = load_at<T>(b, i);
            wi[h] = load_at<T>(wd, i);
            xi[h] = load_at<T>(x, i);
            if constexpr (Dots == 2) {
                ri[h] = load_at<double>(r, i);
                qi[h] = load_at<double>(qv, i);
            }
        });
        l0_rows<H.value>(M, slice, ds, lane, y);
#pragma unroll
        for (int h = 0; h < H.value; ++h) {
            if (inside(row[h], n)) {
                const T z = xi[h] + (f * wi[h]) * (bi[h] - y[h]);
                store_at<T>(o, row[h], z);
                const double zd = static_cast<double>(z);
                if constexpr (Dots == 1) {
                    v[h][0] = static_cast<double>(bi[h]) * zd;
                } else {
                    v[h][0] = ri[h] * zd;
                    v[h][1] = zd * qi[h];
                }
            }
        }
    }, [](int q) { return q == 0 ? SLOT_RZ : SLOT_ZQ; });
}

// Level-0 dot products from a finished V-cycle output v[buf] (used when no Jacobi sweep on
// level 0 could carry them: one-level hierarchies and smoothing-free cycles).
template <class T, int Dots>
__global__ void __launch_bounds__(k_block) k_level0_dots(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int gpb, int buf) {
    CFDG_L0_PROLOGUE(sys, blocks)
    if (S.st->status != ST_RUNNING) {
        return;
    }
    const LevelDev& L = S.lv[0];
    for_groups<Dots, false>(S, bk_.y, gpb, wave_, [&](auto, int slice, int, double (&v)[2][Dots]) {
        const int row = slice * k_wave + lane;
        if (row < S.n) {
            const double z = static_cast<double>(static_cast<const T*>(L.v[buf])[row]);
            if constexpr (Dots == 1) {
                v[0][0] = static_cast<double>(static_cast<const T*>(L.b)[row]) * z;
            } else {
                v[0][0] = S.r[row] * z;
                v[0][1] = z * S.q[row];
            }
        }
    }, [](int q) { return q == 0 ? SLOT_RZ : SLOT_ZQ; });
}

// Workgroup of the level kernels that serve two slices per wavefront.
constexpr int k_block_pair = k_block / 2;

// Rows of one table entry (the 256 / tpr rows a k_block workgroup covers) for a k_block_pair
// workgroup: sliced ELL reads slices 4 y + 2 w and 4 y + 2 w + 1 together in wave w; CSR rows run
// as the two halves of the k_block lanes. epi(row, sub, value) gets every lane's row product
// (complete in every lane of the row's group); rows past the end give 0. Bit-identical to
// mat_row on the same rows.
template <class T, class F, class E>
__device__ __forceinline__ void pair_rows(const EllView& m, int y, F load, E epi) {
    const int lane = static_cast<int>(threadIdx.x) % k_wave;
    const int tpr = m.tpr;
    if (m.csr == 0) {
        const int lg = __builtin_ctz(tpr);
        const int s0 = y * k_slices_per_block + 2 * (static_cast<int>(threadIdx.x) / k_wave);
        T ya;
        T yb;
        ell_row_pair<T>(m, s0, 1, lane, load, ya, yb);
        if (tpr > 1) {
            ya = group_sum(ya, tpr);
            yb = group_sum(yb, tpr);
        }
        const int r0 = s0 * (k_wave >> lg) + (lane >> lg);
        epi(r0, lane & (tpr - 1), ya);
        epi(r0 + (k_wave >> lg), lane & (tpr - 1), yb);
        return;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int vt = static_cast<int>(threadIdx.x) + h * k_block_pair;
        const int row = y * (k_block / tpr) + vt / tpr;
        T v = T(0);
        if (row < m.n_rows) {
            v = csr_lane_sum<T>(gm(m.col), gm(static_cast<const T*>(m.val)), m.sp[row] + (vt & (tpr - 1)),
                                m.sp[row + 1], tpr, load);
        }
        epi(row, vt & (tpr - 1), group_sum(v, tpr));
    }
}

#define CFDG_PAIR_LEVEL_PROLOGUE(sysarr, blocks, level)                                           \
    const int2 bk_ = block_entry(blocks);                                                         \
    const SysDev& S = (sysarr)[bk_.x];                                                            \
    const LevelDev& L = S.lv[level];                                                              \
    if ((S.st->status != ST_RUNNING) | (L.coarsest != 0)) {                                       \
        return;                                                                                   \
    }

// k_prolong with pair_rows: v_l[io] += P_l v_{l+1}[coarse_buf]; X1: v_l[io] = (f wd) b +
// P_l v_{l+1}.
template <class T, bool X1>
__global__ void __launch_bounds__(k_block_pair) k_prolong_pair(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int io,
                                                               int coarse_buf, T f) {
    CFDG_PAIR_LEVEL_PROLOGUE(sys, blocks, level)
    const LevelDev& N = S.lv[level + 1];
    const auto e = gm(static_cast<const T*>(N.v[coarse_buf]));
    const auto x = gm(static_cast<T*>(L.v[io]));
    pair_rows<T>(L.p, bk_.y, GatherX<T>{e}, [&](int row, int sub, T t) {
        if (sub == 0 && row < L.n) {
            if constexpr (X1) {
                x[row] = (f * gm(static_cast<const T*>(L.wd))[row]) * gm(static_cast<const T*>(L.b))[row] + t;
            } else {
                x[row] = x[row] + t;
            }
        }
    });
}

// v[out] = b - A v[in].
template <class T>
__global__ void __launch_bounds__(k_block) k_residual(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int in, int out) {
    CFDG_LEVEL_PROLOGUE(sys, blocks, level, a)
    op_residual<T>(L, M, row, sub, in, out);
}

// b_{l+1} = R_l v_l[in]; rows of level l + 1. With x1_out >= 0 the next level's first
// Jacobi sweep from zero is stored too, v_{l+1}[x1_out] = (f wd) b_{l+1} (what k_jacobi_zero
// would compute from the stored b), unless level l + 1 is the coarsest.
template <class T>
__global__ void __launch_bounds__(k_block) k_restrict(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int in,
                                                      int x1_out, T f) {
    CFDG_LEVEL_PROLOGUE(sys, blocks, level, r)
    op_restrict<T>(L, S.lv[level + 1], M, row, sub, static_cast<const T*>(L.v[in]), x1_out, f);
}

// Down leg of a level with one Jacobi sweep from zero as one product: b_{l+1} = R (I - A W) b_l,
// W = diag(wd) (x1 = W b, r = b - A x1, b_{l+1} = R r in exact arithmetic); rows of level l + 1;
// x1_out as k_restrict.
template <class T>
__global__ void __launch_bounds__(k_block) k_restrict_fused(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level,
                                                            int x1_out, T f) {
    CFDG_LEVEL_PROLOGUE(sys, blocks, level, rt)
    op_restrict<T>(L, S.lv[level + 1], M, row, sub, static_cast<const T*>(L.b), x1_out, f);
}

// v_l[io] += P_l v_{l+1}[coarse_buf]. X1: the level's single pre-sweep from zero was not
// stored; its result (f wd) b is formed here (v[io] = (f wd) b + P v_{l+1}, the same sums).
template <class T, bool X1 = false>
__global__ void __launch_bounds__(k_block) k_prolong(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int io,
                          int coarse_buf, T f) {
    CFDG_LEVEL_PROLOGUE(sys, blocks, level, p)
    op_prolong<T, X1>(L, S.lv[level + 1], M, row, sub, io, coarse_buf, f);
}

// v[out] = b - A x1 with x1 = (f wd) b, the single Jacobi sweep from zero, formed per
// gathered column instead of stored (one pre-sweep per side).
template <class T>
__global__ void __launch_bounds__(k_block) k_residual_x1(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int out,
                                                         T f) {
    CFDG_LEVEL_PROLOGUE(sys, blocks, level, a)
    op_residual_x1<T>(L, M, row, sub, out, f);
}

// Coarsest level: v[out] = C^-1 b with the dense FP64 inverse, one wavefront per row; blocks
// index groups of four rows.
template <class T>
__global__ void __launch_bounds__(k_block) k_coarse(const SysDev* __restrict__ sys, const int2* __restrict__ blocks, int level, int out) {
    const int2 bk = block_entry(blocks);
    const SysDev& S = sys[bk.x];
    const LevelDev& L = S.lv[level]; // fields requested with the status (one wait)
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / k_wave);
    const int lane = threadIdx.x % k_wave;
    const int i = bk.y * k_slices_per_block + wave;
    if ((S.st->status != ST_RUNNING) | (L.coarsest == 0) | (i >= L.n)) {
        return;
    }
    op_coarse_row<T>(L, i, lane, out);
}

// ------------------------------------------------------------------------------------------
// Normalised residual (ldu_matrix.cpp:65-103): res = sum_c |b_c - (Ax)_c| and
// norm = sum_c |(Ax)_c - (A xref)_c| + |b_c - (A xref)_c|, with A xref = rowsum(A) * mean(x).
// Three passes with fixed-order sums: block sums of x, their total, then per row the two terms
// and (b - Ax)^2 (the level-0 FP64 operator, one lane per row, rows of 256-row blocks).
// ------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(k_block) k_nr_xsum(int n, const double* __restrict__ x, double* __restrict__ part) {
    const int i = blockIdx.x * k_block + threadIdx.x;
    double v[1] = {i < n ? x[i] : 0.0};
    double o[1];
    block_sums<1>(v, o);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = o[0];
    }
}

// sums[0] = sum of x (k_nr_reduce); part receives three arrays of nblk block sums.
__global__ void __launch_bounds__(k_block) k_nr_rows(EllView a, int n, const double* __restrict__ x,
                                                     const double* __restrict__ b, const double* __restrict__ sums,
                                                     double* __restrict__ part, int nblk) {
    const int wave = threadIdx.x / k_wave;
    const int lane = threadIdx.x % k_wave;
    const int slice = blockIdx.x * k_slices_per_block + wave;
    const int row = slice * k_wave + lane;
    const double mean = sums[0] / static_cast<double>(n);
    double t[3] = {0.0, 0.0, 0.0};
    if (slice < a.n_slices) {
        const double ax = ell_row<double>(a, slice, lane, x);
        const double rs = ell_row_f<double>(a, slice, lane, GatherOne{});
        if (row < n) {
            const double bi = b[row];
            const double ax_ref = rs * mean;
            const double r = bi - ax;
            t[0] = fabs(r);
            t[1] = fabs(ax - ax_ref) + fabs(bi - ax_ref);
            t[2] = r * r;
        }
    }
    double o[3];
    block_sums<3>(t, o);
    if (threadIdx.x == 0) {
        part[blockIdx.x] = o[0];
        part[nblk + blockIdx.x] = o[1];
        part[2 * nblk + blockIdx.x] = o[2];
    }
}

constexpr int k_fin_block = 1024;

// out[q] = sum over i < nblk of part[q nblk + i], q < count, in a fixed order (one workgroup).
__global__ void __launch_bounds__(k_fin_block) k_nr_reduce(const double* __restrict__ part, int nblk, int count,
                                                           double* __restrict__ out) {
    __shared__ double red[k_fin_block / k_wave];
    for (int q = 0; q < count; ++q) {
        const double* p = part + static_cast<long long>(q) * nblk;
        double s = 0.0;
        for (int i = threadIdx.x; i < nblk; i += k_fin_block) {
            s += p[i];
        }
        s = wave_sum(s);
        if (threadIdx.x % k_wave == 0) {
            red[threadIdx.x / k_wave] = s;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = red[0];
            for (int w = 1; w < k_fin_block / k_wave; ++w) {
                t += red[w];
            }
            out[q] = t;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------
// Assembly kernels
// ------------------------------------------------------------------------------------------

// Level-0 values from LDU coefficients: val[k] = ldu[src[k]] (0 for padding), with
// ldu = [diag | upper | lower]; dinv = 1 / diag (1.0 for a zero diagonal,
// krylov_cuda.cu:557-562); wd = w dinv in FP64 and FP32; FP32 copy of the values.
__global__ void __launch_bounds__(k_block) k_ldu_gather(long long n_slots, const int* __restrict__ src, const double* __restrict__ ldu,
                             double* __restrict__ val64, float* __restrict__ val32) {
    const long long k = static_cast<long long>(blockIdx.x) * k_block + threadIdx.x;
    if (k >= n_slots) {
        return;
    }
    const int s = src[k];
    const double v = s >= 0 ? ldu[s] : 0.0;
    val64[k] = v;
    if (val32 != nullptr) {
        val32[k] = static_cast<float>(v);
    }
}

// flag = 1 if some face's upper and lower coefficients differ in any bit (the operator is not
// exactly symmetric); flag is cleared by the caller.
__global__ void __launch_bounds__(k_block) k_ldu_asymmetric(int nf, const double* __restrict__ upper,
                                                            const double* __restrict__ lower, int* __restrict__ flag) {
    const int f = blockIdx.x * k_block + threadIdx.x;
    if (f < nf && __double_as_longlong(upper[f]) != __double_as_longlong(lower[f])) {
        *flag = 1;
    }
}

// dinv = 1 / a_ii (1.0 for a zero diagonal), wd64 = w64 dinv (FP64 smoother), wd32 = w32 dinv
// (mixed smoother).
__global__ void __launch_bounds__(k_block) k_diag_inverse(int n, const double* __restrict__ diag, double w64, double w32,
                                                          double* __restrict__ dinv, double* __restrict__ wd64,
                                                          float* __restrict__ wd32) {
    const int i = blockIdx.x * k_block + threadIdx.x;
    if (i >= n) {
        return;
    }
    const double d = diag[i];
    const double di = d != 0.0 ? 1.0 / d : 1.0;
    dinv[i] = di;
    wd64[i] = w64 * di;
    if (wd32 != nullptr) {
        wd32[i] = static_cast<float>(w32 * di);
    }
}

// Face coefficients of the convection-diffusion operator (krylov_openmp.cpp:289-295).
__global__ void __launch_bounds__(k_block) k_assemble_faces(int nf, const double* __restrict__ flux, const double* __restrict__ gamma,
                                 const double* __restrict__ delta, double convection,
                                 double* __restrict__ upper, double* __restrict__ lower) {
    const int f = blockIdx.x * k_block + threadIdx.x;
    if (f >= nf) {
        return;
    }
    const double fl = flux[f];
    const double g = gamma[f] * delta[f];
    const double pos = fl > 0.0 ? convection * fl : 0.0;
    const double neg = fl < 0.0 ? convection * fl : 0.0;
    upper[f] = neg - g;
    lower[f] = -pos - g;
}

// Per-cell accumulation of diag / divergence over the cell's faces in ascending face order,
// the order of the reference's serial face loop (krylov_openmp.cpp:296-299).
__global__ void __launch_bounds__(k_block) k_assemble_cells(int nc, const int* __restrict__ cf_ptr, const int* __restrict__ cf_face,
                                 const int* __restrict__ owner, const double* __restrict__ flux,
                                 const double* __restrict__ gamma, const double* __restrict__ delta,
                                 double convection, double* __restrict__ diag,
                                 double* __restrict__ divergence) {
    const int c = blockIdx.x * k_block + threadIdx.x;
    if (c >= nc) {
        return;
    }
    double d = diag[c];
    double dv = divergence[c];
    for (int k = cf_ptr[c]; k < cf_ptr[c + 1]; ++k) {
        const int f = cf_face[k];
        const double fl = flux[f];
        const double g = gamma[f] * delta[f];
        const double pos = fl > 0.0 ? convection * fl : 0.0;
        const double neg = fl < 0.0 ? convection * fl : 0.0;
        if (owner[f] == c) {
            d += pos + g;
            dv += fl;
        } else {
            d += -neg + g;
            dv -= fl;
        }
    }
    diag[c] = d;
    divergence[c] = dv;
}

} // namespace cfdg
