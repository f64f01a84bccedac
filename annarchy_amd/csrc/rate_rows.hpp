// rate_rows.hpp -- row sums of the rate-coded psp (y = W . r), shared by the
// psp kernels (k_rate_psp.hip, k_delay.hip) and by the generated updates that
// sum their own rows (ahip_fuse_args).
//
// FP64: plain sums.  FP32: Neumaier-compensated lane sums and a compensated
// lane reduction.
#pragma once

#include "ahip_device.hpp"

namespace ahip {

template <typename T>
struct Acc;
template <>
struct Acc<double> {
    double s = 0.0;
    __device__ inline void add(double x) { s += x; }
    __device__ inline void join(const Acc& o) { s += o.s; }
    template <int W>
    __device__ inline double reduce() { return group_sum<W>(s); }
    __device__ inline double reduce_rt(int shift) { return group_sum_rt(s, shift); }
};
template <>
struct Acc<float> {
    Kahan k{0.0f, 0.0f};
    __device__ inline void add(float x) { k.add(x); }
    __device__ inline void join(const Acc& o) {
        k.add(o.k.s);
        k.c += o.k.c;
    }
    template <int W>
    __device__ inline float reduce() { return group_sum_kahan<W>(k.s, k.c); }
    __device__ inline float reduce_rt(int shift) {
        float s = k.s, c = k.c;
        group_join_kahan(s, c, shift);
        return s + c;
    }
};

// the accumulators of the 64 lanes of a wave joined (every lane ends with the
// sum, FP32 with its compensation)
__device__ inline void wave_join(Acc<double>& a) { a.s = group_sum<kWave>(a.s); }
__device__ inline void wave_join(Acc<float>& a) { group_join_kahan(a.k.s, a.k.c, log2_of(kWave)); }

typedef double v2d_t __attribute__((ext_vector_type(2)));
typedef float v4f_t __attribute__((ext_vector_type(4)));

// 4 consecutive weights, 16-byte aligned
__device__ inline void load4(double (&v)[4], const double* p) {
    const v2d_t a = reinterpret_cast<const v2d_t*>(p)[0], b = reinterpret_cast<const v2d_t*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y;
}
__device__ inline void load4(float (&v)[4], const float* p) {
    const v4f_t a = *reinterpret_cast<const v4f_t*>(p);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
}

// Entries j, j + stride, ... < end of one lane (32-bit positions: a uniform
// base and a 32-bit offset per load).  4 columns and 4 weights are in flight
// before the first rate is gathered, and the next 4 while these are added (the
// last pass reads its first entry again for those past the end and adds 0 for
// them).  x(c): the rate of column c.
template <typename T>
struct Entries {
    int32_t c[4];
    T v[4];
    __device__ inline void load(uint32_t j, uint32_t end, uint32_t stride, const int32_t* __restrict__ col,
                                const T* __restrict__ w) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t q = j + u * stride;
            const uint32_t at = q < end ? q : j;
            c[u] = col[at];
            v[u] = w[at];
        }
    }
};
template <typename T, typename X>
__device__ inline void lane_entries(Acc<T>& a0, Acc<T>& a1, uint32_t j, uint32_t end, uint32_t stride,
                                    const int32_t* __restrict__ col, const T* __restrict__ w, X x) {
    Entries<T> e, next;
    if (j < end) e.load(j, end, stride, col, w);
    while (j < end) {
        const uint32_t jn = j + 4 * stride;
        if (jn < end) next.load(jn, end, stride, col, w);
        T r[4];
#pragma unroll
        for (int u = 0; u < 4; u++) r[u] = x(e.c[u]);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const T p = j + u * stride < end ? e.v[u] * r[u] : T(0);
            if (u & 1) a1.add(p);
            else a0.add(p);
        }
        e = next;
        j = jn;
    }
}

// The same with a delay of d steps per entry: x is a ring of D slots of
// n_cols values, `now` the slot of the current step (d <= D).
template <typename T>
__device__ inline void lane_entries_delayed(Acc<T>& a0, Acc<T>& a1, uint32_t j, uint32_t end, uint32_t stride,
                                            const int32_t* __restrict__ col, const T* __restrict__ w,
                                            const int16_t* __restrict__ delay, const T* __restrict__ ring,
                                            int32_t now, int32_t D, int32_t n_cols) {
    for (; j < end; j += 4 * stride) {
        int32_t d[4];
        Entries<T> e;
        e.load(j, end, stride, col, w);
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const uint32_t q = j + u * stride;
            d[u] = delay[q < end ? q : j];
        }
        T r[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int32_t s = now - d[u];
            r[u] = ring[(uint32_t)((s < 0 ? s + D : s) * n_cols + e.c[u])];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const T p = j + u * stride < end ? e.v[u] * r[u] : T(0);
            if (u & 1) a1.add(p);
            else a0.add(p);
        }
    }
}

constexpr int kDenseRows = 4;   // rows a workgroup of 4 waves sums together

// An accumulator in LDS (no constructor): sum and compensation.
template <typename T>
struct Partial {
    T s, c;
};
__device__ inline Partial<double> partial_of(const Acc<double>& a) { return {a.s, 0.0}; }
__device__ inline Partial<float> partial_of(const Acc<float>& a) { return {a.k.s, a.k.c}; }
__device__ inline void join_partial(Acc<double>& a, const Partial<double>& p) { a.s += p.s; }
__device__ inline void join_partial(Acc<float>& a, const Partial<float>& p) {
    a.k.add(p.s);
    a.k.c += p.c;
}

// Rows row0 .. row0 + 3 (clamped to n_rows - 1) of a dense matrix by `waves`
// waves: wave v takes every waves-th run of 256 columns for all 4 rows, so a
// rate is read once per 4 weights.  Leaves the wave's partial sums of row r in
// part[r * waves + v]; the reader joins them after a barrier.
template <typename T>
__device__ inline void dense_rows4(const T* __restrict__ W, int64_t ld, int32_t n_cols, int64_t row0, int64_t n_rows,
                                   const T* __restrict__ x, int v, int waves, Partial<T>* part) {
    const int lane = threadIdx.x & (kWave - 1);
    const T* wr[kDenseRows];
#pragma unroll
    for (int r = 0; r < kDenseRows; r++) wr[r] = W + min(row0 + r, n_rows - 1) * ld;
    Acc<T> acc[kDenseRows];
    for (int32_t k = (v * kWave + lane) * 4; k < n_cols; k += waves * 4 * kWave) {
        T wv[kDenseRows][4], xv[4];
#pragma unroll
        for (int r = 0; r < kDenseRows; r++) load4(wv[r], wr[r] + k);
#pragma unroll
        for (int e = 0; e < 4; e++) xv[e] = x[min(k + e, n_cols - 1)];
#pragma unroll
        for (int r = 0; r < kDenseRows; r++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[r].add(k + e < n_cols ? wv[r][e] * xv[e] : T(0));
    }
#pragma unroll
    for (int r = 0; r < kDenseRows; r++) {
        wave_join(acc[r]);
        if (lane == 0) part[r * waves + v] = partial_of(acc[r]);
    }
}

template <typename T>
__device__ inline T join_parts(const Partial<T>* part, int waves) {
    Acc<T> s;
    for (int v = 0; v < waves; v++) join_partial(s, part[v]);
    return s.template reduce<1>();
}

// ---- updates that sum their own rows -------------------------------------
// A workgroup owns F.share units (rows, or SELL slices).  Its first
// F.update_waves waves run the neurons' statements, one lane per row: they load
// the neuron's values and draw its random numbers while the other waves sum
// the rows into LDS, and finish after the barrier.

// Whether a projection feeds psp sum k.
__device__ inline bool has_sum(const ahip_fuse_args& F, int k) { return (F.mask >> k) & 1u; }

// The workgroup's place in row order.  Workgroups go round the 8 XCDs, so each
// XCD takes an eighth of the rows: a line of rates is then written by one XCD.
// The grid is padded to a multiple of 8; places past the last are idle.
__device__ inline int32_t fused_place() { return (int32_t)((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3)); }

// The neuron of update lane `k` of the workgroup at `place` (-1: none).
__device__ inline int32_t fused_neuron(const ahip_fuse_args& F, int32_t place, int32_t k) {
    const int rs = F.perm ? 6 - F.lane_shift : 0;   // log2 of the rows per unit
    const int32_t pos = ((place * F.share) << rs) + k;
    if (k >= (F.share << rs) || pos >= (F.units << rs)) return -1;
    return F.perm ? F.perm[pos] : pos;
}

// The sums of the workgroup's rows over every projection, in creation order,
// by its waves v = 0 .. waves - 1: sums[k][row of the workgroup] (a dense
// projection alone: the waves' partial sums in part).  KIND: the form of every
// projection (AHIP_FUSE_MIX: each by its descriptor).  xs: the staged rates.
template <typename T, int K, int KIND, bool STAGE>
__device__ inline void fused_rows(const ahip_fuse_args& F, int32_t place, int64_t t, int32_t n_rows, int v, int waves,
                                  const T* xs, T (&sums)[K][AHIP_FUSE_ROWS], Partial<T>* part) {
    const int lane = threadIdx.x & (kWave - 1);
    const int L = 1 << F.lane_shift;
    const int32_t lo = place * F.share, hi = min(F.units, lo + F.share);
    if constexpr (KIND == AHIP_FUSE_DENSE) {
        const ahip_fuse_proj& P = F.p[0];
        const T* x = static_cast<const T*>(P.x) + ring_slot(t - P.delay, P.depth) * P.n_cols;
        for (int32_t r = lo; r < hi; r += kDenseRows)
            dense_rows4<T>(static_cast<const T*>(P.w), P.ld, P.n_cols, r, n_rows, x, v, waves, part + (r - lo) * waves);
        return;
    }
    const int rs = F.perm ? 6 - F.lane_shift : 0;
    const int32_t per_wave = F.perm ? 1 : kWave >> F.lane_shift;
    for (int32_t u0 = lo + v * per_wave; u0 < hi; u0 += waves * per_wave) {
        const int32_t unit = u0 + (F.perm ? 0 : lane >> F.lane_shift);
        const bool in = unit < hi;
        const int32_t at = ((unit - lo) << rs) + (F.perm ? lane >> F.lane_shift : 0);   // row of the workgroup
        int32_t i = in ? unit : -1;
        if (KIND == AHIP_FUSE_MIX && F.perm) i = F.perm[(unit << rs) + (lane >> F.lane_shift)];
        T sum[K];
#pragma unroll
        for (int k = 0; k < K; k++) sum[k] = T(0);
        int32_t lds = 0;
        for (int32_t p = 0; p < F.n; p++) {
            const ahip_fuse_proj& P = F.p[p];
            const int kind = KIND == AHIP_FUSE_MIX ? P.kind : KIND;
            const T* w = static_cast<const T*>(P.w);
            const bool slice = kind == AHIP_FUSE_SELL;
            Acc<T> a0, a1;
            uint32_t beg = 0, end = 0;
            if (KIND == AHIP_FUSE_MIX && kind == AHIP_FUSE_DENSE) {
                if (i >= 0) {
                    beg = (uint32_t)i * P.ld;
                    end = beg + P.n_cols;
                }
            } else {
                const int32_t row = slice ? unit : i;
                if (row >= 0) {
                    beg = (uint32_t)P.ptr[row];
                    end = (uint32_t)P.ptr[row + 1];
                }
            }
            const uint32_t j = beg + (slice ? lane : lane & (L - 1));
            const uint32_t stride = slice ? kWave : L;
            if (KIND == AHIP_FUSE_MIX && !STAGE && kind == AHIP_FUSE_CSR_DELAY) {
                lane_entries_delayed<T>(a0, a1, j, end, stride, P.col, w, P.delays, static_cast<const T*>(P.x),
                                        (int32_t)ring_slot(t, P.depth), P.depth, P.n_cols);
            } else if constexpr (STAGE) {
                const T* x = xs + lds;
                lane_entries<T>(a0, a1, j, end, stride, P.col, w, [x](int32_t c) { return x[c]; });
                lds += P.n_cols;
            } else {
                const T* x = static_cast<const T*>(P.x) + ring_slot(t - P.delay, P.depth) * P.n_cols;
                if (KIND == AHIP_FUSE_MIX && kind == AHIP_FUSE_DENSE) {
                    for (uint32_t q = j; q < end; q += stride) a0.add(w[q] * x[q - beg]);
                } else {
                    lane_entries<T>(a0, a1, j, end, stride, P.col, w, [x](int32_t c) { return x[c]; });
                }
            }
            a0.join(a1);
            const T s = a0.reduce_rt(F.lane_shift);
#pragma unroll
            for (int k = 0; k < K; k++)
                if (P.sum == k) sum[k] += s;
        }
        if (in && (lane & (L - 1)) == 0)
#pragma unroll
            for (int k = 0; k < K; k++) sums[k][at] = sum[k];
    }
}

// Stages the rates of every projection, one after another, by `threads`
// threads of index tid.
template <typename T>
__device__ inline void stage_rates(const ahip_fuse_args& F, int64_t t, T* xs, int32_t tid, int32_t threads) {
    int32_t lds = 0;
    for (int32_t p = 0; p < F.n; p++) {
        const ahip_fuse_proj& P = F.p[p];
        const T* x = static_cast<const T*>(P.x) + ring_slot(t - P.delay, P.depth) * P.n_cols;
        constexpr int32_t kB = 8;
        for (int32_t k0 = tid; k0 < P.n_cols; k0 += kB * threads) {
            T v[kB];
#pragma unroll
            for (int u = 0; u < kB; u++) v[u] = x[min(k0 + u * threads, P.n_cols - 1)];
#pragma unroll
            for (int u = 0; u < kB; u++)
                if (k0 + u * threads < P.n_cols) xs[lds + k0 + u * threads] = v[u];
        }
        lds += P.n_cols;
    }
}

// new rate of neuron i into the population's rings
template <typename T>
__device__ inline void push_rate(const ahip_pop_args& a, int64_t t, int32_t i, T r) {
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (a.push_depth[k] > 0)
            static_cast<T*>(a.push_buf[k])[ring_slot(t, a.push_depth[k]) * (int64_t)a.size + i] = r;
}

}  // namespace ahip
