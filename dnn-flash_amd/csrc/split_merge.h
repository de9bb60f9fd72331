// Device code of the key split shared by the attention kernels: which splits
// of a query tile run, partial rows, and their merge inside the launch that
// writes them. Internal header, included by the HIP translation units.
#pragma once

#include "ofh_kernels.h"

namespace ofh {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr float kNegInf = -__builtin_huge_valf();

// s_waitcnt vmcnt(0): every vector-memory load issued so far has returned
// (and every store has completed: gfx9 counts both in vmcnt). Issued once
// before the tile loop, it tells the compiler's wait-count tracking that the
// Q fragments are resident on every path into the loop; without it the loop
// waits on them (and so on every load issued after them, i.e. the K/V
// prefetch) at each use.
__device__ __forceinline__ void wait_vm_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }

// ---------------------------------------------------------------------------
// Key split (FwdArgs::num_splits > 1). Query tile qt has steps(qt) K/V tile
// steps; splits [0, active(qt)) of it run, split s over steps
// [s*range, (s+1)*range), range = split_range(steps(qt)). With one active split, split 0 writes O
// directly. Otherwise every active split writes its unnormalised partial rows
// (O_s, m_s, l_s) and the rows are merged with the log-sum-exp rule of
// attention.cpp:661-674 applied across splits:
//   m* = max_s m_s,  O = sum_s 2^(m_s - m*) O_s / sum_s 2^(m_s - m*) l_s.
// Rows that saw no valid key in any split (l = 0) are written as 0.

// Steps per split of a query tile with `steps` K/V tile steps.
__device__ __forceinline__ int split_range(const FwdArgs& a, int steps) {
    return a.pair_split ? max(1, (steps + a.num_splits - 1) / a.num_splits) : a.split_tiles;
}
__device__ __forceinline__ int split_active(const FwdArgs& a, int steps) {
    const int range = split_range(a, steps);
    return max(1, min(a.num_splits, (steps + range - 1) / range));
}

// Folds partial (m2, l2, o2) into (m, l, o); maxima in log2 units.
__device__ __forceinline__ void lse_fold(float& m, float& l, f32x4& o, float m2, float l2, f32x4 o2) {
    const float mg = fmaxf(m, m2);
    const float mu = mg == kNegInf ? 0.0f : mg;
    const float w1 = __builtin_amdgcn_exp2f(m - mu), w2 = __builtin_amdgcn_exp2f(m2 - mu);  // 0 for -inf
    l = l * w1 + l2 * w2;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = o[t] * w1 + o2[t] * w2;
    m = mg;
}

// Partial rows merged inside the launch that writes them (split_counters set)
// are stored and loaded with agent-scope atomics: each access is coherent
// across the XCDs' L2 caches by itself, so no L2 writeback or invalidation
// (an agent-scope fence) is needed, which would cost every other workgroup on
// the XCD its cached K/V tiles. Partial rows merged by a second launch use
// plain accesses (the launch boundary makes them visible).
__device__ __forceinline__ void put_partial(float* p, float v, bool coherent) {
    if (coherent) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else *p = v;
}
__device__ __forceinline__ void put_partial4(float* p, f32x4 v, bool coherent) {
    if (coherent) {
#pragma unroll
        for (int t = 0; t < 4; ++t) __hip_atomic_store(p + t, v[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        *(f32x4*)p = v;
    }
}
template <bool COHERENT>
__device__ __forceinline__ float get_partial(const float* p) {
    if (COHERENT) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return *p;
}
template <bool COHERENT>
__device__ __forceinline__ f32x4 get_partial4(const float* p) {
    if (COHERENT) {
        f32x4 v;
#pragma unroll
        for (int t = 0; t < 4; ++t) v[t] = __hip_atomic_load(p + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return v;
    }
    return *(const f32x4*)p;
}

// Merges columns [4c, 4c+4) of partial row prow over splits s0, s0+sstep, ...
// below `active`, four splits per group so that their loads are in flight
// together; the running max is raised per group.
template <bool COHERENT>
__device__ __forceinline__ void merge_partials(const FwdArgs& a, int64_t prow, int c, int s0, int sstep,
                                               int active, float& m, float& l, f32x4& acc) {
    const int64_t stride = (int64_t)a.B * a.H * a.M;
    constexpr int G = 4;
    for (int s = s0; s < active; s += G * sstep) {
        float ms[G], ls[G];
        f32x4 os[G];
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const bool ok = s + j * sstep < active;
            const int64_t r = (int64_t)(ok ? s + j * sstep : s) * stride + prow;
            // (plain float loads: element 1 of a loaded u32x2 passed through
            // __builtin_bit_cast was read as element 0 by this compiler)
            ms[j] = ok ? get_partial<COHERENT>(a.part_ml + 2 * r) : kNegInf;
            ls[j] = get_partial<COHERENT>(a.part_ml + 2 * r + 1);
            os[j] = get_partial4<COHERENT>(a.part_o + r * a.Dv + 4 * c);
            if (!ok) os[j] = f32x4{0.f, 0.f, 0.f, 0.f};  // weight 0 must not meet an inf
        }
        float mg = m;
#pragma unroll
        for (int j = 0; j < G; ++j) mg = fmaxf(mg, ms[j]);
        const float mu = mg == kNegInf ? 0.0f : mg;
        const float keep = __builtin_amdgcn_exp2f(m - mu);  // 0 while m is -inf
        l *= keep;
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] *= keep;
#pragma unroll
        for (int j = 0; j < G; ++j) {
            const float w = __builtin_amdgcn_exp2f(ms[j] - mu);  // 0 for splits past `active`
            l += w * ls[j];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] += w * os[j][t];
        }
        m = mg;
    }
}

// Writes columns [4c, 4c+4) of O row `row` of head bh, normalised by l.
template <typename T>
__device__ __forceinline__ void store_merged(const FwdArgs& a, int bh, int row, int c, float l, f32x4 acc) {
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    const int b = bh / a.H, h = bh - b * a.H;
    const int64_t off = b * a.o_sb + h * a.o_sh + (int64_t)row * a.o_sm + 4 * c;
    if (sizeof(T) == 4 || a.out_f32) {
        *(f32x4*)((float*)a.o + off) = acc * inv;
    } else if constexpr (sizeof(T) == 2) {
        typedef T v4 __attribute__((ext_vector_type(4)));
        v4 val;
#pragma unroll
        for (int t = 0; t < 4; ++t) val[t] = (T)(acc[t] * inv);
        *(v4*)((T*)a.o + off) = val;
    }
}

// Counts this workgroup in its query tile's arrival counter once the partial
// rows of every thread are stored (agent-scope atomic stores, complete when
// vmcnt reaches 0); true in the workgroup that arrives last, to which the
// partial rows of all splits of the tile are then visible through agent-scope
// atomic loads. That workgroup sets the counter back to zero for the next
// call on the stream. Every thread calls it; `flag` is one int of LDS.
__device__ __forceinline__ bool split_arrive(unsigned* ctr, int active, int* flag) {
    __atomic_signal_fence(__ATOMIC_SEQ_CST);  // the partial-row stores stay above the wait
    wait_vm_loads();                          // vmcnt(0): this thread's stores have completed
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned prev = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = prev + 1 == (unsigned)active;
        if (last) __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = last ? 1 : 0;
    }
    __syncthreads();
    return *flag != 0;
}

// Merge of the `rows` rows from q0 of head bh by one workgroup of NTHREADS
// threads: a thread per (row, 4-column chunk); when there are fewer such
// items than threads (few rows), the splits are shared out over groups of
// threads whose results are folded through `red` (6 * NTHREADS floats of LDS).
template <typename T, int NTHREADS>
__device__ void merge_split_rows(const FwdArgs& a, int bh, int q0, int rows, int active, float* red) {
    const int chunks = a.Dv >> 2;
    const int items = rows * chunks;
    const int t = threadIdx.x;
    if (items >= NTHREADS) {
        for (int item = t; item < items; item += NTHREADS) {
            const int rr = item / chunks, c = item - rr * chunks;
            float m = kNegInf, l = 0.0f;
            f32x4 acc = {0.f, 0.f, 0.f, 0.f};
            merge_partials<true>(a, (int64_t)bh * a.M + q0 + rr, c, 0, 1, active, m, l, acc);
            store_merged<T>(a, bh, q0 + rr, c, l, acc);
        }
        return;
    }
    const int groups = min(active, NTHREADS / items);
    const int item = t % items, grp = t / items;
    const bool mine = grp < groups;
    const int rr = item / chunks, c = item - rr * chunks;
    float m = kNegInf, l = 0.0f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (mine) merge_partials<true>(a, (int64_t)bh * a.M + q0 + rr, c, grp, groups, active, m, l, acc);
    if (mine && grp > 0) {
        float* e = red + 6 * (grp * items + item);
        e[0] = m;
        e[1] = l;
#pragma unroll
        for (int j = 0; j < 4; ++j) e[2 + j] = acc[j];
    }
    __syncthreads();
    if (grp == 0) {
        for (int j = 1; j < groups; ++j) {
            const float* e = red + 6 * (j * items + item);
            lse_fold(m, l, acc, e[0], e[1], f32x4{e[2], e[3], e[4], e[5]});
        }
        store_merged<T>(a, bh, q0 + rr, c, l, acc);
    }
}

}  // namespace
}  // namespace ofh
