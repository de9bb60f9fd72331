// Attention forward for calls with a few query rows against many keys
// (decoding): up to decode_max_rows() rows of every head, plain scale, no mask.
//
// What bounds it: reading K and V once. The matrix-core kernels give a
// workgroup 32 to 256 query rows and stage K and V through LDS, so on such
// calls all but one of their wavefronts' matrix work is padding and the
// staging's barriers hold the loads back. Here every wavefront streams keys of
// its own straight into registers: a K or V row is one 16-byte load per lane
// over LPR lanes (64 / LPR rows per instruction, U instructions per group), the
// next group's K rows are requested before this group's scores are formed, and
// the products run on the vector units, whose rate at these row counts is a
// multiple of what memory delivers. Measured against the matrix-core kernels:
// fp32 B16 H16 M1 N4096 D64 300 -> 90 us (6.0 TB/s of K and V), B1 H8 M1 N32768
// D128 81 -> 45 us; bf16 B1 H8 M1 N32768 D128 30.4 -> 26.5 us (5.1 TB/s, the
// merge of 32 splits included), B1 H8 M1 N1000 10.9 -> 7.5 us. Non-temporal
// loads changed nothing.
//
// A lane group (the LPR lanes of a row) keeps its own running max, sum and
// output columns over the keys it sees, so the loop has no exchange between
// lane groups beyond the dot product's sum over the row's lanes. The states of
// the lane groups are folded with lane exchanges at the end, those of the
// wavefronts in LDS, and those of a key split by split_merge.h. Probabilities
// stay in fp32.

#include "ofh_kernels.h"
#include "split_merge.h"

namespace ofh {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
    const int y = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, true);
    return x + __builtin_bit_cast(float, y);
}

// Sum over the LPR lanes that hold a row, in every one of them.
template <int LPR>
__device__ __forceinline__ float row_sum(float x) {
    x = dpp_add<0xB1>(x);                      // lanes 1 apart
    x = dpp_add<0x4E>(x);                      // 2 apart
    if (LPR >= 8) x = dpp_add<0x141>(x);       // the other four of eight (mirrored)
    if (LPR >= 16) x = dpp_add<0x140>(x);      // the other eight of sixteen
    if (LPR >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, x),
                                                        __builtin_bit_cast(unsigned, x), false, false);
        x = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
    }
    if (LPR >= 64) {
        const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x),
                                                        __builtin_bit_cast(unsigned, x), false, false);
        x = __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
    }
    return x;
}

// The 16-byte chunk of a row: dot product with the query's chunk, and its
// elements in fp32.
template <typename T>
struct Chunk;
template <>
struct Chunk<float> {
    static constexpr int N = 4;
    static __device__ __forceinline__ float dot(u32x4 k, u32x4 q) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            s = __builtin_fmaf(__builtin_bit_cast(float, (unsigned)k[i]), __builtin_bit_cast(float, (unsigned)q[i]), s);
        return s;
    }
    static __device__ __forceinline__ float at(u32x4 v, int e) { return __builtin_bit_cast(float, (unsigned)v[e]); }
};
template <>
struct Chunk<__bf16> {
    static constexpr int N = 8;
    static __device__ __forceinline__ float dot(u32x4 k, u32x4 q) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            s = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, (unsigned)k[i]),
                                                __builtin_bit_cast(bf16x2, (unsigned)q[i]), s, false);
        return s;
    }
    static __device__ __forceinline__ float at(u32x4 v, int e) {
        const unsigned u = v[e >> 1];
        return __builtin_bit_cast(float, (e & 1) != 0 ? u & 0xffff0000u : u << 16);
    }
};
template <>
struct Chunk<_Float16> {
    static constexpr int N = 8;
    static __device__ __forceinline__ float dot(u32x4 k, u32x4 q) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            s = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, (unsigned)k[i]),
                                       __builtin_bit_cast(f16x2, (unsigned)q[i]), s, false);
        return s;
    }
    static __device__ __forceinline__ float at(u32x4 v, int e) {
        return (float)__builtin_bit_cast(f16x2, (unsigned)v[e >> 1])[e & 1];
    }
};

// LPR: lanes per K or V row (16 bytes each). MQ: query rows held (M <= MQ). FULL:
// a K row fills its lanes (the select that others need costs 0.3 % at one row, 3 % at
// eight: fp32 B4 H64 M8 N4096 D64 114.0 us, without it 110.4).
template <typename T, int LPR, int MQ, bool FULL>
__global__ __launch_bounds__(kDecodeThreads, 2) void flash_fwd_decode_kernel(FwdArgs a) {
    using C = Chunk<T>;
    constexpr int W = kDecodeThreads / 64;
    constexpr int RPI = 64 / LPR;                      // rows per load instruction
    constexpr int U = kDecodeLoads;                    // load instructions per group
    constexpr int G = U * RPI;                         // keys per wavefront group
    constexpr int COLS = LPR * C::N;
    constexpr int kFold = W * MQ * (COLS + 2);
    constexpr int kMerge = 6 * kDecodeThreads + 1;     // merge_split_rows and its flag
    __shared__ __attribute__((aligned(16))) float red[kFold > kMerge ? kFold : kMerge];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sub = lane / LPR, c = lane % LPR;
    const int BH = a.B * a.H;
    const int split = (int)(blockIdx.x / (unsigned)BH), bh = (int)(blockIdx.x % (unsigned)BH);
    const int b = bh / a.H, h = bh - b * a.H;
    const int steps = (a.N + W * G - 1) / (W * G);
    const int active = split_active(a, steps);
    if (split >= active) return;  // uniform over the workgroup
    const int64_t range = (int64_t)split_range(a, steps) * (W * G);
    const int ks = (int)(split * range);
    const int ke = (int)min((int64_t)a.N, ks + range);

    // Lanes at or past the row's real width repeat its last chunk. Their K must not
    // reach the score (an infinity there would be counted twice, as NaN against a
    // zero query), V fills columns that are never stored.
    const bool in_row = FULL || C::N * c < a.D;
    const T* Kp = (const T*)a.k + b * a.k_sb + h * a.k_sh + C::N * min(c, a.D / C::N - 1);
    const T* Vp = (const T*)a.v + b * a.v_sb + h * a.v_sh + C::N * min(c, a.Dv / C::N - 1);
    u32x4 q[MQ];
#pragma unroll
    for (int i = 0; i < MQ; ++i) {
        q[i] = u32x4{0u, 0u, 0u, 0u};
        if (in_row)
            q[i] = *(const u32x4*)((const T*)a.q + b * a.q_sb + h * a.q_sh + (int64_t)min(i, a.M - 1) * a.q_sm + C::N * c);
    }
    float m[MQ], l[MQ], o[MQ][C::N];
#pragma unroll
    for (int i = 0; i < MQ; ++i) {
        m[i] = kNegInf;
        l[i] = 0.0f;
#pragma unroll
        for (int e = 0; e < C::N; ++e) o[i][e] = 0.0f;
    }

    // Rows [k0, k0 + G) of K or V: instruction u holds row k0 + u RPI + sub.
    // Rows past the range repeat its last one.
    auto load = [&](u32x4 (&x)[U], const T* base, int64_t stride, int k0) {
        if (k0 + G <= ke) {
            const T* p = base + (int64_t)(k0 + sub) * stride;
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = *(const u32x4*)(p + u * RPI * stride);
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u)
                x[u] = *(const u32x4*)(base + (int64_t)min(k0 + u * RPI + sub, ke - 1) * stride);
        }
    };
    u32x4 kc[U], kn[U], v[U];
    int k0 = ks + wave * G;
    if (k0 < ke) load(kc, Kp, a.k_sn, k0);
    for (; k0 < ke; k0 += W * G) {
        load(v, Vp, a.v_sn, k0);
        if (k0 + W * G < ke) load(kn, Kp, a.k_sn, k0 + W * G);
        const bool whole = k0 + G <= ke;
        if (!whole) {
            // keys past the range: probability 0, and no inf or NaN to meet it
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (k0 + u * RPI + sub >= ke) v[u] = u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < MQ; ++i) {
            float s[U];
            float mx = m[i];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                s[u] = row_sum<LPR>(in_row ? C::dot(kc[u], q[i]) : 0.0f) * a.scale_log2;
                if (!whole && k0 + u * RPI + sub >= ke) s[u] = kNegInf;
                mx = fmaxf(mx, s[u]);
            }
            const float mu = mx == kNegInf ? 0.0f : mx;
            const float alpha = __builtin_amdgcn_exp2f(m[i] - mu);  // 0 while m is -inf
            m[i] = mx;
            l[i] *= alpha;
#pragma unroll
            for (int e = 0; e < C::N; ++e) o[i][e] *= alpha;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const float p = __builtin_amdgcn_exp2f(s[u] - mu);
                l[i] += p;
#pragma unroll
                for (int e = 0; e < C::N; ++e) o[i][e] = __builtin_fmaf(p, C::at(v[u], e), o[i][e]);
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) kc[u] = kn[u];
    }

    // Fold the lane groups of the wavefront, then the wavefronts.
    float* fold_ml = red + W * MQ * COLS;
#pragma unroll
    for (int i = 0; i < MQ; ++i) {
#pragma unroll
        for (int off = LPR; off < 64; off <<= 1) {
            const float m2 = __shfl_xor(m[i], off), l2 = __shfl_xor(l[i], off);
            const float mg = fmaxf(m[i], m2);
            const float mu = mg == kNegInf ? 0.0f : mg;
            const float w1 = __builtin_amdgcn_exp2f(m[i] - mu), w2 = __builtin_amdgcn_exp2f(m2 - mu);
            l[i] = l[i] * w1 + l2 * w2;
#pragma unroll
            for (int e = 0; e < C::N; ++e) o[i][e] = o[i][e] * w1 + __shfl_xor(o[i][e], off) * w2;
            m[i] = mg;
        }
        if (sub == 0) {
            float* dst = red + (wave * MQ + i) * COLS + C::N * c;
#pragma unroll
            for (int e = 0; e < C::N; e += 4) *(f32x4*)(dst + e) = f32x4{o[i][e], o[i][e + 1], o[i][e + 2], o[i][e + 3]};
            if (c == 0) {
                fold_ml[2 * (wave * MQ + i)] = m[i];
                fold_ml[2 * (wave * MQ + i) + 1] = l[i];
            }
        }
    }
    __syncthreads();
    const int chunks = a.Dv >> 2;
    const int row = (int)threadIdx.x / chunks, ch = (int)threadIdx.x - row * chunks;
    static_assert(MQ * (COLS / 4) <= kDecodeThreads, "a thread per row and four columns");
    if (row < a.M) {
        float mg = kNegInf, lg = 0.0f;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < W; ++w) mg = fmaxf(mg, fold_ml[2 * (w * MQ + row)]);
        const float mu = mg == kNegInf ? 0.0f : mg;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const float ww = __builtin_amdgcn_exp2f(fold_ml[2 * (w * MQ + row)] - mu);
            lg += ww * fold_ml[2 * (w * MQ + row) + 1];
            acc += ww * *(const f32x4*)(red + (w * MQ + row) * COLS + 4 * ch);
        }
        if (active <= 1) {
            store_merged<T>(a, bh, row, ch, lg, acc);
        } else {
            const int64_t prow = ((int64_t)split * BH + bh) * a.M + row;
            const bool coh = a.split_counters != nullptr;
            put_partial4(a.part_o + prow * a.Dv + 4 * ch, acc, coh);
            if (ch == 0) {
                put_partial(a.part_ml + 2 * prow, mg, coh);
                put_partial(a.part_ml + 2 * prow + 1, lg, coh);
            }
        }
    }
    if (active <= 1 || a.split_counters == nullptr) return;  // uniform
    __syncthreads();  // `red` is reused
    if (split_arrive(a.split_counters + bh, active, (int*)(red + 6 * kDecodeThreads)))
        merge_split_rows<T, kDecodeThreads>(a, bh, 0, a.M, active, red);
}

template <typename T, int LPR, int MQ>
void launch_held(const FwdArgs& a, hipStream_t s) {
    const dim3 grid((unsigned)((int64_t)a.B * a.H * a.num_splits)), block(kDecodeThreads);
    if (a.D == LPR * Chunk<T>::N) hipLaunchKernelGGL((flash_fwd_decode_kernel<T, LPR, MQ, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((flash_fwd_decode_kernel<T, LPR, MQ, false>), grid, block, 0, s, a);
}

template <typename T, int LPR>
hipError_t launch_rows(const FwdArgs& a, hipStream_t s) {
    if (a.M <= 1) launch_held<T, LPR, 1>(a, s);
    else if (a.M <= 2) launch_held<T, LPR, 2>(a, s);
    else if constexpr (sizeof(T) == 4) {
        if (a.M <= 4) launch_held<T, LPR, 4>(a, s);
        else launch_held<T, LPR, 8>(a, s);
    }
    return hipGetLastError();
}

template <typename T>
hipError_t launch_width(const FwdArgs& a, int lanes, hipStream_t s) {
    if (lanes == 8) return launch_rows<T, 8>(a, s);
    if (lanes == 16) return launch_rows<T, 16>(a, s);
    if constexpr (sizeof(T) == 4) {
        if (lanes == 32) return launch_rows<T, 32>(a, s);
        if (lanes == 64) return launch_rows<T, 64>(a, s);
    }
    return hipErrorInvalidValue;
}

}  // namespace

hipError_t launch_decode(const FwdArgs& a, int dtype, hipStream_t s) {
    const int lanes = decode_row_lanes(dtype, a.D, a.Dv);
    if (a.M > decode_max_rows(dtype, a.D, a.Dv) || a.split_bn != decode_step_keys(dtype, a.D, a.Dv) || a.num_q_tiles != 1)
        return hipErrorInvalidValue;
    switch (dtype) {
        case DT_F32: return launch_width<float>(a, lanes, s);
        case DT_BF16: return launch_width<__bf16>(a, lanes, s);
        case DT_F16: return launch_width<_Float16>(a, lanes, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ofh
