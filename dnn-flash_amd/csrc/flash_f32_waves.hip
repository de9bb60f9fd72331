// fp32 attention forward for mid-size calls: 32 query rows per workgroup, whose
// eight wavefronts take the block's 32-key tiles in turn (plain scale, causal or
// not, no mask, head dims up to 128).
//
// What bounds it: the fp32 matrix rate and the chain of tiles a wavefront walks.
// K and V come 64 columns at a time as whole 256-byte row pieces (16 lanes x 16
// bytes per row, four rows per load), the next block in flight while this one is
// multiplied, and pass through an LDS block of the wavefront's own that turns
// rows into operands: no barrier in the loop, no key split and no merge over
// workgroups. Rows of 64 + 4 floats keep both operand reads free of bank
// conflicts (K: 16 bytes of rows kappa(0..15); V: rows 8 apart in the halves;
// counted at H8 N1000 D64: 31 conflict cycles per wavefront in the whole kernel,
// beside 227 LDS instructions).
// Every wavefront keeps an online softmax state; the eight are folded in LDS.
// One block per CU (80 to 88 KB of LDS), two wavefronts per SIMD: H8 N1000 D64
// 47.7 -> 25.0 us (43 -> 82 TF of the 154 a large product reaches), causal
// H32 N768 D64 62.1 -> 37.4, H8 N1000 D128 66.1 -> 46.5.

#include "flash_wave32.h"
#include "ofh_kernels.h"

namespace ofh {
namespace {

constexpr int kF32Waves = kF32WavesThreads / 64;
constexpr int kF32Cols = 64;               // columns of K or V per staged block
constexpr int kF32Stride = kF32Cols + 4;   // floats per staged row

// NC: 64-column blocks of K, Q and V (head dims up to 64 NC).
template <int NC>
__global__ __launch_bounds__(kF32WavesThreads) void flash_fwd_f32_waves_kernel(FwdArgs a) {
    constexpr int QS = NC * kF32Cols + 4;
    __shared__ __attribute__((aligned(16))) float q_lds[32 * QS];
    __shared__ __attribute__((aligned(16))) float blocks[kF32Waves * 32 * kF32Stride];
    __shared__ float stat[2 * kF32Waves * 32];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, r = lane & 31;
    int bh, qt;
    map_work((int)blockIdx.x, a.B * a.H, a.num_q_tiles, a.causal, bh, qt);
    const int b = bh / a.H, h = bh - b * a.H;
    const float* Qp = (const float*)a.q + b * a.q_sb + h * a.q_sh;
    const float* Kp = (const float*)a.k + b * a.k_sb + h * a.k_sh;
    const float* Vp = (const float*)a.v + b * a.v_sb + h * a.v_sh;
    float* blk = blocks + wave * 32 * kF32Stride;
    const int q0 = qt * 32;
    const int qi = min(q0 + r, a.M - 1);  // rows past M are not stored
    const int lrow = lane >> 4, lcol = 4 * (lane & 15);  // this lane's row (of four) and columns of a load

    for (int row = threadIdx.x >> 4; row < 32; row += kF32WavesThreads / 16) {
        const float* src = Qp + (int64_t)min(q0 + row, a.M - 1) * a.q_sm;
#pragma unroll
        for (int d = 0; d < NC; ++d) {
            const int col = d * kF32Cols + lcol;
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            if (col < a.D) v = *(const f32x4*)(src + col);
            *(f32x4*)(q_lds + row * QS + col) = v;
        }
    }
    __syncthreads();

    const int kend = a.causal ? min(a.N, q0 + 32) : a.N;
    const int ntiles = (kend + 31) / 32;
    f32x4 reg[8];
    // Columns [64 c, 64 c + 64) of rows 32 t .. of K or V: chunks past the width
    // repeat the last one, rows past the end the last row.
    auto load = [&](const float* base, int64_t stride, int t, int c, int width) {
        const int k0 = 32 * t;
        const float* p = base + min(c * kF32Cols + lcol, width - 4);
        if (k0 + 32 <= a.N) {
            p += (int64_t)(k0 + lrow) * stride;
#pragma unroll
            for (int u = 0; u < 8; ++u) reg[u] = *(const f32x4*)(p + (int64_t)(4 * u) * stride);
        } else {
#pragma unroll
            for (int u = 0; u < 8; ++u) reg[u] = *(const f32x4*)(p + (int64_t)min(k0 + 4 * u + lrow, a.N - 1) * stride);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Staged with zeros in columns at or past `cols` of the block and in rows at or past `rows`.
    auto put = [&](int cols, int rows) {
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < 8; ++u)
            *(f32x4*)(blk + (4 * u + lrow) * kF32Stride + lcol) = lcol < cols && 4 * u + lrow < rows ? reg[u] : zero;
        __builtin_amdgcn_sched_barrier(0);
    };
    float m = kNegInf, l = 0.0f;
    f32x16 o[2 * NC];
#pragma unroll
    for (int db = 0; db < 2 * NC; ++db) o[db] = f32x16{};
    int t = wave;
    if (t < ntiles) load(Kp, a.k_sn, t, 0, a.D);
    for (; t < ntiles; t += kF32Waves) {
        const int k0 = 32 * t;
        f32x16 s = f32x16{};
#pragma unroll
        for (int d = 0; d < NC; ++d) {
            put(a.D - d * kF32Cols, 32);
            if (d + 1 < NC) load(Kp, a.k_sn, t, d + 1, a.D);
            else load(Vp, a.v_sn, t, 0, a.Dv);
            const float* kr = blk + kappa(r) * kF32Stride + 32 * g;
            const float* qr = q_lds + r * QS + d * kF32Cols + 32 * g;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const f32x4 kf = *(const f32x4*)(kr + 4 * i), qf = *(const f32x4*)(qr + 4 * i);
#pragma unroll
                for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j], qf[j], s, 0, 0, 0);
            }
        }
        // key acc_pos(e, g) of the tile is valid below `lim`
        const int lim = (a.causal ? min(a.N, qi + 1) : a.N) - k0;
        float mx = kNegInf;
        if (k0 + 32 <= a.N && (!a.causal || k0 + 31 <= q0)) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[e] *= a.scale_log2;
                mx = fmaxf(mx, s[e]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[e] = acc_pos(e, g) < lim ? s[e] * a.scale_log2 : kNegInf;
                mx = fmaxf(mx, s[e]);
            }
        }
        mx = half_swap_max(mx);
        if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {  // the running max rises for some row
            const float mn = fmaxf(m, mx);
            const float alpha = __builtin_amdgcn_exp2f(m - (mn == kNegInf ? 0.0f : mn));  // 0 while m is -inf
            m = mn;
            l *= alpha;
#pragma unroll
            for (int db = 0; db < 2 * NC; ++db) o[db] *= alpha;
        }
        const float mu = m == kNegInf ? 0.0f : m;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[e] = __builtin_amdgcn_exp2f(s[e] - mu);
            l += s[e];
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            put(kF32Cols, a.N - k0);
            if (c + 1 < NC) load(Vp, a.v_sn, t, c + 1, a.Dv);
            else if (t + kF32Waves < ntiles) load(Kp, a.k_sn, t + kF32Waves, 0, a.D);
            const float* vr = blk + 8 * g * kF32Stride + r;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float* vk = vr + acc_pos(e, 0) * kF32Stride;
                o[2 * c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vk[0], s[e], o[2 * c], 0, 0, 0);
                o[2 * c + 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vk[32], s[e], o[2 * c + 1], 0, 0, 0);
            }
        }
    }

    // Fold the wavefronts: O = sum_w 2^(m_w - m*) O_w / sum_w 2^(m_w - m*) l_w.
    l += __shfl_xor(l, 32);
    if (g == 0) {
        stat[wave * 32 + r] = m;
        stat[(kF32Waves + wave) * 32 + r] = l;
    }
    __syncthreads();
    float mg = kNegInf;
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) mg = fmaxf(mg, stat[w * 32 + r]);
    const float mu = mg == kNegInf ? 0.0f : mg;
    const float weight = __builtin_amdgcn_exp2f(m - mu);  // 0 for a wavefront without a valid key
    float lsum = 0.0f;
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w)
        lsum += __builtin_amdgcn_exp2f(stat[w * 32 + r] - mu) * stat[(kF32Waves + w) * 32 + r];
    const float inv = lsum > 0.0f ? 1.0f / lsum : 0.0f;  // rows without a valid key are written as 0
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        // O^T: this lane's query row r, columns 32 db + 8 (e >> 2) + 4 g + (e & 3)
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = o[2 * c + (x >> 2)][4 * (x & 3) + j] * (weight * inv);
            *(f32x4*)(blk + r * kF32Stride + 32 * (x >> 2) + 8 * (x & 3) + 4 * g) = v;
        }
        __syncthreads();
        const int row = (int)threadIdx.x >> 4, col = c * kF32Cols + lcol;
        static_assert(kF32WavesThreads / 16 == 32, "a thread per row and four columns");
        if (q0 + row < a.M && col < a.Dv) {
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < kF32Waves; ++w) sum += *(const f32x4*)(blocks + (w * 32 + row) * kF32Stride + lcol);
            *(f32x4*)((float*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)(q0 + row) * a.o_sm + col) = sum;
        }
        __syncthreads();
    }
}

}  // namespace

hipError_t launch_f32_waves(const FwdArgs& a, hipStream_t s) {
    if (a.D > 128 || a.Dv > 128 || a.mask != nullptr || a.num_splits != 1 || a.split_bm != 32) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((int64_t)a.B * a.H * a.num_q_tiles)), block(kF32WavesThreads);
    if (a.D <= 64 && a.Dv <= 64) hipLaunchKernelGGL(flash_fwd_f32_waves_kernel<1>, grid, block, 0, s, a);
    else hipLaunchKernelGGL(flash_fwd_f32_waves_kernel<2>, grid, block, 0, s, a);
    return hipGetLastError();
}

}  // namespace ofh
