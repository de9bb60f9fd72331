// Exact two-pass softmax attention for any head_dim and value_dim: the GPU
// counterpart of standard_attention (src/onednn_flash/attention.cpp:88-137 of
// the reference). Pass 1 finds the row max over valid keys; pass 2 recomputes
// the scores, forms p = exp(s - max), the denominator and sum_k p_k * V[k].
// Scores are never stored: they are recomputed rather than materialised. Used
// for OFH_ALGO_ROWWISE and for shapes the MFMA flash kernels do not take (head
// dims that are not a multiple of the 16-byte row chunk or above 256,
// unaligned rows).
//
// rowwise_fwd_kernel (head_dim and value_dim up to 256): 32 query rows per
// workgroup on the fp32 matrix cores. rowwise_wave_kernel (wider heads, and few
// rows per head against few keys): one wavefront per query row on the vector units.

#include "ofh_kernels.h"

namespace ofh {
namespace {

constexpr int kMaxD = 1024;     // rowwise_wave_kernel: its query row staged in LDS (fp32)
constexpr int kAccPerLane = 8;  // ... output columns per lane per pass-2 sweep (512 per sweep)

template <typename T>
__device__ __forceinline__ float to_f32(T x) {
    return (float)x;
}

__device__ __forceinline__ bool row_masked(const FwdArgs& a, int qi, int kj) {
    if (a.causal && kj > qi) return true;
    if (a.mask != nullptr) {
        const int qb = qi / a.mask_qbs, kb = kj / a.mask_kbs;
        if (qb >= a.mask_qb || kb >= a.mask_kb) return true;
        return a.mask[(int64_t)qb * a.mask_kb + kb] == 0;
    }
    return false;
}

template <typename T>
__device__ __forceinline__ float row_score(const FwdArgs& a, const float* qs, const T* krow,
                                           int qi, int kj, float slope, const float* bias_row) {
    float dot = 0.0f;
    for (int d = 0; d < a.D; ++d) dot += qs[d] * to_f32(krow[d]);
    float s = dot * a.scale;
    if (a.bias_kind == BIAS_ALIBI) s += slope * (float)(kj - qi);
    else if (a.bias_kind == BIAS_DENSE) s += bias_row[kj];
    if (a.softcap > 0.0f) s = a.softcap * tanhf(s / a.softcap);
    return s;
}

// Heads wider than rowwise_fwd_kernel takes, and calls that give its 32-row
// blocks little to do: a wavefront here costs a fraction of a block whose
// eight wavefronts stage 32 rows and 32 keys whatever is there (fp32 D50 B1024
// H64 M1 N16 377 us against 2672, one row of three keys 5.1 us against 11.2).
// What bounds it: the latency of the loads behind one another, one per key in
// pass 2. Lanes own keys during the score passes (each lane one key, the query row broadcast from LDS) and own output
// columns during accumulation (each of the 64 probabilities of a key chunk is
// broadcast with a scalar read-lane), so V reads are coalesced along the row.
template <typename T>
__global__ __launch_bounds__(64 * kRowsPerWorkgroup) void rowwise_wave_kernel(FwdArgs a) {
    __shared__ float qs_all[kRowsPerWorkgroup][kMaxD];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t row_id = (int64_t)blockIdx.x * kRowsPerWorkgroup + w;
    const bool valid = row_id < (int64_t)a.B * a.H * a.M;  // wave-uniform
    const int qi = valid ? (int)(row_id % a.M) : 0;
    const int bh = valid ? (int)(row_id / a.M) : 0;
    const int b = bh / a.H, h = bh - b * a.H;
    const T* Qp = (const T*)a.q + b * a.q_sb + h * a.q_sh + (int64_t)qi * a.q_sm;
    const T* Kp = (const T*)a.k + b * a.k_sb + h * a.k_sh;
    const T* Vp = (const T*)a.v + b * a.v_sb + h * a.v_sh;
    float* qs = qs_all[w];
    if (valid) {
        for (int d = lane; d < a.D; d += 64) qs[d] = to_f32(Qp[d]);
    }
    __syncthreads();
    if (!valid) return;

    const float slope = a.bias_kind == BIAS_ALIBI ? a.alibi[h] : 0.0f;
    const float* bias_row = a.bias_kind == BIAS_DENSE
                                ? a.bias + b * a.bias_sb + h * a.bias_sh + (int64_t)qi * a.bias_sm
                                : nullptr;

    // Pass 1: row max over valid keys.
    float mx = -__builtin_huge_valf();
    bool any = false;
    for (int k0 = 0; k0 < a.N; k0 += 64) {
        const int kj = k0 + lane;
        if (kj < a.N && !row_masked(a, qi, kj)) {
            const float s = row_score(a, qs, Kp + (int64_t)kj * a.k_sn, qi, kj, slope, bias_row);
            mx = fmaxf(mx, s);
            any = true;
        }
    }
    for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
    any = __any(any);

    // Pass 2, in sweeps of 64*kAccPerLane output columns. The probability of
    // key k0+jj is broadcast from lane jj with a scalar read-lane.
    for (int dv0 = 0; dv0 < a.Dv; dv0 += 64 * kAccPerLane) {
        float acc[kAccPerLane];
        for (int t = 0; t < kAccPerLane; ++t) acc[t] = 0.0f;
        float denom = 0.0f;
        if (any) {
            for (int k0 = 0; k0 < a.N; k0 += 64) {
                const int kj = k0 + lane;
                float p = 0.0f;
                if (kj < a.N && !row_masked(a, qi, kj)) {
                    const float s = row_score(a, qs, Kp + (int64_t)kj * a.k_sn, qi, kj, slope, bias_row);
                    p = expf(s - mx);
                }
                denom += p;
                const int kn = min(64, a.N - k0);
                for (int jj = 0; jj < kn; ++jj) {
                    const float pj = __builtin_bit_cast(
                        float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p), jj));
                    if (pj == 0.0f) continue;  // uniform
                    const T* vrow = Vp + (int64_t)(k0 + jj) * a.v_sn;
                    for (int t = 0; t < kAccPerLane; ++t) {
                        const int d = dv0 + lane + 64 * t;
                        if (d < a.Dv) acc[t] += pj * to_f32(vrow[d]);
                    }
                }
            }
        }
        for (int off = 32; off > 0; off >>= 1) denom += __shfl_xor(denom, off);
        const float inv = (any && denom > 0.0f) ? 1.0f / denom : 0.0f;
        for (int t = 0; t < kAccPerLane; ++t) {
            const int d = dv0 + lane + 64 * t;
            if (d >= a.Dv) continue;
            const float val = acc[t] * inv;
            const int64_t off = b * a.o_sb + h * a.o_sh + (int64_t)qi * a.o_sm + d;
            if (a.out_f32) ((float*)a.o)[off] = val;
            else ((T*)a.o)[off] = (T)val;
        }
    }
}

// ---------------------------------------------------------------------------
// 32 query rows per workgroup. Its NW wavefronts take the block's 32-key tiles
// in turn (tile t: wavefront t mod NW) and are independent until the end: the
// softmax is taken against the final row max (two passes), so their partial
// sums of p and p V only have to be added. Products run on
// v_mfma_f32_32x32x2_f32 as S^T = K Q^T and O^T = V^T P^T: a lane then holds 16
// scores of one query row, and those registers are the B operand of the second
// product (see flash_fwd_mfma.hip).
//
// What bounds it: the fp32 matrix rate (three products per pair, the scores
// being formed twice: fp32 non-causal B2 H8 N1024 D64 99 us, 65 TFLOP/s of such
// products, against 2657 us for a wavefront per row with its scalar loads and
// no reuse of K and V between rows; causal 61 against 1586, bf16 causal B2 H8
// N1000 D100 116 against 1462). K and V are read 64 columns at a time by one
// 4-byte (2-byte) load per lane and row, 64 consecutive columns of a row per
// instruction, so rows of any width, stride and alignment are read coalesced;
// the next 32x64 block is in flight while this one is multiplied, and goes
// through a wavefront-private LDS block that turns rows into operands (no
// barrier in the loops). Rows of 64 + 4 floats make both operand reads free of
// bank conflicts (K: 16 bytes of rows kappa(0..15); V: rows 8 apart in the lane
// halves).
//
// Keys that the causal rule or the mask hides from a row, and keys whose
// probability is zero, must not reach it through an inf or NaN in their V row:
// in a V block that holds one, such elements are multiplied as 0 and then
// added to the rows that give their key a non-zero probability
// (standard_attention skips masked keys, attention.cpp:126-131).
constexpr int kCols = 64;        // columns of K or V per staged block
constexpr int kColStride = kCols + 4;
// Wavefronts per workgroup, two on every SIMD: fp32 causal B2 H8 N1024 D64 61.5
// us against 67.3 with four (two workgroups per CU), B1 H4 N512 28.7 against
// 34.5, B1 H2 M1 N4096 170 against 217; non-causal B2 H8 N1024 98.9 against 96.3.
constexpr int kRowWaves = kRowBlockThreads / 64;


typedef float rw_f32x16 __attribute__((ext_vector_type(16)));
typedef float rw_f32x4 __attribute__((ext_vector_type(4)));

// Key within a 32-key tile held by accumulator register e of lane half g, and
// the A-operand row order that yields it.
__device__ __forceinline__ constexpr int rw_key(int e, int g) { return 16 * (e >> 3) + 8 * g + (e & 7); }
__device__ __forceinline__ int rw_kappa(int r) {
    return ((r >> 4) << 4) | (((r >> 2) & 1) << 3) | (((r >> 3) & 1) << 2) | (r & 3);
}

// NC: 64-column blocks of V (value_dim <= 64 NC).
template <typename T, int NW, int NC>
__global__ __launch_bounds__(64 * NW) void rowwise_fwd_kernel(FwdArgs a, int num_q_blocks) {
    extern __shared__ __attribute__((aligned(16))) float rw_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, r = lane & 31;
    const int nd = (a.D + kCols - 1) / kCols;
    const int qstride = nd * kCols + 4;
    float* q_lds = rw_lds;                                     // [32][qstride]
    float* blk = rw_lds + kRowBlock * qstride + wave * kRowBlock * kColStride;  // [32][kColStride]
    float* stat = rw_lds + kRowBlock * qstride + NW * kRowBlock * kColStride;   // [NW][32] and [NW][32]

    // Query blocks of a head on one XCD (workgroups go to the XCDs
    // round-robin). Causal blocks differ in length: they run longest first, in
    // every other head shortest first, so that a CU's workgroups add up alike.
    const int BH = a.B * a.H;
    int bh, qb;
    if ((BH & 7) == 0) {
        const int j = (int)(blockIdx.x >> 3), hl = j / num_q_blocks, t = j - hl * num_q_blocks;
        bh = hl * 8 + (int)(blockIdx.x & 7);
        qb = a.causal && (((BH >> 3) - 1 - hl) & 1) == 0 ? num_q_blocks - 1 - t : t;
    } else {
        bh = (int)(blockIdx.x % (unsigned)BH);
        qb = (int)(blockIdx.x / (unsigned)BH);
        if (a.causal) qb = num_q_blocks - 1 - qb;
    }
    const int b = bh / a.H, h = bh - b * a.H;
    const T* Qp = (const T*)a.q + b * a.q_sb + h * a.q_sh;
    const T* Kp = (const T*)a.k + b * a.k_sb + h * a.k_sh;
    const T* Vp = (const T*)a.v + b * a.v_sb + h * a.v_sh;
    const int q0 = qb * kRowBlock;
    const int qi = min(q0 + r, a.M - 1);  // this lane's query row (rows past M are not stored)

    for (int row = wave; row < kRowBlock; row += NW) {
        const T* src = Qp + (int64_t)min(q0 + row, a.M - 1) * a.q_sm;
        for (int d = lane; d < nd * kCols; d += 64) q_lds[row * qstride + d] = d < a.D ? to_f32(src[d]) : 0.0f;
    }
    __syncthreads();

    const float slope = a.bias_kind == BIAS_ALIBI ? a.alibi[h] : 0.0f;
    const float* bias_row =
        a.bias_kind == BIAS_DENSE ? a.bias + b * a.bias_sb + h * a.bias_sh + (int64_t)qi * a.bias_sm : nullptr;
    const int kend = a.causal ? (int)min((int64_t)a.N, (int64_t)q0 + kRowBlock) : a.N;
    const int ntiles = (int)(((int64_t)kend + kRowBlock - 1) / kRowBlock);

    // Bit e: key rw_key(e, g) of tile t is valid for this lane's row.
    auto valid_keys = [&](int t) {
        const int k0 = t * kRowBlock;
        const int lim = (a.causal ? min(a.N, qi + 1) : a.N) - k0;
        unsigned vm = 0;
#pragma unroll
        for (int e = 0; e < 16; ++e) vm |= (rw_key(e, g) < lim ? 1u : 0u) << e;
        if (a.mask != nullptr) {
            const int mq = qi / a.mask_qbs;
            if (mq >= a.mask_qb) return 0u;
            const uint8_t* mrow = a.mask + (int64_t)mq * a.mask_kb;
#pragma unroll 1
            for (int e = 0; e < 16; ++e) {
                const int mk = (k0 + rw_key(e, g)) / a.mask_kbs;
                const bool ok = mk < a.mask_kb && mrow[min(mk, a.mask_kb - 1)] != 0;
                vm &= ~((ok ? 0u : 1u) << e);
            }
        }
        return vm;
    };
    // Next tile of this wavefront from t on that holds a valid pair, with its validity bits.
    unsigned vm = 0;
    auto next_tile = [&](int t) {
        for (; t < ntiles; t += NW) {
            vm = valid_keys(t);
            if (__builtin_amdgcn_ballot_w64(vm != 0) != 0) break;
        }
        return t;
    };

    // 32 rows x 64 columns of K or V on their way through registers: lane = column.
    float reg[kRowBlock];
    auto load = [&](const T* base, int64_t stride, int t, int c0, int width) {
        const int k0 = t * kRowBlock;
        const T* p = base + (int64_t)k0 * stride + min(c0 + lane, width - 1);
#pragma unroll
        for (int u = 0; u < kRowBlock; ++u) {
            reg[u] = to_f32(*p);
            p += a.N - k0 > u + 1 ? stride : 0;  // rows past the end repeat the last one
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto put = [&](bool zero) {
#pragma unroll
        for (int u = 0; u < kRowBlock; ++u) blk[u * kColStride + lane] = zero ? 0.0f : reg[u];
        __builtin_amdgcn_sched_barrier(0);
    };
    // Scores of tile t (its first K block is in `reg`), modified, in s.
    rw_f32x16 s;
    auto scores = [&](int t, auto&& prefetch_next) {
        s = rw_f32x16{};
        for (int d = 0; d < nd; ++d) {
            put(d * kCols + lane >= a.D);  // Q is zero there, K must be finite
            if (d + 1 < nd) load(Kp, a.k_sn, t, (d + 1) * kCols, a.D);
            else prefetch_next();
            const float* kr = blk + rw_kappa(r) * kColStride + 32 * g;
            const float* qr = q_lds + r * qstride + d * kCols + 32 * g;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const rw_f32x4 kf = *(const rw_f32x4*)(kr + 4 * i), qf = *(const rw_f32x4*)(qr + 4 * i);
#pragma unroll
                for (int j = 0; j < 4; ++j) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[j], qf[j], s, 0, 0, 0);
            }
        }
        const int k0 = t * kRowBlock;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] *= a.scale;
        if (a.bias_kind == BIAS_ALIBI) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] += slope * (float)(k0 + rw_key(e, g) - qi);
        } else if (a.bias_kind == BIAS_DENSE) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] += bias_row[min(k0 + rw_key(e, g), a.N - 1)];
        }
        if (a.softcap > 0.0f) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[e] = a.softcap * tanhf(s[e] / a.softcap);
                __builtin_amdgcn_sched_barrier(0);  // one at a time: sixteen at once would spill
            }
        }
    };

    // Pass 1: row max over valid keys.
    const float neg_inf = -__builtin_huge_valf();
    float mx = neg_inf;
    unsigned seen = 0;
    int t = next_tile(wave);
    if (t < ntiles) load(Kp, a.k_sn, t, 0, a.D);
    while (t < ntiles) {
        const unsigned cur = vm;
        const int tn = next_tile(t + NW);
        scores(t, [&] { if (tn < ntiles) load(Kp, a.k_sn, tn, 0, a.D); });
        seen |= cur;
#pragma unroll
        for (int e = 0; e < 16; ++e) mx = (cur >> e) & 1u ? fmaxf(mx, s[e]) : mx;
        t = tn;
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    seen |= __shfl_xor(seen, 32);
    if (g == 0) {
        stat[wave * 32 + r] = mx;
        stat[(NW + wave) * 32 + r] = seen != 0 ? 1.0f : 0.0f;
    }
    __syncthreads();
    float any = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        mx = fmaxf(mx, stat[w * 32 + r]);
        any = fmaxf(any, stat[(NW + w) * 32 + r]);
    }
    __syncthreads();  // `stat` is reused

    // Pass 2: probabilities against the final max, their sum and P V.
    rw_f32x16 o[2 * NC];
#pragma unroll
    for (int db = 0; db < 2 * NC; ++db) o[db] = rw_f32x16{};
    float l = 0.0f;
    t = next_tile(wave);
    if (t < ntiles) load(Kp, a.k_sn, t, 0, a.D);
    while (t < ntiles) {
        const unsigned cur = vm;
        scores(t, [&] { load(Vp, a.v_sn, t, 0, a.Dv); });
        const int tn = next_tile(t + NW);
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            s[e] = (cur >> e) & 1u ? expf(s[e] - mx) : 0.0f;
            l += s[e];
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float fin = 0.0f;  // NaN when the block holds an inf or NaN
#pragma unroll
            for (int u = 0; u < kRowBlock; ++u) fin = __builtin_fmaf(reg[u], 0.0f, fin);
            const float* vr = blk + 8 * g * kColStride + r;
            if (__builtin_amdgcn_ballot_w64(!(fin == 0.0f)) != 0) {
                // +inf, -inf and NaN elements: how many keys of non-zero
                // probability meet one, per output element; then as 0 below
#pragma unroll 1
                for (int cls = 0; cls < 3; ++cls) {
                    const float val = cls == 0 ? -neg_inf : cls == 1 ? neg_inf : __builtin_nanf("");
#pragma unroll
                    for (int u = 0; u < kRowBlock; ++u)
                        blk[u * kColStride + lane] = (cls == 2 ? reg[u] != reg[u] : reg[u] == val) ? 1.0f : 0.0f;
#pragma unroll
                    for (int db = 0; db < 2; ++db) {
                        rw_f32x16 hits = rw_f32x16{};
#pragma unroll
                        for (int e = 0; e < 16; ++e)
                            hits = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[rw_key(e, 0) * kColStride + 32 * db],
                                                                        s[e] != 0.0f ? 1.0f : 0.0f, hits, 0, 0, 0);
#pragma unroll
                        for (int e = 0; e < 16; ++e) o[2 * c + db][e] += hits[e] > 0.0f ? val : 0.0f;
                    }
                }
#pragma unroll
                for (int u = 0; u < kRowBlock; ++u) reg[u] = __builtin_fabsf(reg[u]) < -neg_inf ? reg[u] : 0.0f;
            }
            put(false);
            if (c + 1 < NC) load(Vp, a.v_sn, t, (c + 1) * kCols, a.Dv);
            else if (tn < ntiles) load(Kp, a.k_sn, tn, 0, a.D);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float* vk = vr + rw_key(e, 0) * kColStride;
                o[2 * c] = __builtin_amdgcn_mfma_f32_32x32x2f32(vk[0], s[e], o[2 * c], 0, 0, 0);
                o[2 * c + 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(vk[32], s[e], o[2 * c + 1], 0, 0, 0);
            }
        }
        t = tn;
    }

    // Sum over the wavefronts, normalise, store.
    l += __shfl_xor(l, 32);
    if (g == 0) stat[wave * 32 + r] = l;
    __syncthreads();
    if (wave == 0 && g == 0) {
        float sum = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) sum += stat[w * 32 + r];
        stat[NW * 32 + r] = any > 0.0f && sum > 0.0f ? 1.0f / sum : 0.0f;
    }
    const int64_t obase = b * a.o_sb + h * a.o_sh;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        // O^T: this lane's query row r, columns 32 db + 8 (e >> 2) + 4 g + (e & 3)
#pragma unroll
        for (int x = 0; x < 8; ++x) {
            rw_f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = o[2 * c + (x >> 2)][4 * (x & 3) + j];
            *(rw_f32x4*)(blk + r * kColStride + 32 * (x >> 2) + 8 * (x & 3) + 4 * g) = v;
        }
        __syncthreads();
        const float* all = rw_lds + kRowBlock * qstride;
        const int col = c * kCols + lane;
        if (col < a.Dv) {
            for (int row = wave; row < kRowBlock && q0 + row < a.M; row += NW) {
                float sum = 0.0f;
#pragma unroll
                for (int w = 0; w < NW; ++w) sum += all[(w * kRowBlock + row) * kColStride + lane];
                const float val = sum * stat[NW * 32 + row];
                const int64_t off = obase + (int64_t)(q0 + row) * a.o_sm + col;
                if (a.out_f32) ((float*)a.o)[off] = val;
                else ((T*)a.o)[off] = (T)val;
            }
        }
        __syncthreads();
    }
}

template <typename T, int NW, int NC>
hipError_t launch_row_blocks(const FwdArgs& a, hipStream_t s) {
    const int nqb = (a.M + kRowBlock - 1) / kRowBlock;
    const int nd = (a.D + kCols - 1) / kCols;
    const size_t lds = sizeof(float) * (kRowBlock * (nd * kCols + 4) + NW * kRowBlock * kColStride + 2 * NW * 32);
    hipLaunchKernelGGL((rowwise_fwd_kernel<T, NW, NC>), dim3((unsigned)((int64_t)a.B * a.H * nqb)), dim3(64 * NW), lds, s,
                       a, nqb);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_rowwise_t(const FwdArgs& a, hipStream_t s) {
    if (a.split_bm == kRowBlock) {
        if (a.D > kRowBlockMaxDim || a.Dv > kRowBlockMaxDim) return hipErrorInvalidValue;
        constexpr int NW = kRowWaves;
        if (a.Dv <= 64) return launch_row_blocks<T, NW, 1>(a, s);
        if (a.Dv <= 128) return launch_row_blocks<T, NW, 2>(a, s);
        return launch_row_blocks<T, NW, 4>(a, s);
    }
    const int64_t rows = (int64_t)a.B * a.H * a.M;
    hipLaunchKernelGGL(rowwise_wave_kernel<T>, dim3((unsigned)((rows + kRowsPerWorkgroup - 1) / kRowsPerWorkgroup)),
                       dim3(64 * kRowsPerWorkgroup), 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_rowwise(const FwdArgs& a, int dtype, hipStream_t s) {
    if (a.D > kMaxD) return hipErrorInvalidValue;
    if ((int64_t)a.B * a.H * a.M <= 0) return hipSuccess;
    switch (dtype) {
        case DT_F32: return launch_rowwise_t<float>(a, s);
        case DT_BF16: return launch_rowwise_t<__bf16>(a, s);
        case DT_F16: return launch_rowwise_t<_Float16>(a, s);
        default: return hipErrorInvalidValue;
    }
}

// ---------------------------------------------------------------------------
// Block-mask tile lists: for each query tile of the flash kernel, the ordered
// list of key tiles that hold at least one allowed (query, key) pair. Each
// entry also says, per 32-row slice of the query tile (one wavefront of the
// attention kernel), whether the slice has an allowed pair at all (else that
// wavefront skips the tile) and whether the mask allows all of its pairs
// (else it masks element-wise). Built before the attention launch, so skipped
// tiles issue no loads at all. One workgroup of four wavefronts per query
// tile, 256 key tiles per round; the list is compacted in key order with a
// per-wavefront ballot and a prefix over the wavefronts' counts.
namespace {

constexpr int kListWaves = 4;

__global__ __launch_bounds__(64 * kListWaves) void tile_list_kernel(TileListArgs a) {
    const int qt = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ int wave_counts[kListWaves];
    const int q0 = qt * a.block_m;
    const int slices = a.block_m / 32;
    int count = 0;
    for (int base = 0; base < a.num_k_tiles; base += 64 * kListWaves) {
        const int kt = base + tid;
        unsigned any_bits = 0, full_bits = 0;
        if (kt < a.num_k_tiles) {
            const int k0 = kt * a.block_n;
            const int k1 = min(a.N, k0 + a.block_n);
            for (int w = 0; w < slices; ++w) {
                const int s0 = q0 + 32 * w, s1 = min(a.M, s0 + 32);
                if (s0 >= s1) continue;
                bool any, all;
                classify_mask_slice(a.mask, a.mask_qbs, a.mask_kbs, a.mask_qb, a.mask_kb, a.causal, s0, s1,
                                    k0, k1, any, all);
                any_bits |= (any ? 1u : 0u) << w;
                full_bits |= (all ? 1u : 0u) << w;
            }
        }
        const unsigned long long bal = __ballot(any_bits != 0);
        if (lane == 0) wave_counts[wave] = __popcll(bal);
        __syncthreads();
        int before = count, total = count;
        for (int w = 0; w < kListWaves; ++w) {
            before += w < wave ? wave_counts[w] : 0;
            total += wave_counts[w];
        }
        if (any_bits != 0)
            a.entries[(int64_t)qt * a.num_k_tiles + before + __popcll(bal & ((1ull << lane) - 1ull))] =
                list_entry(kt, any_bits, full_bits);
        __syncthreads();  // wave_counts is rewritten in the next round
        count = total;
    }
    if (tid == 0) a.counts[qt] = count;
}

}  // namespace

hipError_t launch_tile_lists(const TileListArgs& a, hipStream_t s) {
    if (a.num_q_tiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(tile_list_kernel, dim3(a.num_q_tiles), dim3(64 * kListWaves), 0, s, a);
    return hipGetLastError();
}

}  // namespace ofh
