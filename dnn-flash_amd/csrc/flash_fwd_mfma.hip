// Flash-style attention forward on gfx950 matrix cores.
//
// Replaces the CPU loop nest of flash_attention_qk_pv_tile_ws
// (src/onednn_flash/attention.cpp:486-695 of the reference) and its batched
// driver (src/onednn_flash/batched_attention.cpp:9-49): one workgroup owns a
// query block of one (batch, head) (256 rows for bf16/fp16, 128 with a
// block mask or for fp32), each wavefront 32 of its rows; K/V stream through
// LDS in tiles of 64 or 128 keys; QK^T and PV run on MFMA; the
// online-softmax recurrence (running max, rescaled running sum, rescaled
// accumulator, attention.cpp:628-673) lives in registers; the N x N score
// matrix is never formed.
//
// Layout trick. Scores are computed transposed, S^T = K * Q^T, with K as the
// MFMA A operand and Q as the B operand. In the 32x32 accumulator layout lane
// l then holds 16 scores of ONE query (column l%32), so the row max, the row
// sum and the accumulator rescale are per-lane scalars, and the only
// cross-lane step per tile is one exchange between the two 32-lane halves
// for the max. The output is accumulated transposed as well, O^T = V^T * P^T:
// the B operand P^T is exactly the lane's own probabilities (no shuffle). In
// the 16-bit kernels the V^T A-operand fragments come from the row-major V
// tile in LDS through the transposing ds_read_b64_tr_b16; the fp32 kernel
// reads V row-major (one element per lane and operand).
//
// The accumulator row r = 8i + 4g + j (lane half g = l/32, register 4i+j)
// is fed from A-operand row r, and A rows are permuted by kappa(r) =
// 16(i>>1) + 8g + 4(i&1) + j. With that permutation, registers [8c, 8c+8) of
// lane half g hold 8 consecutive positions 16c + 8g + t, which is what the
// next MFMA wants in a lane (k-slots 8g..8g+7 of a 16-wide chunk), and what
// a 16-byte store of the output wants.

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#include "flash_wave32.h"
#include "ofh_kernels.h"
#include "split_merge.h"

namespace ofh {
namespace {

// masked_out (attention.cpp:54-62) plus the key-range bound of a ragged last tile.
__device__ __forceinline__ bool elem_masked(const FwdArgs& a, int qi, int kj) {
    if (kj >= a.N) return true;
    if (a.causal && kj > qi) return true;
    if (a.mask != nullptr) {
        const int qb = qi / a.mask_qbs, kb = kj / a.mask_kbs;
        if (qb >= a.mask_qb || kb >= a.mask_kb) return true;
        return a.mask[(int64_t)qb * a.mask_kb + kb] == 0;
    }
    return false;
}

// tanh(y) = 1 - 2 / (exp(2y) + 1): saturates to +-1 for large |y| (exp2 -> inf / 0).
__device__ __forceinline__ float tanh_exp(float y) {
    const float e = __builtin_amdgcn_exp2f(y * (2.0f * kLog2e));
    return 1.0f - 2.0f * __builtin_amdgcn_rcpf(e + 1.0f);
}

// Scale, additive bias, soft-cap; result in log2 units for exp2.
__device__ __forceinline__ float general_score(const FwdArgs& a, float s, int qi, int kj,
                                               float slope, const float* bias_row) {
    float t = s * a.scale;
    if (a.bias_kind == BIAS_ALIBI) {
        t += slope * (float)(kj - qi);
    } else if (a.bias_kind == BIAS_DENSE) {
        t += bias_row[kj];
    }
    if (a.softcap > 0.0f) t = a.softcap * tanh_exp(t * a.inv_softcap);
    return t * kLog2e;
}

// One K/V tile of online softmax on the 32x32 accumulator blocks `s` (NB
// blocks of 32 keys), in place: raw dot products in, probabilities out.
// Returns alpha, the factor the accumulator must be rescaled by.
template <int NB, bool GENERAL>
__device__ __forceinline__ float online_softmax_tile(const FwdArgs& a, f32x16 (&s)[NB], bool need_mask,
                                                     int my_q, int k0, int g, float slope,
                                                     const float* bias_row, float& m_run,
                                                     float& l_run) {
    float mx = kNegInf;
    if (!GENERAL && !need_mask) {
#pragma unroll
        for (int sb = 0; sb < NB; ++sb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                s[sb][e] *= a.scale_log2;
                mx = fmaxf(mx, s[sb][e]);
            }
        }
    } else {
        const bool row_out = GENERAL && my_q >= a.M;
#pragma unroll
        for (int sb = 0; sb < NB; ++sb) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int kj = k0 + 32 * sb + acc_pos(e, g);
                const bool msk = row_out || (need_mask && elem_masked(a, my_q, kj));
                float x = kNegInf;
                if (!msk) {
                    x = GENERAL ? general_score(a, s[sb][e], my_q, kj, slope, bias_row)
                                : s[sb][e] * a.scale_log2;
                }
                s[sb][e] = x;
                mx = fmaxf(mx, x);
            }
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == kNegInf) ? 0.0f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    float lsum = 0.0f;
#pragma unroll
    for (int sb = 0; sb < NB; ++sb) {
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            const float p = __builtin_amdgcn_exp2f(s[sb][e] - m_use);
            s[sb][e] = p;
            lsum += p;
        }
    }
    l_run = l_run * alpha + lsum;
    return alpha;
}

// Tile steps of the workgroup's query block: their number and, with a block
// mask, the list of entries.
__device__ __forceinline__ void tile_range(const FwdArgs& a, int qt, int block_m, int block_n,
                                           int& ntiles, const int*& list) {
    list = nullptr;
    if (a.tile_counts != nullptr) {
        ntiles = a.tile_counts[qt];
        list = a.tile_entries + (int64_t)qt * a.num_k_tiles;
    } else {
        const int q0 = qt * block_m;
        const int kend = a.causal ? min(a.N, q0 + block_m) : a.N;
        ntiles = (kend + block_n - 1) / block_n;
    }
}

// All wavefronts run S, softmax and PV of a tile step between two barriers;
// double-buffered LDS. The copies of tile it+1 go into the free stage at the
// start of step it and are awaited before the barrier that ends it, so their
// latency hides behind a whole step. With a list, entries are loaded two
// steps ahead of their use.
typedef __attribute__((address_space(3))) int lds_int;

// Block-mask list of query tile q0 built by its own workgroup, in LDS: the key
// tiles (in order) that hold a pair allowed by the mask and the causal rule
// for some 32-row slice, each with per-slice any/all bits (list_entry), the
// list the tile_list kernel builds in global memory (rowwise_fwd.hip). One key
// tile per thread and round; compacted with a per-wavefront ballot and a
// prefix over the wavefronts' counts. Returns the entry count (uniform).
template <int NWAVES>
__device__ int build_tile_list_lds(const FwdArgs& a, int q0, int block_n, lds_int* list, lds_int* wave_counts) {
    constexpr int NT = NWAVES * 64;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int count = 0;
    // The mask-block rows of each slice are the same for every thread (the
    // query tile is the workgroup's); only the key tile differs. They are
    // formed once, and by shifts where the block sizes are powers of two
    // (the common case; a division costs some twenty VALU instructions).
    const bool pow2 = (a.mask_qbs & (a.mask_qbs - 1)) == 0 && (a.mask_kbs & (a.mask_kbs - 1)) == 0;  // uniform
    const int lq = __builtin_ctz((unsigned)a.mask_qbs), lk = __builtin_ctz((unsigned)a.mask_kbs);
    int sq0[NWAVES], sq1[NWAVES], se[NWAVES];
    bool one_qb = true;  // every slice within one mask-block row (uniform)
#pragma unroll
    for (int w = 0; w < NWAVES; ++w) {
        const int s0 = q0 + kQueriesPerWave * w, s1 = min(a.M, s0 + kQueriesPerWave);
        se[w] = s1;
        sq0[w] = s0 < s1 ? (pow2 ? s0 >> lq : s0 / a.mask_qbs) : 1;
        sq1[w] = s0 < s1 ? (pow2 ? (s1 - 1) >> lq : (s1 - 1) / a.mask_qbs) : 0;  // empty slice: no rows
        one_qb = one_qb && sq0[w] >= sq1[w];
    }
    for (int base = 0; base < a.num_k_tiles; base += NT) {
        const int kt = base + tid;
        unsigned any_bits = 0, full_bits = 0;
        if (kt < a.num_k_tiles) {
            const int k0 = kt * block_n, k1 = min(a.N, k0 + block_n);
            const int kb0 = pow2 ? k0 >> lk : k0 / a.mask_kbs;
            const int kb1 = pow2 ? (k1 - 1) >> lk : (k1 - 1) / a.mask_kbs;
            if (one_qb && kb0 == kb1) {
                // One mask byte per slice (the common case: blocks no smaller
                // than a slice and a key tile), all requested before any is
                // used: the loops below would wait for each in turn. Same
                // rule as classify_mask_blocks.
                unsigned char mb[NWAVES];
#pragma unroll
                for (int w = 0; w < NWAVES; ++w)
                    mb[w] = a.mask[(int64_t)min(sq0[w], a.mask_qb - 1) * a.mask_kb + min(kb0, a.mask_kb - 1)];
#pragma unroll
                for (int w = 0; w < NWAVES; ++w) {
                    const int qe = min(se[w], (sq0[w] + 1) * a.mask_qbs);
                    const bool allowed = sq0[w] <= sq1[w] && sq0[w] < a.mask_qb && kb0 < a.mask_kb && mb[w] != 0;
                    const bool any = allowed && (!a.causal || k0 <= qe - 1);
                    any_bits |= (any ? 1u : 0u) << w;
                    full_bits |= (allowed ? 1u : 0u) << w;
                }
            } else {
#pragma unroll
                for (int w = 0; w < NWAVES; ++w) {
                    if (sq0[w] > sq1[w]) continue;
                    bool any, all;
                    classify_mask_blocks(a.mask, a.mask_qbs, a.mask_kbs, a.mask_qb, a.mask_kb, a.causal, se[w],
                                         k0, sq0[w], sq1[w], kb0, kb1, any, all);
                    any_bits |= (any ? 1u : 0u) << w;
                    full_bits |= (all ? 1u : 0u) << w;
                }
            }
        }
        const unsigned long long bal = __ballot(any_bits != 0);
        if (lane == 0) wave_counts[wave] = __popcll(bal);
        __syncthreads();
        int before = count, total = count;
#pragma unroll
        for (int w = 0; w < NWAVES; ++w) {
            const int c = wave_counts[w];
            before += w < wave ? c : 0;
            total += c;
        }
        if (any_bits != 0) list[before + __popcll(bal & ((1ull << lane) - 1ull))] = list_entry(kt, any_bits, full_bits);
        __syncthreads();  // wave_counts is rewritten in the next round
        count = total;
    }
    return count;
}

// Stages of the LDS-list schedule: tiles it+1 .. it+NSTAGE-1 are in flight
// while tile it is computed (three stages up to D = 64, two above, where a
// stage is 32 KB or more).
template <int D>
constexpr int lds_list_stages() { return D <= 64 ? 3 : 2; }
constexpr int kLdsListCountsBytes = 64;  // per-wavefront counts, then the list

// Block-mask query tile with its list in LDS (one workgroup per query tile,
// no key split): the list is built first (mask reads only, before any K/V
// load), then the K/V tiles of its entries stream through a ring of
// NSTAGE stages, NSTAGE-1 tiles ahead of the one being computed. The list is
// read from LDS, so the only vector-memory operations in the loop are the
// tile copies (2 CPT per thread and tile) and the wait before each barrier
// leaves the younger tiles' copies in flight.
template <typename W, int NWAVES, int MOD>
__device__ __forceinline__ void lds_list_qtile(const FwdArgs& a, unsigned char* smem, int bh, int qt, int q0,
                                               int wave) {
    using L = typename W::L;
    constexpr int D = L::CPR * 8;
    constexpr int NSTAGE = lds_list_stages<D>();
    constexpr int VM_PER_TILE = 2 * W::CPT;
    static_assert(W::SN == W::BN, "one compute step per list entry");
    lds_int* counts = (lds_int*)(smem + NSTAGE * L::STAGE);
    lds_int* lst = counts + kLdsListCountsBytes / 4;
    const int ntiles = build_tile_list_lds<NWAVES>(a, q0, W::BN, lst, counts);
    W w(a, smem, bh, q0, wave);
    if (ntiles == 0) {  // uniform over the workgroup
        w.store_output();
        return;
    }
    auto tile_of = [](int e) { return list_tile(e); };
    w.copy_tile(tile_of(lst[0]), 0);
    if (NSTAGE > 2 && ntiles > 1) {
        w.copy_tile(tile_of(lst[1]), L::STAGE);
        wait_vm<VM_PER_TILE>();  // tile 0 (and the Q fragments) landed; tile 1 in flight
    } else {
        wait_vm_loads();
    }
    w.zero_tail(tile_of(lst[0]), 0);
    __syncthreads();
    int stage = 0;
    for (int it = 0; it < ntiles; ++it) {
        const int ahead = it + NSTAGE - 1;  // tile copied during this step
        int astage = stage + (NSTAGE - 1) * L::STAGE;
        if (astage >= NSTAGE * L::STAGE) astage -= NSTAGE * L::STAGE;
        if (ahead < ntiles) w.copy_tile(tile_of(lst[ahead]), astage);
        const int e = lst[it];
        if (w.tile_active(e)) {
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
            w.qk(stage);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
            w.softmax(e);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
            w.pv(stage);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
        }
        // tile it+1 must have landed; the copies of tile it+2 may stay in flight
        if (NSTAGE > 2 && it + 2 < ntiles) wait_vm<VM_PER_TILE>();
        else wait_vm_loads();
        int nstage = stage + L::STAGE;
        if (nstage >= NSTAGE * L::STAGE) nstage = 0;
        if (it + 1 < ntiles) w.zero_tail(tile_of(lst[it + 1]), nstage);
        __syncthreads();
        stage = nstage;
    }
    w.store_output();
}

template <typename T, int D, int MOD, bool LIST, int NWAVES, int BN, int SB, bool SPLIT, int DVK = D>
__device__ __forceinline__ void lockstep_qtile(const FwdArgs& a, unsigned char* smem, int bh, int qt,
                                               int split = 0) {
    constexpr int NTHREADS = NWAVES * 64;
    constexpr int BLOCK_M = NWAVES * kQueriesPerWave;
    static_assert(!LIST || NWAVES <= kListSlices, "list entries carry one bit per wavefront");
    using W = Wave32<T, D, MOD, LIST, NTHREADS, BN, SB, DVK>;
    using L = typename W::L;
    static_assert(2 * L::STAGE >= 24 * NTHREADS + 4, "split merge scratch fits in the LDS stages");
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q0 = qt * BLOCK_M;
    if constexpr (!LIST) {
        // SB compute steps of BN keys per staged tile of SB*BN keys (one
        // barrier per staged tile); no list. Tile
        // st+1 is copied global -> LDS (no registers) into the free stage at
        // the start of step st and awaited before the barrier that ends it.
        static_assert(!LIST, "LDS copies: no list");
        const int kend = a.causal ? min(a.N, q0 + BLOCK_M) : a.N;
        const int nst = (kend + W::SN - 1) / W::SN;      // staged tiles
        const int active = SPLIT ? split_active(a, nst) : 1;
        if (split >= active) return;                     // uniform over the workgroup
        const int range = SPLIT ? split_range(a, nst) : nst;
        const int st0 = SPLIT ? split * range : 0;
        const int st1 = SPLIT ? min(nst, st0 + range) : nst;
        W w(a, smem, bh, q0, wave);
        if (st0 >= st1) {  // uniform over the workgroup
            finish_qtile<W, NTHREADS, SPLIT>(a, w, smem, bh, qt, q0, BLOCK_M, split, active);
            return;
        }
        // (returning early keeps every path into the loop through the wait
        // below, so the compiler sees the Q fragments resident in the loop)
        w.copy_tile(st0, 0);
        wait_vm_loads();
        w.zero_tail(st0, 0);
        __syncthreads();
        for (int st = st0; st < st1; ++st) {
            const int stage = ((st - st0) & 1) * L::STAGE;
            const int nstage = ((st - st0 + 1) & 1) * L::STAGE;
            if (st + 1 < st1) w.copy_tile(st + 1, nstage);
#pragma unroll
            for (int j = 0; j < SB; ++j) {
                const int e = st * SB + j;               // BN-key compute tile
                if (e * BN < kend && w.tile_active(e)) {
                    // Plain scale: matrix phases at wave priority 1 and the
                    // softmax at 0, so that a wavefront ready for MFMAs issues
                    // first when the two wavefronts of a SIMD drift apart
                    // (measured +1-2 %; with a score_mod the longer softmax is
                    // better left at equal priority).
                    if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
                    w.qk(stage, j);
                    if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
                    w.softmax(e);
                    if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
                    w.pv(stage, j);
                    if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
                }
            }
            wait_vm_loads();
            if (st + 1 < st1) w.zero_tail(st + 1, nstage);
            __syncthreads();
        }
        finish_qtile<W, NTHREADS, SPLIT>(a, w, smem, bh, qt, q0, BLOCK_M, split, active);
        return;
    }
    if constexpr (LIST) {
        if (a.tile_counts == nullptr) {  // list built in LDS (no key split)
            lds_list_qtile<W, NWAVES, MOD>(a, smem, bh, qt, q0, wave);
            return;
        }
    }
    int ntiles;
    const int* list;
    tile_range(a, qt, BLOCK_M, BN, ntiles, list);
    const int active = SPLIT ? split_active(a, ntiles) : 1;
    if (split >= active) return;  // uniform over the workgroup
    const int range = SPLIT ? split_range(a, ntiles) : ntiles;
    const int it0 = SPLIT ? split * range : 0;
    const int it1 = SPLIT ? min(ntiles, it0 + range) : ntiles;
    W w(a, smem, bh, q0, wave);
    w.ntiles = ntiles;
    w.list = list;
    // entry it+1 is copied during step it
    if (it0 >= it1) {
        finish_qtile<W, NTHREADS, SPLIT>(a, w, smem, bh, qt, q0, BLOCK_M, split, active);
        return;
    }
    int e_cur = w.entry(it0);
    int e_nxt = it0 + 1 < it1 ? w.entry(it0 + 1) : 0;
    w.copy_tile(w.tile_of(e_cur), 0);
    wait_vm_loads();
    w.zero_tail(w.tile_of(e_cur), 0);
    __syncthreads();
    for (int it = it0; it < it1; ++it) {
        const int stage = ((it - it0) & 1) * L::STAGE;
        const int nstage = ((it - it0 + 1) & 1) * L::STAGE;
        if (it + 1 < it1) w.copy_tile(w.tile_of(e_nxt), nstage);
        const int e_nn = it + 2 < it1 ? w.entry(it + 2) : 0;
        if (w.tile_active(e_cur)) {
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
            w.qk(stage);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
            w.softmax(e_cur);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
            w.pv(stage);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
        }
        wait_vm_loads();
        if (it + 1 < it1) w.zero_tail(w.tile_of(e_nxt), nstage);
        __syncthreads();
        e_cur = e_nxt;
        e_nxt = e_nn;
    }
    finish_qtile<W, NTHREADS, SPLIT>(a, w, smem, bh, qt, q0, BLOCK_M, split, active);
}

// Workgroups per CU the register budget is sized for: one of 8 wavefronts,
// two of 4, or one of 4 from D = 160 up (one wavefront per SIMD, so the O
// accumulators can use the accumulation registers). The plain-scale
// block-mask kernels at D <= 64 fit three of 4 (at most 168 VGPRs: 163 at
// D = 64, 128 at D = 32, no spills; their LDS, three 16 KB stages and the
// list, fits three workgroups too). On the fp16 block-sparse workload the
// third wavefront per SIMD measured within 1 % of two (+0.1 to +0.6 % with
// the timing order alternated). With a score_mod the same bound spills, so
// those keep two.
constexpr int lockstep_min_blocks(int D, int nwaves, int mod, bool list) {
    return nwaves == 8 ? 1 : D >= 160 ? 1 : (list && mod == MOD_PLAIN && D <= 64) ? 3 : 2;
}

// SPLIT (query tiles not paired): the kernel may run a key split; calls with
// one split take the instantiation without it, whose loop then keeps the
// split's values out of its scalar registers (fewer spilled to vector lanes).
template <typename T, int D, int MOD, bool LIST, int NWAVES, bool PAIRED, int BN = kBlockN16, int SB = 1,
          bool SPLIT = true, int DVK = D>
__global__ __launch_bounds__(NWAVES * 64, lockstep_min_blocks(D, NWAVES, MOD, LIST)) void flash_fwd_lockstep_kernel(FwdArgs a) {
    using L = TileLayout<D, BN * SB>;
    // block-mask kernels: LDS sized at launch (list_kernel_lds_bytes)
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
    __shared__ __attribute__((aligned(16))) unsigned char st_smem[LIST ? 16 : 2 * L::STAGE];
    unsigned char* smem = LIST ? dyn_smem : st_smem;
    int bh, qts[2];
    if (!PAIRED) {  // key split s: workgroups [s * tiles, (s+1) * tiles)
        const int tiles = a.B * a.H * a.num_q_tiles;
        const int split = (int)blockIdx.x / tiles;
        map_work((int)blockIdx.x - split * tiles, a.B * a.H, a.num_q_tiles, a.causal, bh, qts[0]);
        lockstep_qtile<T, D, MOD, LIST, NWAVES, BN, SB, SPLIT, DVK>(a, smem, bh, qts[0], split);
        return;
    }
    // (paired query tiles are never split)
    const int n = work_tiles(a, PAIRED, bh, qts);
    lockstep_qtile<T, D, MOD, LIST, NWAVES, BN, SB, false, DVK>(a, smem, bh, qts[0]);
    if (n > 1) {
        __syncthreads();  // LDS stages are reused
        lockstep_qtile<T, D, MOD, LIST, NWAVES, BN, SB, false, DVK>(a, smem, bh, qts[1]);
    }
}

// Block-mask calls whose lists are built in LDS (no key split, no global
// list): the LDS-list path of the lockstep kernel as a kernel of its own, so
// that its loop does not share registers with the global-list path.
template <typename T, int D, int MOD>
__global__ __launch_bounds__(256, lockstep_min_blocks(D, 4, MOD, true)) void flash_fwd_lds_list_kernel(FwdArgs a) {
    extern __shared__ __attribute__((aligned(16))) unsigned char dyn_smem[];
    using W = Wave32<T, D, MOD, true, 256, kBlockN16, 1>;
    int bh, qt;
    map_work((int)blockIdx.x, a.B * a.H, a.num_q_tiles, a.causal, bh, qt);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    lds_list_qtile<W, 4, MOD>(a, dyn_smem, bh, qt, qt * 4 * kQueriesPerWave, wave);
}

// Causal query tile pairs with a key split (FwdArgs::pair_split): workgroup s
// of the pair (nqt-1-p, p) runs split s of both tiles, each tile cut into
// num_splits ranges of its own length, so every workgroup runs about
// (steps(nqt-1-p) + steps(p)) / num_splits staged tiles. A kernel of its own,
// so that the paired kernel without a split keeps its code.
template <typename T, int D, int MOD, int NWAVES, int BN = kBlockN16, int SB = 1>
__global__ __launch_bounds__(NWAVES * 64, lockstep_min_blocks(D, NWAVES, MOD, false)) void flash_fwd_pair_split_kernel(FwdArgs a) {
    using L = TileLayout<D, BN * SB>;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * L::STAGE];
    const int pairs = a.B * a.H * ((a.num_q_tiles + 1) / 2);
    const int split = (int)blockIdx.x / pairs;
    int bh, qa, qb;
    map_work_pair((int)blockIdx.x - split * pairs, a.B * a.H, a.num_q_tiles, bh, qa, qb);
    lockstep_qtile<T, D, MOD, false, NWAVES, BN, SB, true>(a, smem, bh, qa, split);
    if (qb >= 0) {
        __syncthreads();  // LDS stages are reused
        lockstep_qtile<T, D, MOD, false, NWAVES, BN, SB, true>(a, smem, bh, qb, split);
    }
}

// ---------------------------------------------------------------------------
// fp32 inputs: v_mfma_f32_32x32x2_f32. Each MFMA consumes one element per lane
// and operand, so K and V stay row-major in LDS (no transposition): the
// reduction index d of S^T is split as d = g*D/2 + s over the two lane halves,
// and each PV step takes the two keys that the lane halves hold in register u.
// With a key split (FwdArgs::num_splits > 1) the workgroups of a query tile
// each run a range of its K/V tile steps and write partial rows, which
// combine_splits_kernel merges. Causal calls split with FwdArgs::pair_split:
// workgroup s of the pair (nqt-1-p, p) runs split s of both query tiles, each
// tile cut into num_splits ranges of its own length, so a workgroup runs
// about (steps(nqt-1-p) + steps(p)) / num_splits steps whatever p is (with
// one range length for all tiles the longest tile's ranges set the time).

constexpr int kBlockNF32 = 32;  // keys per accumulator block of the fp32 kernel
constexpr int kTilesF32 = 2;    // blocks per K/V tile: 64 keys per barrier (+3 to +5 % over one block)
constexpr int kWaves32 = 4;
constexpr int kThreads32 = kWaves32 * 64;
constexpr int kBlockM32 = kWaves32 * kQueriesPerWave;  // 128

template <int D, int NB>
struct Mfma32Tiles {
    static constexpr int BN = kBlockNF32 * NB;  // NB blocks of 32 keys per K/V tile
    static constexpr int KSTR = D + 4;  // floats; conflict-free 16-byte reads of rows kappa(r)
    static constexpr int VSTR = D + 4;  // floats; lane halves read rows 8 apart -> opposite bank halves
    static constexpr int KTILE = BN * KSTR;
    static constexpr int STAGE = 2 * KTILE;
};

// Query tile qt of head bh, key split `split` (the whole key range without
// one), on the workgroup's LDS `lds` (2 * STAGE floats).
template <int D, bool GENERAL, int NB, bool LISTS = true>
__device__ __forceinline__ void mfma32_qtile(const FwdArgs& a, float* lds, int bh, int qt, int split) {
    using TL = Mfma32Tiles<D, NB>;
    constexpr int BN = TL::BN;
    constexpr int KSTR = TL::KSTR;
    constexpr int VSTR = TL::VSTR;
    constexpr int KTILE = TL::KTILE;
    constexpr int STAGE = TL::STAGE;
    constexpr int CHUNKS = BN * D / 4;
    constexpr int CPT = CHUNKS / kThreads32;
    constexpr int NDC = D / 4;
    static_assert(CHUNKS % kThreads32 == 0, "tile must split evenly over the workgroup");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, r = lane & 31;
    const int b = bh / a.H, h = bh - b * a.H;
    const float* __restrict__ Qp = (const float*)a.q + b * a.q_sb + h * a.q_sh;
    const float* __restrict__ Kp = (const float*)a.k + b * a.k_sb + h * a.k_sh;
    const float* __restrict__ Vp = (const float*)a.v + b * a.v_sb + h * a.v_sh;
    const int q0 = qt * kBlockM32;
    const int qw0 = q0 + wave * kQueriesPerWave;
    const int my_q = qw0 + r;

    // Q^T operand: lane holds Q[my_q][g*D/2 + s]; rows past M and columns at
    // or past a.D (the kernel's D is the head dim rounded up) are zero
    float qf[D / 2];
    {
        const float* qrow = Qp + (int64_t)my_q * a.q_sm + g * (D / 2);
#pragma unroll
        for (int c = 0; c < D / 8; ++c) {
            f32x4 u = {0.f, 0.f, 0.f, 0.f};
            if (my_q < a.M && g * (D / 2) + 4 * c < a.D) u = *(const f32x4*)(qrow + 4 * c);
#pragma unroll
            for (int t = 0; t < 4; ++t) qf[4 * c + t] = u[t];
        }
    }

    int ntiles;
    const int* list = nullptr;
    if (LISTS && a.tile_counts != nullptr) {
        ntiles = a.tile_counts[qt];
        list = a.tile_entries + (int64_t)qt * a.num_k_tiles;
    } else {
        const int kend = a.causal ? min(a.N, q0 + kBlockM32) : a.N;
        ntiles = (kend + BN - 1) / BN;
    }
    // tile steps [it0, it1) of this workgroup's key split
    const int active = split_active(a, ntiles);
    if (split >= active) return;  // uniform over the workgroup
    const int range = split_range(a, ntiles);
    const int it0 = split * range;
    const int it1 = min(ntiles, it0 + range);

    f32x4 kreg[CPT], vreg[CPT];
    auto load_tile = [&](int kt) {
        const int k0 = kt * BN;
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const int ci = tid + kThreads32 * u;
            const int row = ci / NDC, cc = ci % NDC;
            const int kj = k0 + row;
            kreg[u] = f32x4{0.f, 0.f, 0.f, 0.f};
            vreg[u] = f32x4{0.f, 0.f, 0.f, 0.f};
            // columns past the head dims stay zero
            if (kj < a.N && 4 * cc < a.D) kreg[u] = *(const f32x4*)(Kp + (int64_t)kj * a.k_sn + 4 * cc);
            if (kj < a.N && 4 * cc < a.Dv) vreg[u] = *(const f32x4*)(Vp + (int64_t)kj * a.v_sn + 4 * cc);
        }
    };
    auto store_tile = [&](int buf) {
        float* Ks = lds + buf * STAGE;
        float* Vs = Ks + KTILE;
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const int ci = tid + kThreads32 * u;
            const int row = ci / NDC, cc = ci % NDC;
            *(f32x4*)(Ks + row * KSTR + 4 * cc) = kreg[u];
            *(f32x4*)(Vs + row * VSTR + 4 * cc) = vreg[u];
        }
    };
    auto tile_at = [&](int it, int& ent) -> int {
        if (list != nullptr) {
            ent = list[it];
            return list_tile(ent);
        }
        ent = 0;
        return it;
    };

    f32x16 o[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) o[db] = f32x16{};
    float m_run = kNegInf, l_run = 0.0f;
    const float slope = (GENERAL && a.bias_kind == BIAS_ALIBI) ? a.alibi[h] : 0.0f;
    const float* bias_row = nullptr;
    if (GENERAL && a.bias_kind == BIAS_DENSE && my_q < a.M)
        bias_row = a.bias + b * a.bias_sb + h * a.bias_sh + (int64_t)my_q * a.bias_sm;

    if (it0 < it1) {
        int e0;
        load_tile(tile_at(it0, e0));
    }
    wait_vm_loads();
    if (it0 < it1) store_tile(0);
    __syncthreads();

    for (int it = it0; it < it1; ++it) {
        int ent;
        const int kt = tile_at(it, ent);
        if (it + 1 < it1) {
            int en;
            load_tile(tile_at(it + 1, en));
        }
        const float* Ks = lds + ((it - it0) & 1) * STAGE;
        const float* Vs = Ks + KTILE;
        const int k0 = kt * BN;
        const bool active = list != nullptr ? list_any(ent, wave)
                                            : !(a.causal && k0 > qw0 + kQueriesPerWave - 1);
        if (active) {
            const bool need_mask = ((k0 + BN > a.N) || (a.causal && k0 + BN - 1 > qw0)) ||
                                   (list != nullptr && !list_full(ent, wave));
            f32x16 s[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] = f32x16{};
            const float* krow = Ks + kappa(r) * KSTR + g * (D / 2);
#pragma unroll
            for (int c = 0; c < D / 8; ++c) {
                f32x4 kv[NB];
#pragma unroll
                for (int b = 0; b < NB; ++b) kv[b] = *(const f32x4*)(krow + 32 * b * KSTR + 4 * c);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        s[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(kv[b][t], qf[4 * c + t], s[b], 0, 0, 0);
            }
            const float alpha = online_softmax_tile<NB, GENERAL>(a, s, need_mask, my_q, k0, g, slope,
                                                                 bias_row, m_run, l_run);
#pragma unroll
            for (int db = 0; db < D / 32; ++db) o[db] *= alpha;
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    const float* vrow = Vs + (32 * b + acc_pos(u, g)) * VSTR + r;
#pragma unroll
                    for (int db = 0; db < D / 32; ++db)
                        o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vrow[32 * db], s[b][u], o[db], 0, 0, 0);
                }
        }
        if (it + 1 < it1) store_tile((it + 1 - it0) & 1);
        __syncthreads();
    }

    const float l_tot = l_run + __shfl_xor(l_run, 32);
    if (active > 1) {
        // partial row: unnormalised O and (m, l), merged by the last split to arrive
        if (my_q < a.M) {
            const int64_t prow = ((int64_t)split * a.B * a.H + bh) * a.M + my_q;
            float* po = a.part_o + prow * a.Dv + 4 * g;
            const bool coh = a.split_counters != nullptr;
#pragma unroll
            for (int db = 0; db < D / 32; ++db) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (32 * db + 8 * i + 4 * g >= a.Dv) continue;  // past the value dim
                    f32x4 val;
#pragma unroll
                    for (int j = 0; j < 4; ++j) val[j] = o[db][4 * i + j];
                    put_partial4(po + 32 * db + 8 * i, val, coh);
                }
            }
            if (g == 0) {
                put_partial(a.part_ml + 2 * prow, m_run, coh);
                put_partial(a.part_ml + 2 * prow + 1, l_tot, coh);
            }
        }
        if (a.split_counters == nullptr) return;  // merged by combine_splits_kernel
        __syncthreads();                          // LDS below is reused
        static_assert(2 * STAGE * 4 >= 24 * kThreads32 + 4, "split merge scratch fits in the LDS stages");
        int* flag = (int*)(lds + 6 * kThreads32);
        if (split_arrive(a.split_counters + (int64_t)bh * a.num_q_tiles + qt, active, flag))
            merge_split_rows<float, kThreads32>(a, bh, q0, min(kBlockM32, a.M - q0), active, lds);
        return;
    }
    const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
    if (my_q < a.M) {
        float* orow = (float*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)my_q * a.o_sm + 4 * g;
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (32 * db + 8 * i + 4 * g >= a.Dv) continue;  // past the value dim
                f32x4 val;
#pragma unroll
                for (int j = 0; j < 4; ++j) val[j] = o[db][4 * i + j] * inv;
                *(f32x4*)(orow + 32 * db + 8 * i) = val;
            }
        }
    }
}

// PAIRS_ONLY: causal calls without a block mask, which always run query tile
// pairs: an instantiation without the unpaired and list paths, whose values
// then stay out of its scalar registers (57 -> 10 spilled at D = 64; +1 %).
template <int D, bool GENERAL, int NB = 1, bool PAIRS_ONLY = false>
__global__ __launch_bounds__(kThreads32) void flash_fwd_mfma32_kernel(FwdArgs a) {
    __shared__ __attribute__((aligned(16))) float lds[2 * Mfma32Tiles<D, NB>::STAGE];
    if (PAIRS_ONLY || a.pair_split) {  // causal query tile pairs, split s of both tiles
        const int pairs = a.B * a.H * ((a.num_q_tiles + 1) / 2);
        const int split = (int)blockIdx.x / pairs;
        int bh, qa, qb;
        map_work_pair((int)blockIdx.x - split * pairs, a.B * a.H, a.num_q_tiles, bh, qa, qb);
        mfma32_qtile<D, GENERAL, NB, !PAIRS_ONLY>(a, lds, bh, qa, split);
        if (qb >= 0) {
            __syncthreads();  // LDS stages are reused
            mfma32_qtile<D, GENERAL, NB, !PAIRS_ONLY>(a, lds, bh, qb, split);
        }
        return;
    }
    int bh, qt;
    const int tiles_per_split = a.B * a.H * a.num_q_tiles;
    const int split = (int)blockIdx.x / tiles_per_split;
    map_work((int)blockIdx.x - split * tiles_per_split, a.B * a.H, a.num_q_tiles, a.causal, bh, qt);
    mfma32_qtile<D, GENERAL, NB>(a, lds, bh, qt, split);
}

// fp32 calls with few query rows (latency-bound: fewer 128-row query tiles
// than CUs). A workgroup of four wavefronts covers one 32-row query block and
// the wavefronts take its 32-key tiles in turn (wavefront w: steps it0 + w,
// it0 + w + 4, ...), so four times as many wavefronts share the work as in
// the 128-row kernel. Each keeps its own running (m, l, O) and reads its K and
// V tiles straight from global memory into the MFMA operand registers (no LDS
// staging, no barrier in the loop); at the end the four states are folded
// through LDS with the log-sum-exp rule (attention.cpp:661-674). Key splits
// across workgroups, and their merge, are those of the 128-row kernel.
template <int D, bool GENERAL>
__global__ __launch_bounds__(kThreads32) void flash_fwd_f32_rows32_kernel(FwdArgs a) {
    constexpr int NO = D / 2;  // O floats per lane
    constexpr int FS = NO + 2;  // folded floats per lane: O, m, l
    __shared__ __attribute__((aligned(16))) float fold[3 * FS * 64];
    static_assert(3 * FS * 64 >= 6 * kThreads32 + 1, "split merge scratch fits in the fold buffer");

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, r = lane & 31;
    int bh, qt;
    const int tiles_per_split = a.B * a.H * a.num_q_tiles;
    const int split = (int)blockIdx.x / tiles_per_split;
    map_work((int)blockIdx.x - split * tiles_per_split, a.B * a.H, a.num_q_tiles, a.causal, bh, qt);
    const int b = bh / a.H, h = bh - b * a.H;
    const float* __restrict__ Qp = (const float*)a.q + b * a.q_sb + h * a.q_sh;
    const float* __restrict__ Kp = (const float*)a.k + b * a.k_sb + h * a.k_sh;
    const float* __restrict__ Vp = (const float*)a.v + b * a.v_sb + h * a.v_sh;
    const int q0 = qt * kRowsF32;
    const int my_q = q0 + r;

    const int kend = a.causal ? min(a.N, q0 + kRowsF32) : a.N;
    const int ntiles = (kend + kBlockNF32 - 1) / kBlockNF32;
    const int active = split_active(a, ntiles);
    if (split >= active) return;  // uniform over the workgroup
    const int it0 = split * a.split_tiles;
    const int it1 = min(ntiles, it0 + a.split_tiles);

    // Q^T operand: lane holds Q[my_q][g*D/2 + s] (rows past M: zero)
    float qf[D / 2];
    {
        const float* qrow = Qp + (int64_t)min(my_q, a.M - 1) * a.q_sm + g * (D / 2);
#pragma unroll
        for (int c = 0; c < D / 8; ++c) {
            f32x4 u = {0.f, 0.f, 0.f, 0.f};
            // columns at or past a.D (the kernel's D rounds the head dim up) are zero
            if (g * (D / 2) + 4 * c < a.D) u = *(const f32x4*)(qrow + 4 * c);
            if (my_q >= a.M) u = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < 4; ++t) qf[4 * c + t] = u[t];
        }
    }
    f32x16 o[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) o[db] = f32x16{};
    float m_run = kNegInf, l_run = 0.0f;
    const float slope = (GENERAL && a.bias_kind == BIAS_ALIBI) ? a.alibi[h] : 0.0f;
    const float* bias_row = nullptr;
    if (GENERAL && a.bias_kind == BIAS_DENSE && my_q < a.M)
        bias_row = a.bias + b * a.bias_sb + h * a.bias_sh + (int64_t)my_q * a.bias_sm;

    // K/V operand registers of tile it (A operands of S^T = K Q^T and of
    // O^T += V^T P^T): K[k0 + kappa(r)][g*D/2 + s] and V[k0 + acc_pos(u, g)][r + 32 db].
    // Rows past N read row N-1 (their scores are masked) and V past N is zero.
    // Up to D = 64 the next tile of the wavefront is loaded while this one is
    // computed (registers allow two sets).
    constexpr bool PREFETCH = D <= 64;
    struct KV {
        f32x4 k[D / 8];
        float v[16][D / 32];
    };
    auto load_kv = [&](int it, KV& t) {
        const int k0 = it * kBlockNF32;
        const float* krow = Kp + (int64_t)min(k0 + kappa(r), a.N - 1) * a.k_sn + g * (D / 2);
#pragma unroll
        for (int c = 0; c < D / 8; ++c) {
            t.k[c] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (g * (D / 2) + 4 * c < a.D) t.k[c] = *(const f32x4*)(krow + 4 * c);
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const int kj = k0 + acc_pos(u, g);
            const float* vrow = Vp + (int64_t)min(kj, a.N - 1) * a.v_sn + r;
#pragma unroll
            for (int db = 0; db < D / 32; ++db) {
                float x = 0.0f;
                if (r + 32 * db < a.Dv) x = vrow[32 * db];
                t.v[u][db] = kj < a.N ? x : 0.0f;
            }
        }
    };
    auto compute = [&](int it, const KV& t) {
        const int k0 = it * kBlockNF32;
        f32x16 s[1] = {f32x16{}};
#pragma unroll
        for (int c = 0; c < D / 8; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                s[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(t.k[c][j], qf[4 * c + j], s[0], 0, 0, 0);
        const bool need_mask = (k0 + kBlockNF32 > a.N) || (a.causal && k0 + kBlockNF32 - 1 > q0);
        const float alpha =
            online_softmax_tile<1, GENERAL>(a, s, need_mask, my_q, k0, g, slope, bias_row, m_run, l_run);
#pragma unroll
        for (int db = 0; db < D / 32; ++db) o[db] *= alpha;
#pragma unroll
        for (int u = 0; u < 16; ++u)
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
                o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(t.v[u][db], s[0][u], o[db], 0, 0, 0);
    };
    if constexpr (PREFETCH) {
        KV cur, nxt;
        int it = it0 + wave;
        if (it < it1) load_kv(it, cur);
        for (; it < it1; it += kWaves32) {
            const bool more = it + kWaves32 < it1;
            if (more) load_kv(it + kWaves32, nxt);
            compute(it, cur);
            if (more) cur = nxt;
        }
    } else {
        for (int it = it0 + wave; it < it1; it += kWaves32) {
            KV cur;
            load_kv(it, cur);
            compute(it, cur);
        }
    }

    // Fold wavefronts 1-3 into wavefront 0 (the four hold the same rows in the
    // same lane layout); a wavefront that saw no tile has m = -inf, l = 0, O = 0.
    if (wave > 0) {
        float* f = fold + (wave - 1) * FS * 64 + lane;
#pragma unroll
        for (int i = 0; i < NO; ++i) f[64 * i] = o[i >> 4][i & 15];
        f[64 * NO] = m_run;
        f[64 * (NO + 1)] = l_run;
    }
    __syncthreads();
    if (wave == 0) {
        float mg = m_run;
#pragma unroll
        for (int w = 0; w < kWaves32 - 1; ++w) mg = fmaxf(mg, fold[w * FS * 64 + 64 * NO + lane]);
        const float mu = mg == kNegInf ? 0.0f : mg;
        const float w0 = __builtin_amdgcn_exp2f(m_run - mu);  // 0 while m_run is -inf
        l_run *= w0;
#pragma unroll
        for (int db = 0; db < D / 32; ++db) o[db] *= w0;
#pragma unroll
        for (int w = 0; w < kWaves32 - 1; ++w) {
            const float* f = fold + w * FS * 64 + lane;
            const float ww = __builtin_amdgcn_exp2f(f[64 * NO] - mu);
            l_run += ww * f[64 * (NO + 1)];
#pragma unroll
            for (int i = 0; i < NO; ++i) o[i >> 4][i & 15] += ww * f[64 * i];
        }
        m_run = mg;
    }
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    if (active > 1) {
        // partial row: unnormalised O and (m, l), merged by the last split to arrive
        const bool coh = a.split_counters != nullptr;
        if (wave == 0 && my_q < a.M) {
            const int64_t prow = ((int64_t)split * a.B * a.H + bh) * a.M + my_q;
            float* po = a.part_o + prow * a.Dv + 4 * g;
#pragma unroll
            for (int db = 0; db < D / 32; ++db) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (32 * db + 8 * i + 4 * g >= a.Dv) continue;  // past the value dim
                    f32x4 val;
#pragma unroll
                    for (int j = 0; j < 4; ++j) val[j] = o[db][4 * i + j];
                    put_partial4(po + 32 * db + 8 * i, val, coh);
                }
            }
            if (g == 0) {
                put_partial(a.part_ml + 2 * prow, m_run, coh);
                put_partial(a.part_ml + 2 * prow + 1, l_tot, coh);
            }
        }
        if (!coh) return;  // merged by combine_splits_kernel
        __syncthreads();   // the fold buffer below is reused
        int* flag = (int*)(fold + 6 * kThreads32);
        if (split_arrive(a.split_counters + (int64_t)bh * a.num_q_tiles + qt, active, flag))
            merge_split_rows<float, kThreads32>(a, bh, q0, min(kRowsF32, a.M - q0), active, fold);
        return;
    }
    if (wave == 0 && my_q < a.M) {
        const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        float* orow = (float*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)my_q * a.o_sm + 4 * g;
#pragma unroll
        for (int db = 0; db < D / 32; ++db) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (32 * db + 8 * i + 4 * g >= a.Dv) continue;  // past the value dim
                f32x4 val;
#pragma unroll
                for (int j = 0; j < 4; ++j) val[j] = o[db][4 * i + j] * inv;
                *(f32x4*)(orow + 32 * db + 8 * i) = val;
            }
        }
    }
}

// One 32-key tile of online softmax on two 16x16 score blocks (keys k0 + 16 kb
// + 4 kq + i of query my_q in register i of block kb), in place; the four
// lanes of a query (kq = 0..3) exchange their maxima. Returns alpha.
template <bool GENERAL>
__device__ __forceinline__ float online_softmax_16(const FwdArgs& a, f32x4 (&s)[2], bool need_mask, int my_q,
                                                   int k0, int kq, float slope, const float* bias_row,
                                                   float& m_run, float& l_run) {
    float mx = kNegInf;
    const bool row_out = GENERAL && my_q >= a.M;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kj = k0 + 16 * kb + 4 * kq + i;
            float x;
            if (!GENERAL && !need_mask) {
                x = s[kb][i] * a.scale_log2;
            } else {
                x = kNegInf;
                if (!(row_out || (need_mask && elem_masked(a, my_q, kj))))
                    x = GENERAL ? general_score(a, s[kb][i], my_q, kj, slope, bias_row) : s[kb][i] * a.scale_log2;
            }
            s[kb][i] = x;
            mx = fmaxf(mx, x);
        }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == kNegInf) ? 0.0f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
    m_run = m_new;
    float lsum = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float p = __builtin_amdgcn_exp2f(s[kb][i] - m_use);
            s[kb][i] = p;
            lsum += p;
        }
    }
    l_run = l_run * alpha + lsum;
    return alpha;
}

// fp32 calls with few query rows and few keys: 16-row query blocks, one
// workgroup of sixteen wavefronts per block (one workgroup per CU), no key
// split, so no partial rows leave the CU. Wavefront w takes the block's
// 32-key tiles w, w + 16, ... on v_mfma_f32_16x16x4f32: its K tile copied
// into LDS, its V tile read straight into the operand registers, the block's
// Q rows read once per workgroup through LDS; the sixteen (m, l, O) states
// are folded through LDS with the log-sum-exp rule (attention.cpp:661-674).
//
// Operand layout (lane l: n = l % 16, kq = l / 16). The head dim is permuted
// inside each contraction, which leaves every sum unchanged:
//   S^T = K Q^T: instruction c = 4 cc + t (< D/4) contracts over d = 16 cc +
//     4 kq + t, so lane l holds K[key][16 cc + 4 kq, +4) and Q[q0 + n][16 cc
//     + 4 kq, +4) as one 16-byte chunk per cc (the four lanes of a row read
//     64 contiguous bytes); score block kb lands as
//     S^T[k0 + 16 kb + 4 kq + i][q0 + n] in register i.
//   O^T += V^T P^T: instruction (kb, i) contracts over keys k0 + 16 kb +
//     4 kq + i, whose probability is the lane's own register i of block kb;
//     output block db holds d = (D/16) m + db in row m, so lane l reads
//     V[key][(D/16) n, +D/16) in one load, and holds O[q0 + n][(D/4) kq, +D/4)
//     with d = (D/4) kq + e in element e = (D/16) i + db.
constexpr int kWavesRows16 = 16;
constexpr int kThreadsRows16 = kWavesRows16 * 64;

template <int D, bool GENERAL>
__global__ __launch_bounds__(kThreadsRows16) void flash_fwd_f32_rows16_kernel(FwdArgs a) {
    static_assert(D == 32 || D == 64, "16-row fp32 blocks: D = 32 or 64");
    constexpr int NC = D / 4;   // contraction floats per lane of S^T, O floats per lane
    constexpr int NDB = D / 16;  // 16-row blocks of O^T
    typedef float vrow_t __attribute__((ext_vector_type(NDB)));
    constexpr int QSTR = D + 4;  // LDS row stride of the Q block (16 rows at distinct banks)
    constexpr int CPR = D / 4;   // 16-byte chunks per K row
    constexpr int KT = kBlockNF32 * D;  // floats of one wavefront's K tile in LDS
    static_assert(64 * NC <= KT, "a wavefront's folded state fits in its K tile");
    // K tiles, one per wavefront (later its folded state); Q block; (m, l) per wavefront and query
    __shared__ __attribute__((aligned(16))) float k_lds[kWavesRows16 * KT];
    __shared__ float fold_ml[kWavesRows16 * 32];
    __shared__ __attribute__((aligned(16))) float q_lds[kRowsF32Narrow * QSTR];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15, kq = lane >> 4;
    int bh, qt;
    map_work((int)blockIdx.x, a.B * a.H, a.num_q_tiles, a.causal, bh, qt);
    const int b = bh / a.H, h = bh - b * a.H;
    const float* __restrict__ Qp = (const float*)a.q + b * a.q_sb + h * a.q_sh;
    const float* __restrict__ Kp = (const float*)a.k + b * a.k_sb + h * a.k_sh;
    const float* __restrict__ Vp = (const float*)a.v + b * a.v_sb + h * a.v_sh;
    const int q0 = qt * kRowsF32Narrow;
    const int my_q = q0 + n;
    const int kend = a.causal ? min(a.N, q0 + kRowsF32Narrow) : a.N;
    const int ntiles = (kend + kBlockNF32 - 1) / kBlockNF32;

    // K tile it is copied into the wavefront's LDS tile (global -> LDS, 1 KB
    // of whole rows per instruction); chunk c of row r sits at slot
    // c ^ kswz(r), so that the operand reads (16 rows at one chunk per 16
    // lanes) meet distinct banks. V is read straight into the operand
    // registers once the K operands are consumed. Rows past N read row N-1
    // (their scores are masked, so their probabilities are exactly 0); K
    // chunks past D re-read the row's last chunk (Q is zero there), V columns
    // past Dv its last columns (those output rows are not stored).
    float* const kw = k_lds + wave * KT;
    auto kswz = [](int r) { return D == 64 ? (r & 15) : ((r >> 1) & 7); };
    auto load_k = [&](int it) {
        const unsigned base = (unsigned)(uintptr_t)kw;
#pragma unroll
        for (int j = 0; j < KT / 256; ++j) {
            const int sl = 64 * j + lane, r = sl / CPR, c = (sl % CPR) ^ kswz(r);
            dma16(Kp + (int64_t)min(it * kBlockNF32 + r, a.N - 1) * a.k_sn + min(4 * c, a.D - 4), base + 1024 * j);
        }
    };
    vrow_t vf[2][4];
    auto load_v = [&](int it) {
        const int vc = min(NDB * n, a.Dv - NDB);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                vf[kb][i] = *(const vrow_t*)(Vp + (int64_t)min(it * kBlockNF32 + 16 * kb + 4 * kq + i, a.N - 1) *
                                                       a.v_sn + vc);
    };
    // The Q block is read by the first 4 D threads (one 16-byte chunk each;
    // rows past M and chunks past D are zero), after which the wavefront's
    // first K tile is requested, and staged through LDS.
    f32x4 qv = {0.f, 0.f, 0.f, 0.f};
    const int qr = tid / (D / 4), qc = 4 * (tid - qr * (D / 4));
    if (tid < 4 * D) {
        qv = *(const f32x4*)(Qp + (int64_t)min(q0 + qr, a.M - 1) * a.q_sm + min(qc, a.D - 4));
        if (q0 + qr >= a.M || qc >= a.D) qv = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (wave < ntiles) load_k(wave);
    if (tid < 4 * D) *(f32x4*)(q_lds + qr * QSTR + qc) = qv;
    __syncthreads();
    float qf[NC];  // Q[my_q][16 cc + 4 kq + t] at 4 cc + t
#pragma unroll
    for (int cc = 0; cc < NC / 4; ++cc) {
        const f32x4 u = *(const f32x4*)(q_lds + n * QSTR + 16 * cc + 4 * kq);
#pragma unroll
        for (int t = 0; t < 4; ++t) qf[4 * cc + t] = u[t];
    }
    f32x4 o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = kNegInf, l_run = 0.0f;
    const float slope = (GENERAL && a.bias_kind == BIAS_ALIBI) ? a.alibi[h] : 0.0f;
    const float* bias_row = nullptr;
    if (GENERAL && a.bias_kind == BIAS_DENSE && my_q < a.M)
        bias_row = a.bias + b * a.bias_sb + h * a.bias_sh + (int64_t)my_q * a.bias_sm;

    for (int it = wave; it < ntiles; it += kWavesRows16) {
        const int k0 = it * kBlockNF32;
        if (it != wave) load_k(it);
        wait_vm_loads();  // this wavefront's K copy has landed
        f32x4 kf[2][NC / 4];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int cc = 0; cc < NC / 4; ++cc)
                kf[kb][cc] = *(const f32x4*)(kw + (16 * kb + n) * D + 4 * ((4 * cc + kq) ^ kswz(16 * kb + n)));
        f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                s[kb] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[kb][c >> 2][c & 3], qf[c], s[kb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_v(it);
        const bool need_mask = (k0 + kBlockNF32 > a.N) || (a.causal && k0 + kBlockNF32 - 1 > q0);
        const float alpha =
            online_softmax_16<GENERAL>(a, s, need_mask, my_q, k0, kq, slope, bias_row, m_run, l_run);
#pragma unroll
        for (int db = 0; db < NDB; ++db) o[db] *= alpha;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int db = 0; db < NDB; ++db)
                    o[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[kb][i][db], s[kb][i], o[db], 0, 0, 0);
    }

    // Every wavefront (one that saw no tile has m = -inf, l = 0, O = 0) leaves
    // its O in d order (in its K tile, whose reads are done) and the (m, l)
    // of its 16 queries in LDS.
    l_run += __shfl_xor(l_run, 16);
    l_run += __shfl_xor(l_run, 32);
    {
        float* f = kw + lane * NC;
#pragma unroll
        for (int c = 0; c < NC / 4; ++c) {
            f32x4 val;
#pragma unroll
            for (int t = 0; t < 4; ++t) val[t] = o[(4 * c + t) % NDB][(4 * c + t) / NDB];
            *(f32x4*)(f + 4 * c) = val;
        }
        if (kq == 0) {
            fold_ml[wave * 32 + n] = m_run;
            fold_ml[wave * 32 + 16 + n] = l_run;
        }
    }
    __syncthreads();
    // Thread t folds 4 output columns: lane slot L = t / (NC / 4), chunk t % (NC / 4).
    if (tid < 64 * (NC / 4)) {
        const int L = tid / (NC / 4), c = tid - L * (NC / 4);
        const int qn = L & 15, kqL = L >> 4;
        float mg = kNegInf;
#pragma unroll
        for (int w = 0; w < kWavesRows16; ++w) mg = fmaxf(mg, fold_ml[w * 32 + qn]);
        const float mu = mg == kNegInf ? 0.0f : mg;
        float l = 0.0f;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWavesRows16; ++w) {
            const float ww = __builtin_amdgcn_exp2f(fold_ml[w * 32 + qn] - mu);  // 0 for m = -inf
            l += ww * fold_ml[w * 32 + 16 + qn];
            acc += ww * *(const f32x4*)(k_lds + w * KT + L * NC + 4 * c);
        }
        const int q = q0 + qn, d = NC * kqL + 4 * c;
        if (q < a.M && d < a.Dv) {
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
            *(f32x4*)((float*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)q * a.o_sm + d) = acc * inv;
        }
    }
}

// Merge of key-split partial rows in a launch of its own (no arrival
// counters). A workgroup merges `rows` consecutive rows of one head (a power
// of two, so they lie in one query tile): thread t takes (row, 4-column chunk)
// item t % (rows * chunks) and the splits grp, grp + groups, ... with
// grp = t / (rows * chunks), so that a row's splits are read by `groups`
// threads at once; the groups' results are folded through LDS. T is the
// input type (the output type unless out_f32).
template <typename T>
__global__ __launch_bounds__(256) void combine_splits_kernel(FwdArgs a, int rows, int groups) {
    __shared__ float red[6 * 256];
    const int chunks = a.Dv >> 2;
    const int per_head = (a.M + rows - 1) / rows;
    const int bh = (int)blockIdx.x / per_head;
    const int row0 = ((int)blockIdx.x - bh * per_head) * rows;
    const int qt = row0 / a.split_bm;
    int steps;
    if (a.tile_counts != nullptr) {
        steps = a.tile_counts[qt];
    } else {
        const int kend = a.causal ? min(a.N, (qt + 1) * a.split_bm) : a.N;
        steps = (kend + a.split_bn - 1) / a.split_bn;
    }
    const int active = split_active(a, steps);
    if (active <= 1) return;  // split 0 wrote these rows (uniform over the workgroup)
    const int items = rows * chunks;  // items * groups <= 256
    const int t = threadIdx.x;
    const int item = t % items, grp = t / items;
    const int rr = item / chunks, c = item - rr * chunks;
    const int row = row0 + rr;
    const int ng = min(groups, active);
    const bool mine = grp < ng && row < a.M;
    float m = kNegInf, l = 0.0f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (mine) merge_partials<false>(a, (int64_t)bh * a.M + row, c, grp, ng, active, m, l, acc);
    if (ng > 1) {
        if (mine && grp > 0) {
            float* e = red + 6 * t;
            e[0] = m;
            e[1] = l;
#pragma unroll
            for (int j = 0; j < 4; ++j) e[2 + j] = acc[j];
        }
        __syncthreads();
        if (mine && grp == 0)
            for (int j = 1; j < ng; ++j) {
                const float* e = red + 6 * (j * items + item);
                lse_fold(m, l, acc, e[0], e[1], f32x4{e[2], e[3], e[4], e[5]});
            }
    }
    if (mine && grp == 0) store_merged<T>(a, bh, row, c, l, acc);
}

template <typename K>
hipError_t launch(K kernel, int threads, const FwdArgs& a, hipStream_t s, bool paired = false, size_t lds = 0) {
    const int64_t grid = (int64_t)a.B * a.H * (paired ? (a.num_q_tiles + 1) / 2 : a.num_q_tiles) * a.num_splits;
    if (grid <= 0) return hipSuccess;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(threads), lds, s, a);
    return hipGetLastError();
}

}  // namespace

// 16-bit kernel workgroups: 8 wavefronts (256 query rows) without a
// block-mask list, 4 wavefronts (128 rows, finer skipping) with one, and 4
// wavefronts from D = 192 up (register file), except without score_mod at
// D = 192, where O (96 registers), Q (48) and a 64-key score tile fit two
// wavefronts per SIMD, and at D = 256 with 32-key compute steps (64 keys
// staged; 34-54 VGPRs spilled): 8 wavefronts there whenever the 4-wavefront
// grid (one workgroup per CU) would take more than one round of the CUs (B4
// H32 N4096, D = 192: 0.81 against 1.21 ms causal, 1.44 against 2.22 ms
// non-causal, bit-identical; D = 256: 1.41 against 1.45 ms causal, 2.59
// against 2.82 ms non-causal; bf16 B1 H24 N2048 D192 non-causal, 192
// workgroups of 8 against 384 of 4: 80 against 141 us), 4 on calls that one
// round holds (whose 4-wavefront grid or key split runs faster: bf16 causal
// B2 H16 N2048 D192 84 against 99 us with 8 wavefronts and a pair split, B1
// H8 N2048 43 against 59 us). The 8-wavefront grid then never takes a key
// split: it has more than half as many workgroups as CUs.
static bool eight_waves_wide(bool causal, int64_t bh, int64_t query_tokens) {
    const int64_t nqt4 = (query_tokens + 127) / 128;
    return bh * (causal ? (nqt4 + 1) / 2 : nqt4) > kComputeUnits;
}

// Causal calls without a block-mask list pair query tiles per workgroup.
static bool pairs_causal_tiles(bool causal, bool tile_list) { return causal && !tile_list; }

// Keys per staged K/V tile (one barrier each) of a 16-bit call: 128 without
// score_mod or block mask (half the barriers and tile stores per key), else 64
// (with a block mask a wider tile skips at a coarser grain; the score_mod
// kernel holds all fragments of a tile). At D = 64 the 128 keys are one compute
// step (+9 to +13 %); at D = 128, where S and P for 128 keys would spill, they
// are computed in two 64-key steps between the same barriers (+1 to +5 %).
// D = 32 stages 128 keys in every kernel without a block mask (a 64-key tile
// of 64-byte rows is fewer 16-byte chunks than the 8 wavefronts copy), as do
// D = 96 and 160 (their 64-key tiles do not split evenly over 512 threads);
// D > 160 runs 64-key tiles throughout, on 4 wavefronts (128 query rows) or,
// at D = 192 and 256 without score_mod, 8 (two 32-key compute steps per
// staged tile at D = 256).
static int block_n16(int D, bool general_mod, bool tile_list) {
    if (D > 160 || tile_list) return kBlockN16;
    if (D == 32 || D == 96 || D == 160) return kBlockN16Wide;
    return !general_mod ? kBlockN16Wide : kBlockN16;
}

// LDS of the 16-bit block-mask kernel (4 wavefronts, 64-key tiles): two
// stages with the tile_list kernel's global list, or lds_list_stages stages,
// the per-wavefront counts and the list itself with a list built in LDS.
template <int D>
static size_t list_kernel_lds_bytes_d(bool lds_list, int num_k_tiles) {
    using L = TileLayout<D, kBlockN16>;
    if (!lds_list) return 2 * (size_t)L::STAGE;
    return (size_t)lds_list_stages<D>() * L::STAGE + kLdsListCountsBytes + 4 * (size_t)num_k_tiles;
}

size_t list_kernel_lds_bytes(int D, bool lds_list, int num_k_tiles) {
    switch (D) {
        case 32: return list_kernel_lds_bytes_d<32>(lds_list, num_k_tiles);
        case 64: return list_kernel_lds_bytes_d<64>(lds_list, num_k_tiles);
        case 96: return list_kernel_lds_bytes_d<96>(lds_list, num_k_tiles);
        case 128: return list_kernel_lds_bytes_d<128>(lds_list, num_k_tiles);
        case 160: return list_kernel_lds_bytes_d<160>(lds_list, num_k_tiles);
        case 192: return list_kernel_lds_bytes_d<192>(lds_list, num_k_tiles);
        case 224: return list_kernel_lds_bytes_d<224>(lds_list, num_k_tiles);
        case 256: return list_kernel_lds_bytes_d<256>(lds_list, num_k_tiles);
        default: return 0;
    }
}

template <typename T, int D>
static hipError_t launch16(const FwdArgs& a, bool general_mod, hipStream_t s) {
    const bool list = a.mask != nullptr;
    const bool paired = pairs_causal_tiles(a.causal != 0, list) && a.num_splits == 1;
    if (list) {
        const size_t lds = list_kernel_lds_bytes(D, a.tile_counts == nullptr, a.num_k_tiles);
        if (a.tile_counts == nullptr && a.num_splits == 1)
            return general_mod ? launch(flash_fwd_lds_list_kernel<T, D, MOD_GENERAL>, 256, a, s, false, lds)
                               : launch(flash_fwd_lds_list_kernel<T, D, MOD_PLAIN>, 256, a, s, false, lds);
        return general_mod ? launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, true, 4, false>, 256, a, s, false, lds)
                           : launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, true, 4, false>, 256, a, s, false, lds);
    }
    const bool pair_split = a.pair_split != 0;
    if constexpr (D > 160) {
        if (general_mod) {
            if (pair_split) return launch(flash_fwd_pair_split_kernel<T, D, MOD_GENERAL, 4>, 256, a, s, true);
            return paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, false, 4, true>, 256, a, s, true)
                 : a.num_splits > 1 ? launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, false, 4, false>, 256, a, s)
                          : launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, false, 4, false, kBlockN16, 1, false>, 256, a, s);
        }
        if constexpr (D == 256) {  // 256-row query tiles: 8 wavefronts, 64 keys staged as two 32-key steps
            if (a.split_bm == 8 * kQueriesPerWave) {
                if (pair_split || a.num_splits > 1) return hipErrorInvalidValue;
                return paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, true, 32, 2>, 512, a, s, true)
                              : launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, false, 32, 2, false>, 512, a, s);
            }
        }
        if constexpr (D == 192) {  // 256-row query tiles: 8 wavefronts on 64-key tiles
            // (chosen only where its workgroups outnumber half the CUs, so never with a key split)
            if (a.split_bm == 8 * kQueriesPerWave) {
                if (pair_split || a.num_splits > 1) return hipErrorInvalidValue;
                if (a.Dv <= 128)  // value columns 128 (e.g. 192/128 query-key/value heads): PV over those only
                    return paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, true, kBlockN16, 1, true, 128>, 512, a, s, true)
                                  : launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, false, kBlockN16, 1, false, 128>, 512, a, s);
                return paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, true>, 512, a, s, true)
                              : launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, false, kBlockN16, 1, false>, 512, a, s);
            }
        }
        if (a.split_bm != 4 * kQueriesPerWave) return hipErrorInvalidValue;
        if (pair_split) return launch(flash_fwd_pair_split_kernel<T, D, MOD_PLAIN, 4>, 256, a, s, true);
        return paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 4, true>, 256, a, s, true)
             : a.num_splits > 1 ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 4, false>, 256, a, s)
                      : launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 4, false, kBlockN16, 1, false>, 256, a, s);
    } else {
        // score_mod: 64-key compute steps (two per staged tile at D = 32, 96, 160)
        constexpr int GSB = (D == 32 || (D & (D - 1)) != 0) ? 2 : 1;
        if (general_mod)
            return pair_split ? launch(flash_fwd_pair_split_kernel<T, D, MOD_GENERAL, 8, kBlockN16, GSB>, 512, a, s, true)
                 : paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, false, 8, true, kBlockN16, GSB>, 512, a, s, true)
                 : a.num_splits > 1 ? launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, false, 8, false, kBlockN16, GSB>, 512, a, s)
                          : launch(flash_fwd_lockstep_kernel<T, D, MOD_GENERAL, false, 8, false, kBlockN16, GSB, false>, 512, a, s);
        // D <= 64: 128-key tiles; D = 128: 128 keys staged per barrier, two 64-key compute steps
        constexpr int BN = D <= 64 ? kBlockN16Wide : kBlockN16;
        constexpr int SB = D <= 64 ? 1 : kBlockN16Wide / kBlockN16;
        if (pair_split) return launch(flash_fwd_pair_split_kernel<T, D, MOD_PLAIN, 8, BN, SB>, 512, a, s, true);
        return paired ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, true, BN, SB>, 512, a, s, true)
             : a.num_splits > 1 ? launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, false, BN, SB>, 512, a, s)
                      : launch(flash_fwd_lockstep_kernel<T, D, MOD_PLAIN, false, 8, false, BN, SB, false>, 512, a, s);
    }
}

// fp32 128-row query tiles: causal pairs without a block mask take the
// pairs-only instantiation. Above D = 128 a K/V tile is one block of 32 keys
// (two stages of 64-key tiles would not fit the LDS).
template <int D>
static hipError_t launch32(const FwdArgs& a, bool general_mod, hipStream_t s) {
    constexpr int NB = D > 128 ? 1 : kTilesF32;
    if (a.split_bn != kBlockNF32 * NB) return hipErrorInvalidValue;
    if (a.pair_split && a.tile_counts == nullptr)
        return general_mod ? launch(flash_fwd_mfma32_kernel<D, true, NB, true>, kThreads32, a, s, true)
                           : launch(flash_fwd_mfma32_kernel<D, false, NB, true>, kThreads32, a, s, true);
    return general_mod ? launch(flash_fwd_mfma32_kernel<D, true, NB>, kThreads32, a, s, a.pair_split != 0)
                       : launch(flash_fwd_mfma32_kernel<D, false, NB>, kThreads32, a, s, a.pair_split != 0);
}

hipError_t launch_flash_mfma(const FwdArgs& a, int dtype, bool general_mod, hipStream_t s) {
    // the kernel's head dim: D and Dv rounded up (the kernels zero-pad Q and
    // mask the stores past Dv)
    const int kd = flash_mfma_kernel_dim(dtype, a.D, a.Dv);
    if (dtype == DT_BF16 || dtype == DT_F16) {
        const bool f16 = dtype == DT_F16;
        switch (kd) {
            case 32: return f16 ? launch16<_Float16, 32>(a, general_mod, s) : launch16<__bf16, 32>(a, general_mod, s);
            case 64: return f16 ? launch16<_Float16, 64>(a, general_mod, s) : launch16<__bf16, 64>(a, general_mod, s);
            case 96: return f16 ? launch16<_Float16, 96>(a, general_mod, s) : launch16<__bf16, 96>(a, general_mod, s);
            case 128: return f16 ? launch16<_Float16, 128>(a, general_mod, s) : launch16<__bf16, 128>(a, general_mod, s);
            case 160: return f16 ? launch16<_Float16, 160>(a, general_mod, s) : launch16<__bf16, 160>(a, general_mod, s);
            case 192: return f16 ? launch16<_Float16, 192>(a, general_mod, s) : launch16<__bf16, 192>(a, general_mod, s);
            case 224: return f16 ? launch16<_Float16, 224>(a, general_mod, s) : launch16<__bf16, 224>(a, general_mod, s);
            case 256: return f16 ? launch16<_Float16, 256>(a, general_mod, s) : launch16<__bf16, 256>(a, general_mod, s);
            default: return hipErrorInvalidValue;
        }
    } else if (dtype == DT_F32) {
        if (a.split_bm == kRowsF32Narrow) {  // few query rows and keys: 16-row blocks, no key split
            if (a.tile_counts != nullptr || a.mask != nullptr || a.num_splits != 1) return hipErrorInvalidValue;
            switch (kd) {
                case 32: return general_mod ? launch(flash_fwd_f32_rows16_kernel<32, true>, kThreadsRows16, a, s)
                                            : launch(flash_fwd_f32_rows16_kernel<32, false>, kThreadsRows16, a, s);
                case 64: return general_mod ? launch(flash_fwd_f32_rows16_kernel<64, true>, kThreadsRows16, a, s)
                                            : launch(flash_fwd_f32_rows16_kernel<64, false>, kThreadsRows16, a, s);
                default: return hipErrorInvalidValue;
            }
        }
        if (a.split_bm == kRowsF32) {  // few query rows: 32-row blocks (no block mask)
            if (a.tile_counts != nullptr) return hipErrorInvalidValue;
            switch (kd) {
                case 32: return general_mod ? launch(flash_fwd_f32_rows32_kernel<32, true>, kThreads32, a, s)
                                            : launch(flash_fwd_f32_rows32_kernel<32, false>, kThreads32, a, s);
                case 64: return general_mod ? launch(flash_fwd_f32_rows32_kernel<64, true>, kThreads32, a, s)
                                            : launch(flash_fwd_f32_rows32_kernel<64, false>, kThreads32, a, s);
                case 96: return general_mod ? launch(flash_fwd_f32_rows32_kernel<96, true>, kThreads32, a, s)
                                            : launch(flash_fwd_f32_rows32_kernel<96, false>, kThreads32, a, s);
                case 128: return general_mod ? launch(flash_fwd_f32_rows32_kernel<128, true>, kThreads32, a, s)
                                             : launch(flash_fwd_f32_rows32_kernel<128, false>, kThreads32, a, s);
                default: return hipErrorInvalidValue;
            }
        }
        switch (kd) {
            case 32: return launch32<32>(a, general_mod, s);
            case 64: return launch32<64>(a, general_mod, s);
            case 96: return launch32<96>(a, general_mod, s);
            case 128: return launch32<128>(a, general_mod, s);
            case 160: return launch32<160>(a, general_mod, s);
            case 192: return launch32<192>(a, general_mod, s);
            case 224: return launch32<224>(a, general_mod, s);
            case 256: return launch32<256>(a, general_mod, s);
            default: break;
        }
    }
    return hipErrorInvalidValue;
}

hipError_t launch_combine_splits(const FwdArgs& a, int dtype, hipStream_t s) {
    const int chunks = a.Dv / 4;
    if (a.B * a.H * a.M <= 0 || chunks <= 0 || chunks > 256 || a.split_bm <= 0) return hipErrorInvalidValue;
    // splits per row read in parallel: a thread keeps four splits' loads in
    // flight, so a group is added only while each would read more than four
    // (up to 8 groups: two rounds of four loads per thread for 64 splits);
    // rows per workgroup: a power of two dividing the query tile, with
    // rows * chunks * groups <= 256
    int groups = 1;
    while (groups < 8 && 4 * groups < a.num_splits && 2 * groups * chunks <= 256) groups *= 2;
    int rows = 1;
    while (2 * rows * chunks * groups <= 256 && 2 * rows <= a.split_bm && a.split_bm % (2 * rows) == 0) rows *= 2;
    const int64_t nblk = (int64_t)a.B * a.H * ((a.M + rows - 1) / rows);
    if (nblk > 0x7fffffff) return hipErrorInvalidValue;
    const dim3 grid((unsigned)nblk);
    if (dtype == DT_F32 || a.out_f32) hipLaunchKernelGGL(combine_splits_kernel<float>, grid, dim3(256), 0, s, a, rows, groups);
    else if (dtype == DT_BF16) hipLaunchKernelGGL(combine_splits_kernel<__bf16>, grid, dim3(256), 0, s, a, rows, groups);
    else if (dtype == DT_F16) hipLaunchKernelGGL(combine_splits_kernel<_Float16>, grid, dim3(256), 0, s, a, rows, groups);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

namespace {
// Arrival counters of the single-launch key-split merge (see FwdArgs).
static __device__ __align__(256) unsigned split_counters[kSplitCounterSlots * kMaxSplitTiles];
std::mutex g_counter_mu;
std::map<int, unsigned*> g_counter_addr;  // device -> address of its copy of split_counters
}  // namespace

hipError_t split_counter_slot(int slot, unsigned** ptr) {
    if (slot < 0 || slot >= kSplitCounterSlots) return hipErrorInvalidValue;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(g_counter_mu);
    auto it = g_counter_addr.find(dev);
    if (it == g_counter_addr.end()) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(split_counters));
        if (e != hipSuccess) return e;
        it = g_counter_addr.emplace(dev, static_cast<unsigned*>(p)).first;
    }
    *ptr = it->second + (size_t)slot * kMaxSplitTiles;
    return hipSuccess;
}

bool flash_mfma_head_dim(int dtype, int D) {
    (void)dtype;  // every dtype: multiples of 32 up to 256
    return D % 32 == 0 && D >= 32 && D <= 256;
}

int flash_mfma_kernel_dim(int dtype, int D, int Dv) {
    const int unit = dtype == DT_F32 ? 4 : 8;  // elements per 16-byte row chunk
    if (D <= 0 || Dv <= 0 || D % unit != 0 || Dv % unit != 0) return 0;
    const int kd = (std::max(D, Dv) + 31) / 32 * 32;
    return flash_mfma_head_dim(dtype, kd) ? kd : 0;
}

const char* flash_mfma_kernel_name(int dtype, int D, bool general_mod, bool tile_list, int threads) {
    if (dtype < 0 || dtype > 2 || !flash_mfma_head_dim(dtype, D)) return "none";
    // [dtype][D / 32 - 1][score_mod][list][8 wavefronts]
    static const std::vector<std::string> names = [] {
        std::vector<std::string> v;
        const char* tn[3] = {"f32", "bf16", "f16"};
        for (int dt = 0; dt < 3; ++dt)
            for (int d = 32; d <= 256; d += 32)
                for (int mod = 0; mod < 2; ++mod)
                    for (int list = 0; list < 2; ++list)
                        for (int w8 = 0; w8 < 2; ++w8) {
                            std::string n;
                            if (dt == DT_F32) {
                                n = "flash_fwd_mfma32_kernel<" + std::to_string(d) + (mod ? ",general>" : ",plain>");
                            } else {
                                n = std::string("flash_fwd_lockstep_kernel<") + tn[dt] + "," + std::to_string(d) +
                                    (mod ? ",mod" : ",plain");
                                const bool pow2 = (d & (d - 1)) == 0;
                                if (list) n += ",list,4w>";
                                else if (d == 192 && !mod && w8) n += ",8w>";
                                else if (d == 256 && !mod && w8) n += ",8w,2x32keys>";
                                else if (d > 160) n += ",4w>";
                                else if (!mod && d <= 64) n += ",8w,128keys>";
                                else if (!mod) n += ",8w,2x64keys>";
                                else if (d == 32 || !pow2) n += ",8w,2x64keys>";
                                else n += ",8w>";
                            }
                            v.push_back(n);
                        }
        return v;
    }();
    const int di = D / 32 - 1;
    return names[((((size_t)dtype * 8 + di) * 2 + (general_mod ? 1 : 0)) * 2 + (tile_list ? 1 : 0)) * 2 +
                 (threads >= 512 ? 1 : 0)]
        .c_str();
}

MfmaTiles flash_mfma_tiles(int dtype, int D, bool general_mod, bool tile_list, bool causal, int64_t bh,
                           int64_t query_tokens) {
    if (dtype == DT_F32) return MfmaTiles{kBlockM32, kBlockNF32 * (D > 128 ? 1 : kTilesF32), kThreads32, false};
    const bool paired = pairs_causal_tiles(causal, tile_list);
    const int bn = block_n16(D, general_mod, tile_list);
    const bool four =
        tile_list || (D > 160 && !((D == 192 || D == 256) && !general_mod && eight_waves_wide(causal, bh, query_tokens)));
    if (four) return MfmaTiles{128, bn, 256, paired};
    return MfmaTiles{256, bn, 512, paired};
}

}  // namespace ofh
