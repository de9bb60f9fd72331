// 16-bit attention forward with a dense fp32 bias (with or without a soft-cap)
// and no block mask: the lockstep schedule of flash_fwd_mfma.hip with the bias
// staged through LDS.
//
// What bounds such calls: a bias tile read by the score_mod kernel's lanes sits
// behind the next K/V tile's copies in the in-order memory counter, so every
// step waited for those copies and for the bias's own latency, and a 16-byte
// read per lane touched 32 rows. Here each wavefront copies the bias of its 32
// rows x 64 keys global -> LDS itself, whole 256-byte row pieces, right after
// its softmax has read the previous one (8 KB per wavefront, no barrier and no
// registers), so the copy has a whole step to land. Without a soft-cap the
// scores stay in natural units (one multiply less per score) and D <= 64 takes
// the row-sum bound of Wave32::softmax.
//
// Measured (us, score_mod kernel -> this): fp16 B2 H16 N2048 D64, shared bias
// 104.5 -> 67.2 (a bias per head, 537 MB of it: 141 -> 126, 4.3 TB/s), causal 78.7
// -> 57.7; D32 B4 H16 N1024 41.8 -> 28.6; D128 H16 N4096 218 -> 178. Rows that
// are not 16-byte aligned would need four times the copies, 4 bytes per lane:
// built and measured within 15 % of the score_mod kernel on either side (N2047
// D64 107 -> 94, causal H96 N1767 D128 192 -> 225), so they stay there.

#include "flash_wave32.h"
#include "ofh_kernels.h"
#include "split_merge.h"

namespace ofh {
namespace {

constexpr int kBiasWaves = 8;
constexpr int kBiasThreads = kBiasWaves * 64;

// 64-key compute steps; two per staged tile where a 64-key tile would not
// split evenly over the eight wavefronts (as in the score_mod kernel).
constexpr int bias_steps(int D) { return D == 32 || D == 96 ? 2 : 1; }

template <typename T, int D, bool SPLIT>
__device__ __forceinline__ void bias_qtile(const FwdArgs& a, unsigned char* smem, int bh, int qt, int split) {
    constexpr int BN = kBlockN16, SB = bias_steps(D);
    constexpr int BLOCK_M = kBiasWaves * kQueriesPerWave;
    using W = Wave32<T, D, MOD_DENSE, false, kBiasThreads, BN, SB>;
    using L = typename W::L;
    constexpr int COPIES = 2 * W::CPT;  // K and V copies of a wavefront per staged tile
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q0 = qt * BLOCK_M;
    const int kend = a.causal ? min(a.N, q0 + BLOCK_M) : a.N;
    const int nst = (kend + W::SN - 1) / W::SN;
    const int active = SPLIT ? split_active(a, nst) : 1;
    if (split >= active) return;  // uniform over the workgroup
    const int range = SPLIT ? split_range(a, nst) : nst;
    const int st0 = SPLIT ? split * range : 0;
    const int st1 = SPLIT ? min(nst, st0 + range) : nst;
    W w(a, smem, bh, q0, wave);
    w.bias_lds = 2 * L::STAGE + wave * W::BIAS_BYTES;
    if (st0 >= st1) {  // uniform over the workgroup
        finish_qtile<W, kBiasThreads, SPLIT>(a, w, smem, bh, qt, q0, BLOCK_M, split, active);
        return;
    }
    const int e1 = min(st1 * SB, (kend + BN - 1) / BN);  // compute steps [st0 SB, e1)
    w.copy_tile(st0, 0);
    w.copy_bias(st0 * SB);
    wait_vm_loads();
    w.zero_tail(st0, 0);
    __syncthreads();
    for (int st = st0; st < st1; ++st) {
        const int stage = ((st - st0) & 1) * L::STAGE;
        const int nstage = ((st - st0 + 1) & 1) * L::STAGE;
        if (st + 1 < st1) w.copy_tile(st + 1, nstage);
        bool bias_pending = false;  // a bias copy younger than this step's K/V copies (uniform per wavefront)
#pragma unroll
        for (int j = 0; j < SB; ++j) {
            const int e = st * SB + j;
            if (e < e1 && w.tile_active(e)) {
                w.qk(stage, j);
                // the bias of this step has landed; the next tile's K/V copies may still be in flight
                if (j == 0 && st + 1 < st1) wait_vm<COPIES>();
                else wait_vm_loads();
                w.softmax(e);
                bias_pending = false;
                if (e + 1 < e1 && w.tile_active(e + 1)) {
                    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the softmax has read its bias
                    w.copy_bias(e + 1);
                    bias_pending = true;
                }
                w.pv(stage, j);
            }
        }
        // the K/V copies have landed; the next step's bias may still be in flight
        if (!bias_pending) wait_vm_loads();
        else wait_vm<8>();
        if (st + 1 < st1) w.zero_tail(st + 1, nstage);
        __syncthreads();
    }
    finish_qtile<W, kBiasThreads, SPLIT>(a, w, smem, bh, qt, q0, BLOCK_M, split, active);
}

// MODE 0: a query tile (and key split) per workgroup; 1: causal pairs of query
// tiles; 2: causal pairs, each tile split in ranges of its own length.
template <typename T, int D, int MODE>
__global__ __launch_bounds__(kBiasThreads, 1) void flash_fwd_bias_kernel(FwdArgs a) {
    using W = Wave32<T, D, MOD_DENSE, false, kBiasThreads, kBlockN16, bias_steps(D)>;
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * W::L::STAGE + kBiasWaves * W::BIAS_BYTES];
    int bh, qts[2];
    if constexpr (MODE == 0) {
        const int tiles = a.B * a.H * a.num_q_tiles;
        const int split = (int)blockIdx.x / tiles;
        map_work((int)blockIdx.x - split * tiles, a.B * a.H, a.num_q_tiles, a.causal, bh, qts[0]);
        bias_qtile<T, D, true>(a, smem, bh, qts[0], split);
    } else {
        const int pairs = a.B * a.H * ((a.num_q_tiles + 1) / 2);
        const int split = MODE == 2 ? (int)blockIdx.x / pairs : 0;
        map_work_pair((int)blockIdx.x - split * pairs, a.B * a.H, a.num_q_tiles, bh, qts[0], qts[1]);
        bias_qtile<T, D, MODE == 2>(a, smem, bh, qts[0], split);
        if (qts[1] >= 0) {
            __syncthreads();  // LDS stages are reused
            bias_qtile<T, D, MODE == 2>(a, smem, bh, qts[1], split);
        }
    }
}

template <typename T, int D>
hipError_t launch_bias_d(const FwdArgs& a, hipStream_t s) {
    const bool paired = a.pair_split != 0 || (a.causal && a.num_splits == 1);
    const int64_t tiles = paired ? (a.num_q_tiles + 1) / 2 : a.num_q_tiles;
    const dim3 grid((unsigned)((int64_t)a.B * a.H * tiles * a.num_splits)), block(kBiasThreads);
    if (a.pair_split) hipLaunchKernelGGL((flash_fwd_bias_kernel<T, D, 2>), grid, block, 0, s, a);
    else if (paired) hipLaunchKernelGGL((flash_fwd_bias_kernel<T, D, 1>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((flash_fwd_bias_kernel<T, D, 0>), grid, block, 0, s, a);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_bias_t(const FwdArgs& a, int kd, hipStream_t s) {
    switch (kd) {
        case 32: return launch_bias_d<T, 32>(a, s);
        case 64: return launch_bias_d<T, 64>(a, s);
        case 96: return launch_bias_d<T, 96>(a, s);
        case 128: return launch_bias_d<T, 128>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace

hipError_t launch_bias(const FwdArgs& a, int dtype, hipStream_t s) {
    const int kd = flash_mfma_kernel_dim(dtype, a.D, a.Dv);
    if (a.mask != nullptr || a.bias_kind != BIAS_DENSE || a.split_bm != kBiasWaves * kQueriesPerWave ||
        !bias_can_be_staged(a.bias, a.N, a.bias_sb, a.bias_sh, a.bias_sm))
        return hipErrorInvalidValue;
    return dtype == DT_F16 ? launch_bias_t<_Float16>(a, kd, s) : launch_bias_t<__bf16>(a, kd, s);
}

}  // namespace ofh
