// 16-bit attention forward for calls whose 256-row query tiles do not fill the
// GPU (one prompt of a few thousand tokens, small batches): the eight
// wavefronts of a workgroup share fewer query rows and split the keys among
// themselves.
//
// A workgroup takes R = 8 / KS row slices of 32 query rows; KS wavefronts work
// on a slice, each on its own BN keys of every staged K/V tile (KS BN keys,
// copied global -> LDS as in the lockstep kernel), and their (m, l, O) are
// folded in LDS at the end. Against 256-row tiles with the keys split over
// workgroups this gives the same number of wavefronts per CU without partial
// rows in memory, a merge launch or a long chain for the last causal tile: a
// tile's chain is 1/KS as long, and KS times as many tiles spread over the CUs.
// The price is KS times the K/V copies per query row. It is bound by what a
// step of 32 rows x 64 keys takes a SIMD (about 1.05 us: 32 MFMAs and the
// softmax one after the other) times the longest chain. Measured (us, split
// 256-row tiles -> this): bf16 causal H32 D128 N512 25.8 -> 13.3, N1000 42.7 ->
// 23.2, N1500 54 -> 45; H128 N512 54.6 -> 32.7; D64 H16 N1500 non-causal 28.7 ->
// 21.0. With a score_mod: ALiBi + soft-cap H32 D128 N512 26.2 -> 15.1 causal,
// N1000 44.5 -> 30.8 non-causal; shared bias H16 D64 N1000 30.7 -> 18.8. (A dense
// bias is read by the lanes here: its LDS tiles would not fit beside four
// groups' keys.) Asking for a head's K and V rows ahead (one load per line at the start)
// gained 0-3 % up to N1500, so it is not done.

#include "flash_wave32.h"
#include "ofh_kernels.h"

namespace ofh {
namespace {

constexpr int kGroupThreads = 512;

// Keys per wavefront and staged tile: 64 where KS * 64 staged keys fit twice
// into the LDS, else 32.
constexpr int group_keys(int D, int KS) { return KS == 4 && D > 64 ? 32 : 64; }

template <typename T, int D, int KS, int MOD>
__global__ __launch_bounds__(kGroupThreads, 1) void flash_fwd_keygroups_kernel(FwdArgs a) {
    constexpr int BN = group_keys(D, KS);
    constexpr int R = 8 / KS;
    using W = Wave32<T, D, MOD, false, kGroupThreads, BN, KS>;
    using L = typename W::L;
    constexpr int NDB = D / 32;
    constexpr int kStateFloats = NDB * 16 + 4;        // O, m, l of a lane (padded to 16 bytes)
    constexpr int kStateBytes = 64 * 4 * kStateFloats;
    static_assert((8 - R) * kStateBytes <= 2 * L::STAGE, "the folded states fit the LDS stages");
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * L::STAGE];
    int bh, qt;
    map_work((int)blockIdx.x, a.B * a.H, a.num_q_tiles, a.causal, bh, qt);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slice = wave % R, kg = wave / R;
    const int q0 = qt * R * kQueriesPerWave;
    const int kend = a.causal ? min(a.N, q0 + R * kQueriesPerWave) : a.N;
    const int nst = (kend + W::SN - 1) / W::SN;
    W w(a, smem, bh, q0 + (slice - wave) * kQueriesPerWave, wave);  // rows q0 + 32 slice ..
    w.copy_tile(0, 0);
    wait_vm_loads();
    w.zero_tail(0, 0);
    __syncthreads();
    for (int st = 0; st < nst; ++st) {
        const int stage = (st & 1) * L::STAGE;
        const int nstage = ((st + 1) & 1) * L::STAGE;
        if (st + 1 < nst) w.copy_tile(st + 1, nstage);
        const int e = st * KS + kg;  // this wavefront's BN keys
        if (e * BN < kend && w.tile_active(e)) {
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
            w.qk(stage, kg);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
            w.softmax(e);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(1);
            w.pv(stage, kg);
            if (MOD == MOD_PLAIN) __builtin_amdgcn_s_setprio(0);
        }
        wait_vm_loads();
        if (st + 1 < nst) w.zero_tail(st + 1, nstage);
        __syncthreads();
    }

    // Fold the states of the slice's wavefronts into key group 0's.
    const int lane = threadIdx.x & 63;
    if (kg > 0) {
        float* st = (float*)(smem + (wave - R) * kStateBytes);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                *(f32x4*)(st + 4 * (64 * (4 * db + c) + lane)) =
                    f32x4{w.o[db][4 * c], w.o[db][4 * c + 1], w.o[db][4 * c + 2], w.o[db][4 * c + 3]};
        *(f32x4*)(st + 4 * (64 * 4 * NDB + lane)) = f32x4{w.m_run, w.l_run, 0.f, 0.f};
    }
    __syncthreads();
    if (kg == 0) {
        f32x4 ml[KS];
        float mg = w.m_run;
#pragma unroll
        for (int k = 1; k < KS; ++k) {
            ml[k] = *(const f32x4*)(smem + ((k - 1) * R + slice) * kStateBytes + 16 * (64 * 4 * NDB + lane));
            mg = fmaxf(mg, ml[k][0]);
        }
        const float mu = mg == kNegInf ? 0.0f : mg;
        const float w0 = __builtin_amdgcn_exp2f(w.m_run - mu);  // 0 for a group without a valid key
        w.l_run *= w0;
        w.m_run = mg;
#pragma unroll
        for (int db = 0; db < NDB; ++db) w.o[db] *= w0;
#pragma unroll
        for (int k = 1; k < KS; ++k) {
            const float wk = __builtin_amdgcn_exp2f(ml[k][0] - mu);
            w.l_run += wk * ml[k][1];
            const unsigned char* st = smem + ((k - 1) * R + slice) * kStateBytes;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const f32x4 v = *(const f32x4*)(st + 16 * (64 * (4 * db + c) + lane));
#pragma unroll
                    for (int j = 0; j < 4; ++j) w.o[db][4 * c + j] += wk * v[j];
                }
        }
        w.store_output();
    }
}

template <typename T, int D, int MOD>
hipError_t launch_groups_mod(const FwdArgs& a, int groups, hipStream_t s) {
    const dim3 grid((unsigned)((int64_t)a.B * a.H * a.num_q_tiles)), block(kGroupThreads);
    if (groups == 2) hipLaunchKernelGGL((flash_fwd_keygroups_kernel<T, D, 2, MOD>), grid, block, 0, s, a);
    else if (groups == 4) hipLaunchKernelGGL((flash_fwd_keygroups_kernel<T, D, 4, MOD>), grid, block, 0, s, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
template <typename T, int D>
hipError_t launch_groups(const FwdArgs& a, int groups, hipStream_t s) {
    return a.bias_kind != BIAS_NONE || a.softcap > 0.0f ? launch_groups_mod<T, D, MOD_GENERAL>(a, groups, s)
                                                        : launch_groups_mod<T, D, MOD_PLAIN>(a, groups, s);
}

}  // namespace

int key_group_keys(int D, int groups) { return groups * group_keys(D, groups); }

hipError_t launch_key_groups(const FwdArgs& a, int dtype, int groups, hipStream_t s) {
    const int kd = flash_mfma_kernel_dim(dtype, a.D, a.Dv);
    if (a.split_bm * groups != 8 * kQueriesPerWave || a.split_bn != key_group_keys(kd, groups) || a.mask != nullptr ||
        a.num_splits != 1)
        return hipErrorInvalidValue;
    const bool f16 = dtype == DT_F16;
    switch (kd) {
        case 32: return f16 ? launch_groups<_Float16, 32>(a, groups, s) : launch_groups<__bf16, 32>(a, groups, s);
        case 64: return f16 ? launch_groups<_Float16, 64>(a, groups, s) : launch_groups<__bf16, 64>(a, groups, s);
        case 96: return f16 ? launch_groups<_Float16, 96>(a, groups, s) : launch_groups<__bf16, 96>(a, groups, s);
        case 128: return f16 ? launch_groups<_Float16, 128>(a, groups, s) : launch_groups<__bf16, 128>(a, groups, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ofh
