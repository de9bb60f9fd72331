// Device code of one wavefront of the 16-bit attention kernels: 32 query rows
// against K/V tiles staged in LDS (see flash_fwd_mfma.hip for the layout of the
// products), shared by the kernels that arrange such wavefronts differently.
// Internal header, included by the HIP translation units.
#pragma once

#include "ofh_kernels.h"
#include "split_merge.h"

namespace ofh {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr float kLog2e = 1.4426950408889634f;

// s_waitcnt vmcnt(N): at most N vector-memory operations still outstanding
// (they complete in issue order, so every older one has completed).
template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

__device__ __forceinline__ int kappa(int r) {
    return ((r >> 4) << 4) | (((r >> 2) & 1) << 3) | (((r >> 3) & 1) << 2) | (r & 3);
}

// Position (within a 32-row block) held by accumulator register e of lane half g.
__device__ __forceinline__ int acc_pos(int e, int g) { return ((e >> 3) << 4) + (g << 3) + (e & 7); }

template <typename T>
struct Mfma16;
template <>
struct Mfma16<__bf16> {
    typedef bf16x8 v8;
    static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Mfma16<_Float16> {
    typedef f16x8 v8;
    static __device__ __forceinline__ f32x16 mma(v8 a, v8 b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

// Workgroup id -> (flat head, query tile). Workgroups are handed to the 8 XCDs
// round-robin, so when B*H is a multiple of 8 the heads are partitioned over
// XCDs (all query tiles of a head run on one XCD and share its L2 for K/V),
// and each XCD walks its heads one after another. Causal query tiles run
// heaviest (longest key range) first.
__device__ __forceinline__ void map_work(int id, int BH, int nqt, int causal, int& bh, int& qt) {
    int t;
    if ((BH & 7) == 0) {
        const int xcd = id & 7, j = id >> 3;
        const int hl = j / nqt;
        t = j - hl * nqt;
        bh = hl * 8 + xcd;
    } else {
        bh = id % BH;
        t = id / BH;
    }
    qt = causal ? nqt - 1 - t : t;
}

// Causal attention without a block mask: workgroup id -> (flat head, query
// tiles nqt-1-p and p). The heavy tile runs first, then the light one, so
// every workgroup does the same number of tile steps (no tail of short
// workgroups) and both tiles share the head's K/V in one XCD's L2. qt_b is
// -1 when p is the middle tile of an odd count.
__device__ __forceinline__ void map_work_pair(int id, int BH, int nqt, int& bh, int& qt_a, int& qt_b) {
    const int np = (nqt + 1) / 2;
    int p;
    if ((BH & 7) == 0) {
        const int xcd = id & 7, j = id >> 3;
        const int hl = j / np;
        p = j - hl * np;
        bh = hl * 8 + xcd;
    } else {
        bh = id % BH;
        p = id / BH;
    }
    qt_a = nqt - 1 - p;
    qt_b = (p != qt_a) ? p : -1;
}

// Query tiles of this workgroup: one, or a causal pair (see map_work_pair).
__device__ __forceinline__ int work_tiles(const FwdArgs& a, bool paired, int& bh, int (&qts)[2]) {
    if (paired) {
        map_work_pair(blockIdx.x, a.B * a.H, a.num_q_tiles, bh, qts[0], qts[1]);
        return qts[1] >= 0 ? 2 : 1;
    }
    map_work(blockIdx.x, a.B * a.H, a.num_q_tiles, a.causal, bh, qts[0]);
    return 1;
}

// ---------------------------------------------------------------------------
// bf16 / fp16 inputs, fp32 accumulate: v_mfma_f32_32x32x16_{bf16,f16}.
//
// Every wavefront owns 32 query rows. K/V tiles are staged one tile ahead
// by global_load_lds_dwordx4 copies straight into LDS (no staging registers,
// no LDS store instructions). With the plain scale and no block mask a
// staged tile is 128 keys (two 64-key compute steps at D=128), otherwise 64.
// Loads are unconditional: rows past the end are clamped to the last row,
// their V zeroed and their scores masked, so no exec-masked branch breaks
// the compiler's wait counting.
//
// LDS layout (TileLayout): both tiles row-major [key][d], unpadded, with the
// 16-byte chunks of a row XOR-swizzled so that the K A-operand reads
// (ds_read_b128) and the V reads (ds_read_b64_tr_b16, which deliver V^T
// fragments directly, so V is never transposed in a separate pass) are free
// of bank conflicts at one XOR per read.
//
// Workgroup schedule (every 16-bit call): lockstep. All wavefronts run S,
// softmax and PV of a tile between two barriers; double-buffered LDS.
// Without a block-mask list the workgroup has 8 wavefronts (256 query rows);
// with one it has 4 (128 rows), which wastes fewer partial tiles on fine
// masks.
//
// Online softmax with lazy rescaling: the running max m that probabilities
// are taken against is raised only when a tile's max exceeds it by more than
// kRescaleSlack (log2 units), so p <= 2^8 and the O/l rescale (a wave-uniform
// branch) runs on a few tiles per row instead of every tile. The result is
// exact in real arithmetic: O and l share the same stale max.

constexpr int kBlockN16 = 64;      // keys per K/V tile (16-bit kernels) ...
constexpr int kBlockN16Wide = 128; // ... and for D = 64 without score_mod or block mask
constexpr float kRescaleSlack = 8.0f;
constexpr float kSumBound = 256.0f;  // 2^kRescaleSlack
constexpr int kFragAhead = 4;  // LDS fragment reads in flight ahead of the MFMAs (plain scale)

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef short i16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
typedef __attribute__((address_space(3))) unsigned char lds_u8;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

// Score modification of a 16-bit kernel instantiation: the plain scale, or
// any mix of ALiBi / dense bias / soft-cap selected per call.
// MOD_DENSE: a dense bias (with or without a soft-cap) whose tiles are copied
// to LDS ahead of their use (flash_bias.hip).
enum ScoreMod { MOD_PLAIN = 0, MOD_GENERAL = 1, MOD_DENSE = 2 };


// One 16-byte global -> LDS copy per lane (lane L writes lds + 16 L; lds is
// wave-uniform). Written as assembly so that the compiler does not make LDS
// reads of the other stage wait for it; completion is awaited explicitly
// (wait_vm_loads) before the barrier that publishes the tile. M0 is restored.
__device__ __forceinline__ void dma16(const void* g, unsigned lds) {
    unsigned save;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
                 : "=&s"(save) : "v"(g), "s"(lds) : "memory");
}

// The same from a wave-uniform base plus a per-lane byte offset.
__device__ __forceinline__ void dma16s(const void* base, unsigned off, unsigned lds) {
    unsigned save;
    asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
                 : "=&s"(save) : "v"(off), "s"(base), "s"(lds) : "memory");
}
// K and V tiles in LDS: row-major [key][d], unpadded (each global -> LDS
// copy instruction writes 1 KB of consecutive LDS). Chunk c (16 bytes) of row
// r sits at position c ^ kswz(r) (K) or c ^ vswz(r) (V), which keeps both
// read patterns free of bank conflicts (measured with SQ_LDS_BANK_CONFLICT):
// K fragments read rows kappa(0..15) at one chunk per 16 lanes; V^T fragments
// are transposing reads of 4 rows x 2 chunks per 16 lanes. For D = 64 two rows
// share a 256-byte bank line, hence row >> 1.
//
// Head dims that are not powers of two (96, 160, 192, 224) XOR only inside
// aligned groups of chunks that divide the row (see kswz), and their reads add
// per-lane bases to compile-time offsets instead of XORing the address.
template <int D, int BN>
struct TileLayout {
    static constexpr int RB = D * 2;              // bytes of one K/V row
    static constexpr int CPR = D / 8;             // 16-byte chunks per row
    static constexpr bool POW2 = (D & (D - 1)) == 0;
    static_assert(D % 32 == 0 && D >= 32 && D <= 256, "head dims of the 16-bit kernels: multiples of 32 up to 256");
    // Both swizzles must repeat every 8 rows or less at D = 256 (every 16 at
    // D = 128, 32 at D = 64, 64 at D = 32): a copy lane reuses one swizzled
    // chunk offset for the rows DSTEP = 64 * wavefronts / CPR apart that it
    // copies (8 rows with 4 wavefronts at D = 256). The V swizzle must also
    // repeat every 4 rows: a V^T fragment is two transposing reads 4 rows
    // apart at one lane offset.
    //
    // Rows that are not a power of two wide (D = 96, 160, 192, 224): a
    // 16-byte K read serves 16 lanes at a time, rows kappa(0..15) at one
    // chunk, and with 12, 20 or 28 chunks per row those rows start on only 4
    // distinct 16-byte bank groups (2 at 24 chunks). The chunk index is XORed
    // inside aligned groups of KG chunks (KG divides the row): by (row>>2)&3
    // (KG = 4), so the 16 rows cover the 16 bank groups, or by (row>>1)&7 at
    // D = 192 (KG = 8). A V^T read serves rows 4 apart in 64-byte runs, which
    // already fall on distinct banks except at D = 192 (rows 384 bytes apart):
    // there chunks are XORed with 4 on (row>>1)&1.
    static constexpr int KG = POW2 ? 1 : (D == 192 ? 8 : 4);
    static_assert(POW2 || CPR % KG == 0, "the K swizzle group divides the row");
    static __device__ __forceinline__ int kswz(int row) {
        if (!POW2) return D == 192 ? (row >> 1) & 7 : (row >> 2) & 3;
        if (D == 256) return row & 7;
        if (D == 128) return row & 15;
        if (D == 64) return (row >> 1) & 7;
        return (row >> 2) & 3;  // D = 32: four rows share a bank line
    }
    static __device__ __forceinline__ int vswz(int row) {
        if (!POW2) return D == 192 ? 4 * ((row >> 1) & 1) : 0;
        if (D >= 128) return 4 * (row & 3);
        if (D == 64) return 4 * ((row >> 1) & 1);
        return 0;  // D = 32: a row is one 32-column block
    }
    static constexpr int KSTR = RB;
    static constexpr int VSTR = RB;
    static constexpr int KTILE = BN * KSTR;
    static constexpr int VTILE = BN * VSTR;
    static constexpr int STAGE = KTILE + VTILE;   // K tile then V tile
};

// max over both 32-lane halves (lane l and l^32 hold the same query row)
__device__ __forceinline__ float half_swap_max(float x) {
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, x),
                                                    __builtin_bit_cast(unsigned, x), false, false);
    return fmaxf(__builtin_bit_cast(float, (unsigned)r[0]), __builtin_bit_cast(float, (unsigned)r[1]));
}

template <typename T>
struct Dot2;
template <>
struct Dot2<__bf16> {
    typedef __bf16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ float sum2(v2 a, float acc) {
        return __builtin_amdgcn_fdot2_f32_bf16(a, v2{(__bf16)1.0f, (__bf16)1.0f}, acc, false);
    }
};
template <>
struct Dot2<_Float16> {
    typedef _Float16 v2 __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ float sum2(v2 a, float acc) {
        return __builtin_amdgcn_fdot2(a, v2{(_Float16)1.0f, (_Float16)1.0f}, acc, false);
    }
};

// Position of accumulator register e of sub-block sb within a 64-key tile,
// relative to the lane half's first key (8g): 32sb + 16(e>>3) + (e&7).
__device__ __forceinline__ constexpr int tile_pos(int sb, int e) { return 32 * sb + 16 * (e >> 3) + (e & 7); }

// The per-wavefront state and the tile operations of one 32-row wavefront.
// A "tile step" is identified by its entry: the key tile index, or with a
// block-mask list (LIST) the list entry (key tile + per-slice bits).
template <typename T, int D, int MOD, bool LIST, int NTHREADS, int BN_, int SB = 1, int DVK = D>
struct Wave32 {
    // DVK: value columns the kernel computes (a multiple of 32 up to D; O and
    // PV cover only those, the K side and the LDS rows stay D wide)
    static_assert(DVK % 32 == 0 && DVK <= D, "value columns: a multiple of 32 up to D");
    using T_ = T;
    using M16 = Mfma16<T>;
    using v8 = typename M16::v8;
    // K/V staged by global -> LDS copies in every kernel without a block-mask
    // list (register staging with one)
    using L = TileLayout<D, BN_ * SB>;
    static constexpr int BN = BN_;
    static constexpr int SN = BN_ * SB;                 // keys per staged tile
    static constexpr int CPT = SN * L::CPR / NTHREADS;  // 16-byte chunks per thread per tile
    static_assert(CPT >= 1 && SN * L::CPR % NTHREADS == 0, "tile must split evenly");

    const FwdArgs& a;
    unsigned char* smem;
    const T* Kp;
    const T* Vp;
    int tid, g, h, b, wave;
    int qw0, my_q;
    int ntiles;
    const int* list;
    v8 qf[D / 16];
    f32x16 o[DVK / 32];
    f32x16 s[BN / 32];
    v8 pf[BN / 16];
    float m_run, l_run;
    float slope;
    float alibi_step[8];  // soft-capped ALiBi: 2^(slope c_b t), t = 0..7 (wave-uniform)
    const float* bias_row;  // this lane's row; MOD_DENSE: the head's first row
    int bias_lds;           // MOD_DENSE: LDS offset of this wavefront's bias rows
    // LDS read lane offsets
    int k_lane_off, v_lane_off;
    // rows that are not a power of two wide: per-lane bases of the swizzled
    // chunk pairs (K) and 32-column blocks (V at D = 192), the rest of the
    // offset is a compile-time immediate
    int k_base[L::POW2 ? 1 : L::KG / 2];
    int v_base[L::POW2 ? 1 : 2];
    // K/V copies: lane offsets (elements) of its chunk in rows dma_row0 + u*DSTEP
    // when a copy instruction covers whole rows (64 * wavefronts divisible by
    // the chunks per row: every power-of-two D); otherwise each instruction's
    // row and chunk are derived from its slot index.
    static constexpr bool UNIFORM_COPY = (64 * (NTHREADS / 64)) % L::CPR == 0;
    static constexpr int DSTEP = UNIFORM_COPY ? 64 * (NTHREADS / 64) / L::CPR : 0;
    static_assert(!UNIFORM_COPY || !L::POW2 ||
                      DSTEP % (D == 256 ? 8 : D == 128 ? 16 : D == 64 ? 32 : 64) == 0,
                  "the K/V swizzles must repeat within the rows one copy lane covers");
    static_assert(UNIFORM_COPY || !L::POW2, "power-of-two rows are copied by whole-row instructions");
    static_assert(L::POW2 || !UNIFORM_COPY, "rows that are not a power of two wide are copied slot by slot");
    int dma_row0, dma_koff, dma_voff;
    // K fragment c (chunks 2c, 2c+1) and V^T block db at the lane's read offsets
    __device__ __forceinline__ int k_off(int c) const {
        if constexpr (L::POW2) return k_lane_off ^ (32 * c);
        // chunk (2c + g) ^ s = (2c & ~(KG-1)) + ((2c & (KG-1)) ^ (g ^ s))
        else return k_base[c % (L::KG / 2)] + 16 * ((2 * c) & ~(L::KG - 1));
    }
    __device__ __forceinline__ int v_off(int db) const {
        if constexpr (L::POW2) return v_lane_off ^ (64 * db);
        else if constexpr (D == 192) return v_base[db & 1] + 64 * (db & ~1);
        else return v_lane_off + 64 * db;
    }

    __device__ __forceinline__ Wave32(const FwdArgs& args, unsigned char* sm, int bh, int q0, int wv)
        : a(args), smem(sm), wave(wv) {
        tid = threadIdx.x;
        const int lane = tid & 63;
        g = lane >> 5;
        const int r = lane & 31;
        b = bh / a.H;
        h = bh - b * a.H;
        const T* Qp = (const T*)a.q + b * a.q_sb + h * a.q_sh;
        Kp = (const T*)a.k + b * a.k_sb + h * a.k_sh;
        Vp = (const T*)a.v + b * a.v_sb + h * a.v_sh;
        qw0 = q0 + wave * kQueriesPerWave;
        my_q = qw0 + r;
        // Q^T fragments (B operand of S^T = K Q^T): lane holds Q[my_q][16c + 8g .. +7].
        // Rows past the end read the last row; their results are never stored.
        // Columns at or past a.D (the kernel's D is the head dim rounded up) are zero.
        const T* qrow = Qp + (int64_t)min(my_q, a.M - 1) * a.q_sm + 8 * g;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) {
            u32x4 u = {0u, 0u, 0u, 0u};
            if (16 * c + 8 * g < a.D) u = *(const u32x4*)(qrow + 16 * c);
            qf[c] = __builtin_bit_cast(v8, u);
        }
#pragma unroll
        for (int db = 0; db < DVK / 32; ++db) o[db] = f32x16{};
        m_run = kNegInf;
        l_run = 0.0f;
        slope = 0.0f;
        bias_row = nullptr;
        if (MOD == MOD_GENERAL) {
            if (a.bias_kind == BIAS_ALIBI) slope = a.alibi[h];
            const float sl8 = slope * (2.0f * kLog2e) * a.inv_softcap;
#pragma unroll
            for (int t = 0; t < 8; ++t)
                alibi_step[t] = __builtin_bit_cast(
                    float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, __builtin_amdgcn_exp2f(sl8 * (float)t))));
            if (a.bias_kind == BIAS_DENSE)
                bias_row = a.bias + b * a.bias_sb + h * a.bias_sh + (int64_t)min(my_q, a.M - 1) * a.bias_sm;
        }
        if (MOD == MOD_DENSE) bias_row = a.bias + b * a.bias_sb + h * a.bias_sh;
        // K: A-operand row kappa(r) of a 32-key block, chunk 2c+g. V (transposed
        // reads): input lane j of a 16-lane group reads key (j/4) of a 4-key
        // group at d-chunk cmap(j%4) of the group's 16 columns; cmap = {0,2,1,3}
        // applies kappa to the output rows.
        const int G = lane >> 4, j = lane & 15;
        const int v_dquad = 16 * (G & 1) + 4 * ((j & 1) * 2 + ((j >> 1) & 1));  // d offset within 32
        // K chunk 2c+g of row kappa(r) sits at 32 (c ^ kh) + 16 gl: read at k_lane_off ^ 32c
        const int ksw = L::kswz(kappa(r));
        k_lane_off = kappa(r) * L::KSTR + 16 * ((g ^ ksw) & 1) + 32 * (ksw >> 1);
        if constexpr (!L::POW2) {
#pragma unroll
            for (int jj = 0; jj < L::KG / 2; ++jj) k_base[jj] = kappa(r) * L::KSTR + 16 * ((2 * jj) ^ (g ^ ksw));
        }
        // V chunk (v_dquad>>3) + 4 db of row 8g + j/4 sits at chunk + 4 (db ^ rq): read at v_lane_off ^ 64 db
        const int rq = L::vswz(8 * g + (j >> 2)) >> 2;
        v_lane_off = L::KTILE + (8 * g + (j >> 2)) * L::VSTR + (v_dquad >> 3) * 16 + (v_dquad & 4) * 2 + 64 * rq;
        if constexpr (!L::POW2) {
            const int vb0 = L::KTILE + (8 * g + (j >> 2)) * L::VSTR + (v_dquad >> 3) * 16 + (v_dquad & 4) * 2;
            v_base[0] = vb0 + 64 * rq;
            v_base[1] = vb0 + 64 * (1 ^ rq);
        }
        // copies: wave instruction u covers 16-byte slots 64 (u NWAVES + wave) + lane
        const int slot0 = 64 * wave + lane;
        dma_row0 = slot0 / L::CPR;
        const int pos = slot0 % L::CPR;
        dma_koff = dma_row0 * (int)a.k_sn + 8 * src_chunk(pos ^ L::kswz(dma_row0), a.D);
        dma_voff = dma_row0 * (int)a.v_sn + 8 * src_chunk(pos ^ L::vswz(dma_row0), a.Dv);
    }

    // Source chunk of the 16-byte chunk c of a K/V row whose real width is
    // `width` elements (the kernel's D may round the head dims up): chunks at
    // or past the real width repeat the row's last real chunk, finite data
    // that meets the zero Q columns (K) or fills O^T rows that are never
    // stored (V).
    static __device__ __forceinline__ int src_chunk(int c, int width) { return min(c, (width >> 3) - 1); }

    // Entry of tile step `it` (a global load with a list: issue it early).
    __device__ __forceinline__ int entry(int it) const { return LIST ? list[it] : it; }
    __device__ __forceinline__ int tile_of(int e) const { return LIST ? list_tile(e) : e; }
    __device__ __forceinline__ bool tile_active(int e) const {
        if (LIST) return list_any(e, wave);
        return qw0 < a.M && !(a.causal && e * BN > qw0 + kQueriesPerWave - 1);
    }
    // causal diagonal or ragged end inside the tile
    __device__ __forceinline__ bool tile_crosses(int kt) const {
        return (kt * BN + BN > a.N) || (a.causal && kt * BN + BN - 1 > qw0);
    }

    // Global -> LDS copy of staged tile kt into `stage_off` (asynchronous).
    // Rows past N read row N-1; zero_tail clears their V rows once landed.
    __device__ __forceinline__ void copy_tile(int kt, int stage_off) {
        const int k0 = kt * SN;
        const T* kt_base = Kp + (int64_t)k0 * a.k_sn;
        const T* vt_base = Vp + (int64_t)k0 * a.v_sn;
        const unsigned lds0 = (unsigned)(uintptr_t)smem + stage_off + 1024 * wave;
        constexpr int NW = NTHREADS / 64;
        if constexpr (!UNIFORM_COPY) {
            // slot 64 (u NW + wave) + lane: row slot / CPR, position slot % CPR
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                const int slot = 64 * (u * NW + wave) + (tid & 63);
                const int row = slot / L::CPR, pos = slot - row * L::CPR;
                const int rr = min(k0 + row, a.N - 1) - k0;
                dma16(kt_base + (int64_t)rr * a.k_sn + 8 * src_chunk(pos ^ L::kswz(row), a.D), lds0 + 1024 * NW * u);
                dma16(vt_base + (int64_t)rr * a.v_sn + 8 * src_chunk(pos ^ L::vswz(row), a.Dv),
                      lds0 + L::KTILE + 1024 * NW * u);
            }
            return;
        }
        if (k0 + SN <= a.N) {
            const T* kp = kt_base + dma_koff;
            const T* vp = vt_base + dma_voff;
            const int64_t kstep = (int64_t)DSTEP * a.k_sn, vstep = (int64_t)DSTEP * a.v_sn;
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                dma16(kp, lds0 + 1024 * NW * u);
                dma16(vp, lds0 + L::KTILE + 1024 * NW * u);
                kp += kstep;
                vp += vstep;
            }
        } else {
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                const int row = min(k0 + dma_row0 + u * DSTEP, a.N - 1) - k0 - dma_row0;
                dma16(kt_base + (int64_t)row * a.k_sn + dma_koff, lds0 + 1024 * NW * u);
                dma16(vt_base + (int64_t)row * a.v_sn + dma_voff, lds0 + L::KTILE + 1024 * NW * u);
            }
        }
    }
    __device__ __forceinline__ void zero_tail(int kt, int stage_off) {
        const int k0 = kt * SN;
        if (k0 + SN <= a.N) return;
        constexpr int NW = NTHREADS / 64;
        const u32x4 zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const int row = UNIFORM_COPY ? dma_row0 + u * DSTEP : (64 * (u * NW + wave) + (tid & 63)) / L::CPR;
            if (k0 + row >= a.N)
                *(u32x4*)(smem + stage_off + L::KTILE + 1024 * wave + 1024 * NW * u + 16 * (tid & 63)) = zero;
        }
    }

    // MOD_DENSE: the bias of compute step e for this wavefront's 32 rows, copied
    // global -> LDS (asynchronous) into 32 rows of BN floats of its own at
    // bias_lds. 16-byte chunk c of row r sits at chunk c ^ (r & 15): a read
    // takes one chunk of 16 rows, 256 bytes apart. Rows past M and keys past N
    // repeat the last one (their scores are masked or never stored). Eight copies
    // of four rows each; rows are 16-byte aligned, N is a multiple of 4 and the
    // row stride within [0, 2^24] (bias_can_be_staged).
    static constexpr int BIAS_BYTES = 32 * BN * 4;  // per wavefront
    __device__ __forceinline__ void copy_bias(int e) {
        static_assert(BN == 64, "a bias row is 16 chunks");
        const int k0 = e * BN;
        const unsigned lds0 = (unsigned)(uintptr_t)smem + bias_lds;
        const float* base = bias_row + (int64_t)min(qw0, a.M - 1) * a.bias_sm + k0;  // uniform
        // (the lane is hidden from the compiler so that the copies' offsets are
        // formed here each time instead of kept in registers: at D = 128 those spill)
        int lane = tid & 63;
        asm volatile("" : "+v"(lane));
        if (k0 + BN <= a.N && qw0 + kQueriesPerWave <= a.M) {
            // copy u: rows 4u + lane / 16, chunk (lane % 16) ^ (lane / 16) ^ 4 (u % 4)
            const unsigned roff = 4u * (unsigned)((lane >> 4) * (int)a.bias_sm);
            const unsigned c0 = 16u * (unsigned)((lane & 15) ^ (lane >> 4));
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                dma16s(base, (c0 ^ (64u * (u & 3))) + roff, lds0 + 1024 * u);
                base += 4 * a.bias_sm;
            }
        } else {
            const int last_row = max(0, a.M - 1 - qw0), last = a.N - 4 - k0;
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int row = 4 * u + (lane >> 4);
                const int key = min(4 * ((lane & 15) ^ (row & 15)), last);
                dma16s(base, 4u * (unsigned)(min(row, last_row) * (int)a.bias_sm + key), lds0 + 1024 * u);
            }
        }
    }

    // S^T = K Q^T for the tile in LDS stage `stage_off`.
    __device__ __forceinline__ void qk(int stage_off, int sub = 0) {
        // Fragments are read kFragAhead MFMAs ahead of their use; the
        // scheduling fences keep the compiler from sinking each read next to
        // its MFMA (it otherwise keeps two in flight).
        constexpr int NF = (BN / 32) * (D / 16);
        const lds_u8* kbs = (const lds_u8*)smem + stage_off + sub * BN * L::KSTR;
        auto rd = [&](int i) {
            const int sb = i / (D / 16), c = i % (D / 16);
            return __builtin_bit_cast(v8, *(const lds_u32x4*)(kbs + 32 * sb * L::KSTR + k_off(c)));
        };
        v8 f[kFragAhead];
#pragma unroll
        for (int i = 0; i < kFragAhead; ++i) f[i] = rd(i);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int sb = 0; sb < BN / 32; ++sb) s[sb] = f32x16{};
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            s[i / (D / 16)] = M16::mma(f[i % kFragAhead], qf[i % (D / 16)], s[i / (D / 16)]);
            if (i + kFragAhead < NF) f[i % kFragAhead] = rd(i + kFragAhead);
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // O^T += V^T P^T for the tile in LDS stage `stage_off` (A operand from two
    // transposed 4-key reads).
    __device__ __forceinline__ void pv(int stage_off, int sub = 0) {
        const lds_u8* vbs = (const lds_u8*)smem + stage_off + sub * BN * L::VSTR;
        auto vfrag = [&](int c, int db) {
            const int off = v_off(db);
            const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vbs + (16 * c) * L::VSTR + off));
            const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4*)(vbs + (16 * c + 4) * L::VSTR + off));
            return __builtin_bit_cast(v8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        };
        // V^T fragments kFragAhead MFMAs ahead (see qk)
        constexpr int NF = (DVK / 32) * (BN / 16);
        v8 f[kFragAhead];
#pragma unroll
        for (int i = 0; i < kFragAhead; ++i) f[i] = vfrag(i % (BN / 16), i / (BN / 16));
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            o[i / (BN / 16)] = M16::mma(f[i % kFragAhead], pf[i % (BN / 16)], o[i / (BN / 16)]);
            if (i + kFragAhead < NF)
                f[i % kFragAhead] = vfrag((i + kFragAhead) % (BN / 16), (i + kFragAhead) / (BN / 16));
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    // Scores in log2 units with the call's score_mod: scale, then ALiBi
    // slope*(key - query) or a dense bias, then cap*tanh(x/cap). Constants are
    // folded so ALiBi costs two FMAs per score and the soft-cap an exp2, an
    // add and a reciprocal:
    //   u = 2 log2e t / cap, tanh = 1 - 2/(2^u + 1), x = log2e cap tanh
    //     = cap_hi + cap_m2 * r with r = 1/(2^u + 1), cap_hi = log2e cap,
    //   cap_m2 = -2 log2e cap < 0;
    // with a soft-cap s is left holding r (the softmax takes the row max from
    // min r and folds cap_hi + cap_m2 * r into its exp2 argument).
    template <int BIAS, bool CAP>
    __device__ __forceinline__ void score_mod_tile(int k0) {
        const float c_s = CAP ? a.scale * (2.0f * kLog2e) * a.inv_softcap : a.scale_log2;
        const float c_b = CAP ? (2.0f * kLog2e) * a.inv_softcap : kLog2e;
        const float sl = slope * c_b;
        const float base = sl * (float)(k0 + 8 * g - my_q);
        float bvals[BN / 2];
        if constexpr (MOD == MOD_DENSE) {
            const lds_u8* br = (const lds_u8*)smem + bias_lds + (my_q - qw0) * BN * 4;
            const int sw = (my_q - qw0) & 15;
#pragma unroll
            for (int q4 = 0; q4 < BN / 8; ++q4) {  // keys 16 (q4 >> 1) + 8 g + 4 (q4 & 1) .. + 3
                const f32x4 v = __builtin_bit_cast(
                    f32x4, *(const lds_u32x4*)(br + 16 * ((4 * (q4 >> 1) + 2 * g + (q4 & 1)) ^ sw)));
#pragma unroll
                for (int t = 0; t < 4; ++t) bvals[4 * q4 + t] = v[t];
            }
        } else if (BIAS == BIAS_DENSE) {
            const float* br = bias_row + k0 + 8 * g;
            if (k0 + BN <= a.N) {
#pragma unroll
                for (int q4 = 0; q4 < BN / 8; ++q4) {
                    const f32x4 v = *(const f32x4*)(br + 16 * (q4 >> 1) + 4 * (q4 & 1));
#pragma unroll
                    for (int t = 0; t < 4; ++t) bvals[4 * q4 + t] = v[t];
                }
            } else {
#pragma unroll
                for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
                    for (int e = 0; e < 16; ++e)
                        bvals[16 * sb + e] = bias_row[min(k0 + 8 * g + tile_pos(sb, e), a.N - 1)];
            }
        }
        if constexpr (BIAS == BIAS_ALIBI && CAP) {
            // 2^u = 2^(c_s s + base_j) * 2^(sl t) with key 8-group base_j and t = key & 7: the ALiBi step
            // inside a group rides on the "+ 1" of the soft-cap as a multiply-add
#pragma unroll
            for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
                for (int hh = 0; hh < 2; ++hh) {
                    const float bj = __builtin_fmaf(sl, (float)(32 * sb + 16 * hh), base);
#pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        const float x = __builtin_amdgcn_exp2f(__builtin_fmaf(s[sb][8 * hh + t], c_s, bj));
                        s[sb][8 * hh + t] = __builtin_amdgcn_rcpf(__builtin_fmaf(x, alibi_step[t], 1.0f));
                    }
                }
            return;
        }
#pragma unroll
        for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                float u;
                if (BIAS == BIAS_ALIBI)
                    u = __builtin_fmaf(s[sb][e], c_s, __builtin_fmaf(sl, (float)tile_pos(sb, e), base));
                else if (MOD == MOD_DENSE && !CAP)  // natural units: the softmax's exp2 argument applies log2e
                    u = __builtin_fmaf(s[sb][e], a.scale, bvals[16 * sb + e]);
                else if (BIAS == BIAS_DENSE)
                    u = __builtin_fmaf(s[sb][e], c_s, bvals[16 * sb + e] * c_b);
                else
                    u = s[sb][e] * c_s;
                // with a soft-cap, s keeps r = 1 / (2^u + 1): the log2 score is
                // cap_hi + cap_m2 * r, formed inside the softmax's exp2 argument
                if (CAP) u = __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(u) + 1.0f);
                s[sb][e] = u;
            }
    }
    __device__ __forceinline__ void general_scores(int k0) {
        const bool cap = a.softcap > 0.0f;
        if constexpr (MOD == MOD_DENSE) {
            if (cap) score_mod_tile<BIAS_DENSE, true>(k0);
            else score_mod_tile<BIAS_DENSE, false>(k0);
            return;
        }
        if (a.bias_kind == BIAS_ALIBI) {
            if (cap) score_mod_tile<BIAS_ALIBI, true>(k0);
            else score_mod_tile<BIAS_ALIBI, false>(k0);
        } else if (a.bias_kind == BIAS_DENSE) {
            if (cap) score_mod_tile<BIAS_DENSE, true>(k0);
            else score_mod_tile<BIAS_DENSE, false>(k0);
        } else {
            if (cap) score_mod_tile<BIAS_NONE, true>(k0);
            else score_mod_tile<BIAS_NONE, false>(k0);
        }
    }

    // Masked scores -> `masked` (-inf, or +inf for soft-capped scores held as
    // r). Causal / ragged end: key k0+8g+pos is valid iff pos < lim. With a
    // block mask whose blocks cut the slice: per element.
    __device__ __forceinline__ void apply_mask(int e_ent, int k0, float masked = kNegInf) {
        if (LIST && !list_full(e_ent, wave)) {
            // masked_out (attention.cpp:54-62) per element, branch-free: the
            // bitmap bytes are read at clamped indices and combined by selects
            const int qb = my_q / a.mask_qbs;
            const bool row_ok = qb < a.mask_qb;
            const uint8_t* mrow = a.mask + (int64_t)min(qb, a.mask_qb - 1) * a.mask_kb;
            const int klim = a.causal ? min(a.N - 1, my_q) : a.N - 1;  // last valid key
            // 8 consecutive keys at a time: their bitmap bytes are loaded together
#pragma unroll
            for (int q8 = 0; q8 < BN / 16; ++q8) {
                const int sb = q8 >> 1, e0 = 8 * (q8 & 1);
                unsigned char byte[8];
                int kbs[8];
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    kbs[t] = min(k0 + 8 * g + tile_pos(sb, e0 + t), a.N - 1) / a.mask_kbs;
                    byte[t] = mrow[min(kbs[t], a.mask_kb - 1)];
                }
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const int kj = k0 + 8 * g + tile_pos(sb, e0 + t);
                    const bool ok = row_ok & (kj <= klim) & (kbs[t] < a.mask_kb) & (byte[t] != 0);
                    s[sb][e0 + t] = ok ? s[sb][e0 + t] : masked;
                }
            }
            return;
        }
        const int lim = (a.causal ? min(a.N, my_q + 1) : a.N) - k0 - 8 * g;
#pragma unroll
        for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
            for (int e = 0; e < 16; ++e)
                if (tile_pos(sb, e) >= lim) s[sb][e] = masked;
    }

    // Online softmax of the scores in s (tile step with entry e_ent): running
    // max with lazy rescale of O and l, probabilities packed into pf, row sum.
    __device__ __forceinline__ void softmax(int e_ent) {
        const int kt = tile_of(e_ent);
        const int k0 = kt * BN;
        const bool need_mask = tile_crosses(kt) || (LIST && !list_full(e_ent, wave));
        float mx = kNegInf;
        const bool capped = MOD != MOD_PLAIN && a.softcap > 0.0f;  // uniform
        const bool natural = MOD == MOD_DENSE && !capped;          // s in natural units
        if (natural) {
            general_scores(k0);
            if (need_mask) apply_mask(e_ent, k0);
        }
        // s still holds raw dot products (or natural scores): the log2 score is s * to_log2
        const bool raw = (MOD == MOD_PLAIN && !need_mask) || natural;
        const float to_log2 = MOD == MOD_DENSE ? kLog2e : a.scale_log2;
        // 128-key tiles (D <= 64, no list): p is taken against the running max
        // first, without the tile's max. A row sum of at most 2^kRescaleSlack
        // proves every p <= 2^kRescaleSlack, the bound the lazy rescale keeps,
        // so the result is the one the max would have given (the max raises
        // nothing then). Otherwise (a larger sum, inf or NaN) the tile is redone
        // below with its max. Measured +5-6 % at D = 32 and 64; at D = 96 and
        // 128 (64-key tiles) the same code measured slower (3-6 %).
        if (D <= 64 && !LIST && raw && __builtin_amdgcn_ballot_w64(m_run == kNegInf) == 0) {
            float fsum = 0.0f;
#pragma unroll
            for (int c = 0; c < BN / 16; ++c) {
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    pf[c][t] = (T)__builtin_amdgcn_exp2f(
                        __builtin_fmaf(s[c >> 1][8 * (c & 1) + t], to_log2, -m_run));
#pragma unroll
                for (int t = 0; t < 8; t += 2)
                    fsum = Dot2<T>::sum2(typename Dot2<T>::v2{pf[c][t], pf[c][t + 1]}, fsum);
            }
            if (__builtin_amdgcn_ballot_w64(!(fsum <= kSumBound)) == 0) {
                l_run += fsum;
                return;
            }
        }
        const float cap_hi = a.softcap * kLog2e, cap_m2 = -2.0f * a.softcap * kLog2e;
        if (raw) {
            if (MOD == MOD_DENSE || a.scale_log2 >= 0.0f) {
#pragma unroll
                for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[sb][e]);
                mx *= to_log2;
            } else {
                float mn = __builtin_huge_valf();
#pragma unroll
                for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
                    for (int e = 0; e < 16; ++e) mn = fminf(mn, s[sb][e]);
                mx = mn * a.scale_log2;
            }
        } else if (capped) {
            general_scores(k0);  // s = r, log2 score cap_hi + cap_m2 * r, decreasing in r
            if (need_mask) apply_mask(e_ent, k0, __builtin_huge_valf());
            float mn = __builtin_huge_valf();
#pragma unroll
            for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
                for (int e = 0; e < 16; ++e) mn = fminf(mn, s[sb][e]);
            mx = __builtin_fmaf(mn, cap_m2, cap_hi);  // -inf when every score is masked
        } else {
            if (MOD != MOD_PLAIN) {
                general_scores(k0);
            } else {
#pragma unroll
                for (int sb = 0; sb < BN / 32; ++sb) s[sb] *= a.scale_log2;
            }
            if (need_mask) apply_mask(e_ent, k0);
#pragma unroll
            for (int sb = 0; sb < BN / 32; ++sb)
#pragma unroll
                for (int e = 0; e < 16; ++e) mx = fmaxf(mx, s[sb][e]);
        }
        mx = half_swap_max(mx);

        // Lazy rescale (wave-uniform branch).
        const bool raise = mx > m_run + kRescaleSlack;
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {
            // lanes that do not raise keep their max and scale by exactly 1
            // (their m_run may be -inf: -inf - -inf must not reach exp2)
            const float alpha = raise ? __builtin_amdgcn_exp2f(m_run - mx) : 1.0f;
            m_run = raise ? mx : m_run;
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < DVK / 32; ++db) o[db] *= alpha;
        }
        const float m_use = (m_run == kNegInf) ? 0.0f : m_run;

        if (raw) {
#pragma unroll
            for (int c = 0; c < BN / 16; ++c)
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    pf[c][t] = (T)__builtin_amdgcn_exp2f(
                        __builtin_fmaf(s[c >> 1][8 * (c & 1) + t], to_log2, -m_use));
        } else if (capped) {
            const float c0 = cap_hi - m_use;
#pragma unroll
            for (int c = 0; c < BN / 16; ++c)
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    pf[c][t] = (T)__builtin_amdgcn_exp2f(__builtin_fmaf(s[c >> 1][8 * (c & 1) + t], cap_m2, c0));
        } else {
#pragma unroll
            for (int c = 0; c < BN / 16; ++c)
#pragma unroll
                for (int t = 0; t < 8; ++t)
                    pf[c][t] = (T)__builtin_amdgcn_exp2f(s[c >> 1][8 * (c & 1) + t] - m_use);
        }
        float lsum = 0.0f;
#pragma unroll
        for (int c = 0; c < BN / 16; ++c)
#pragma unroll
            for (int t = 0; t < 8; t += 2)
                lsum = Dot2<T>::sum2(typename Dot2<T>::v2{pf[c][t], pf[c][t + 1]}, lsum);
        l_run += lsum;
    }

    // Key split: the unnormalised rows and (m, l) of split `split`.
    __device__ __forceinline__ void store_partial(int split) {
        const float l_tot = l_run + __shfl_xor(l_run, 32);
        if (my_q >= a.M) return;
        const int64_t prow = ((int64_t)split * a.B * a.H + (int64_t)b * a.H + h) * a.M + my_q;
        float* po = a.part_o + prow * a.Dv + 8 * g;
        const bool coh = a.split_counters != nullptr;
#pragma unroll
        for (int db = 0; db < DVK / 32; ++db) {
#pragma unroll
            for (int cc = 0; cc < 2; ++cc) {
                if (32 * db + 16 * cc + 8 * g >= a.Dv) continue;  // past the value dim
                f32x4 lo, hi;
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    lo[t] = o[db][8 * cc + t];
                    hi[t] = o[db][8 * cc + 4 + t];
                }
                put_partial4(po + 32 * db + 16 * cc, lo, coh);
                put_partial4(po + 32 * db + 16 * cc + 4, hi, coh);
            }
        }
        if (g == 0) {
            put_partial(a.part_ml + 2 * prow, m_run, coh);
            put_partial(a.part_ml + 2 * prow + 1, l_tot, coh);
        }
    }

    // Normalise and store; rows that saw no valid key have l = 0 and are written as 0.
    __device__ __forceinline__ void store_output() {
        const float l_tot = l_run + __shfl_xor(l_run, 32);
        const float inv = l_tot > 0.0f ? 1.0f / l_tot : 0.0f;
        if (my_q >= a.M) return;
        if (a.out_f32) {
            float* orow = (float*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)my_q * a.o_sm + 8 * g;
#pragma unroll
            for (int db = 0; db < DVK / 32; ++db) {
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    if (32 * db + 16 * cc + 8 * g >= a.Dv) continue;  // past the value dim
                    f32x4 lo, hi;
#pragma unroll
                    for (int t = 0; t < 4; ++t) {
                        lo[t] = o[db][8 * cc + t] * inv;
                        hi[t] = o[db][8 * cc + 4 + t] * inv;
                    }
                    *(f32x4*)(orow + 32 * db + 16 * cc) = lo;
                    *(f32x4*)(orow + 32 * db + 16 * cc + 4) = hi;
                }
            }
        } else {
            T* orow = (T*)a.o + b * a.o_sb + h * a.o_sh + (int64_t)my_q * a.o_sm + 8 * g;
#pragma unroll
            for (int db = 0; db < DVK / 32; ++db) {
#pragma unroll
                for (int cc = 0; cc < 2; ++cc) {
                    if (32 * db + 16 * cc + 8 * g >= a.Dv) continue;  // past the value dim
                    v8 val;
#pragma unroll
                    for (int t = 0; t < 8; ++t) val[t] = (T)(o[db][8 * cc + t] * inv);
                    *(u32x4*)(orow + 32 * db + 16 * cc) = __builtin_bit_cast(u32x4, val);
                }
            }
        }
    }
};

// End of a query tile (or of its key split `split` of `active`): O, or the
// partial rows followed by the merge in the split workgroup that arrives last.
template <typename W, int NTHREADS, bool SPLIT>
__device__ __forceinline__ void finish_qtile(const FwdArgs& a, W& w, unsigned char* smem, int bh, int qt,
                                             int q0, int block_m, int split, int active) {
    if (!SPLIT || active <= 1) {
        w.store_output();
        return;
    }
    w.store_partial(split);
    if (a.split_counters == nullptr) return;  // merged by combine_splits_kernel
    __syncthreads();                          // LDS below is reused
    int* flag = (int*)(smem + 24 * NTHREADS);
    if (split_arrive(a.split_counters + (int64_t)bh * a.num_q_tiles + qt, active, flag))
        merge_split_rows<typename W::T_, NTHREADS>(a, bh, q0, min(block_m, a.M - q0), active, (float*)smem);
}

}  // namespace
}  // namespace ofh
