// QK score tile with post-ops on the device: S = (Q K^T) * scale + bias
// (+ soft-cap), for a batch of strided tiles.
//
// Follows the reference's QK score tile (src/onednn_flash/qk_score_tile.cpp:
// 48-69 post-ops after matmul_tile_strided_inplace, whose reference kernel
// sums over k sequentially in fp32, src/onednn_flash/tile_kernel.cpp:49-86).
// Every product and every partial sum is rounded once, in the same order, so
// fp32 results are bit-identical to the reference. 32x32 or 64x64 output blocks
// per workgroup; Q and K^T chunks of 32 along k are staged through LDS as fp32.
//
// For bf16/fp16 inputs a matrix-core variant computes the same scores with
// v_mfma_f32_32x32x16_{bf16,f16}: the products are exact in fp32 and only the
// summation order differs from the sequential sum (error within k * 2^-24 *
// sum_k |q k| per score). It needs rows contiguous along k and 16-byte aligned.

#include "k_chunks.h"
#include "ofh_kernels.h"

#include <algorithm>

namespace ofh {
namespace {

constexpr int64_t kMaxGridZ = 65535;   // tiles per launch (grid z)

template <typename T>
__device__ __forceinline__ float to_f32(T x) { return (float)x; }

// Exact scores. A workgroup of 16 x 16 threads forms a block of 16 PT x 16 PT
// scores, PT x PT per thread; chunks of 32 along k of its Q and K rows are
// staged in LDS as fp32, k-major, so that a wavefront reads consecutive K
// elements and broadcasts Q. The next chunk is on its way through registers
// while this one is multiplied, and the LDS is double-buffered (one barrier per
// chunk).
//
// What bounds it: the vector ALU, two instructions per multiply-add because
// product and sum are rounded separately, and the LDS: per k a thread reads 2 PT
// floats for PT^2 multiply-adds. Measured, fp32 32 tiles 1024^2 x 128: 343 us
// with 4 scores of one column per thread (a read per multiply-add, 64-bit index
// arithmetic per load), 195 us with PT = 4 (44 TFLOP/s of useful work; the ALU's rate,
// one instruction per lane and multiply or add, allows 78).
template <typename T, int PT>
__global__ __launch_bounds__(256) void qk_score_kernel(QkScoreArgs a) {
    // Products, sums, scale and bias are each rounded: no contraction to FMA.
#pragma clang fp contract(off)
    constexpr int BT = 16 * PT;      // scores per block side
    constexpr int BK = 32;           // k per chunk
    constexpr int STR = BT + 4;      // floats per k row of a staged chunk
    constexpr int LOADS = BT * BK / 256;
    constexpr int GW = PT < 4 ? PT : 4, NG = PT / GW;  // a thread's rows (columns): NG groups of GW, 16 GW apart
    typedef float vec __attribute__((ext_vector_type(GW)));
    __shared__ __attribute__((aligned(16))) float qs[2][BK * STR], ks[2][BK * STR];
    const int tid = threadIdx.x;
    const int tx = tid & 15, ty = tid >> 4;
    const int64_t bt = blockIdx.z;
    const int64_t i0 = (int64_t)blockIdx.y * BT, j0 = (int64_t)blockIdx.x * BT;
    // Lanes walk whichever axis has the smaller stride (row-major Q [m,k] and
    // K [n,k] are both contiguous along k): load u of a thread is element
    // (row r0 + u rs, k kk0 + u kks) of the chunk. Elements outside the tile are 0.
    struct Side {
        int r0, rs, kk0, kks, rows, lds, lds_step;
        const T* p;
        int64_t step, chunk;
    };
    auto side = [&](const T* base, int64_t sr, int64_t sk, int64_t row0, int64_t rows) {
        const bool k_fast = sk <= sr;  // uniform
        Side d;
        d.r0 = k_fast ? tid / BK : tid % BT;
        d.rs = k_fast ? 256 / BK : (256 % BT);  // (BT divides 256 or 256 BT; k_fast false: rows repeat)
        d.kk0 = k_fast ? tid % BK : tid / BT;
        d.kks = k_fast ? 0 : 256 / BT;
        d.rows = (int)min((int64_t)BT, rows - row0);
        d.lds = d.kk0 * STR + d.r0;
        d.lds_step = d.kks * STR + d.rs;
        d.p = base + (row0 + d.r0) * sr + d.kk0 * sk;
        d.step = d.rs * sr + d.kks * sk;
        d.chunk = BK * sk;
        return d;
    };
    static_assert(256 % BT == 0 && 256 % BK == 0, "a load covers whole rows or whole k steps");
    Side sq = side((const T*)a.q + bt * a.a_sb, a.a_sm, a.a_sk, i0, a.M);
    Side sk = side((const T*)a.k + bt * a.b_sb, a.b_sn, a.b_sk, j0, a.N);
    float rq[LOADS], rk[LOADS];
    auto load = [&](Side& d, float (&r)[LOADS], int klen) {  // klen: k elements of this chunk
        const T* p = d.p;
        if (d.rows == BT && klen == BK) {
#pragma unroll
            for (int u = 0; u < LOADS; ++u) r[u] = to_f32(p[u * d.step]);
        } else {
#pragma unroll
            for (int u = 0; u < LOADS; ++u)
                r[u] = d.r0 + u * d.rs < d.rows && d.kk0 + u * d.kks < klen ? to_f32(p[u * d.step]) : 0.0f;
        }
        d.p += d.chunk;
    };
    auto put = [&](const Side& d, const float (&r)[LOADS], float* lds) {
#pragma unroll
        for (int u = 0; u < LOADS; ++u) lds[d.lds + u * d.lds_step] = r[u];
    };
    float acc[PT][PT];
#pragma unroll
    for (int x = 0; x < PT; ++x)
#pragma unroll
        for (int y = 0; y < PT; ++y) acc[x][y] = 0.0f;
    KChunks<BK> kc(a.K);
    load(sq, rq, kc.len());
    load(sk, rk, kc.len());
    put(sq, rq, qs[0]);
    put(sk, rk, ks[0]);
    __syncthreads();
    int buf = 0;
    for (; kc.any(); kc.next()) {
        const bool more = kc.more();
        if (more) {
            KChunks<BK> nc = kc;
            nc.next();
            load(sq, rq, nc.len());
            load(sk, rk, nc.len());
        }
        const float *ql = &qs[buf][GW * ty], *kl = &ks[buf][GW * tx];
        auto step = [&](int t) {
#pragma clang fp contract(off)  // (a lambda's body does not take the function's pragma)
            vec qv[NG], kv[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                qv[g] = *(const vec*)(ql + t * STR + 16 * GW * g);
                kv[g] = *(const vec*)(kl + t * STR + 16 * GW * g);
            }
#pragma unroll
            for (int x = 0; x < PT; ++x)
#pragma unroll
                for (int y = 0; y < PT; ++y) acc[x][y] = acc[x][y] + qv[x / GW][x % GW] * kv[y / GW][y % GW];
        };
        const int len = kc.len();
        if (len == BK) {
#pragma unroll 8
            for (int t = 0; t < BK; ++t) step(t);
        } else {
            for (int t = 0; t < len; ++t) step(t);
        }
        if (more) {
            put(sq, rq, qs[buf ^ 1]);
            put(sk, rk, ks[buf ^ 1]);
        }
        __syncthreads();
        buf ^= 1;
    }
#pragma unroll
    for (int x = 0; x < PT; ++x) {
        const int64_t i = i0 + 16 * GW * (x / GW) + GW * ty + x % GW;
        if (i >= a.M) continue;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const int64_t j = j0 + 16 * GW * g + GW * tx;
            vec v;
#pragma unroll
            for (int e = 0; e < GW; ++e) {
                float w = acc[x][GW * g + e];
                if (a.has_scale) w = w * a.scale;
                if (a.bias != nullptr && j + e < a.N) w = w + a.bias[bt * a.bias_sb + i * a.bias_sm + (j + e) * a.bias_sn];
                if (a.softcap > 0.0f) w = a.softcap * tanhf(w / a.softcap);
                v[e] = w;
            }
            float* c = a.c + bt * a.c_sb + i * a.c_sm + j * a.c_sn;
            if (a.vec4 && j + GW <= a.N) {
                *(vec*)c = v;
            } else {
#pragma unroll
                for (int e = 0; e < GW; ++e)
                    if (j + e < a.N) c[e * a.c_sn] = v[e];
            }
        }
    }
}

typedef __bf16 qk_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 qk_f16x8 __attribute__((ext_vector_type(8)));
typedef float qk_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int qk_u32x4 __attribute__((ext_vector_type(4)));

template <typename T>
struct QkMfma;
template <>
struct QkMfma<__bf16> {
    static __device__ __forceinline__ qk_f32x16 run(qk_u32x4 a, qk_u32x4 b, qk_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(qk_bf16x8, a),
                                                       __builtin_bit_cast(qk_bf16x8, b), c, 0, 0, 0);
    }
};
template <>
struct QkMfma<_Float16> {
    static __device__ __forceinline__ qk_f32x16 run(qk_u32x4 a, qk_u32x4 b, qk_f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(qk_f16x8, a),
                                                      __builtin_bit_cast(qk_f16x8, b), c, 0, 0, 0);
    }
};

// 128x128 score block per workgroup, 4 wavefronts of 64x64 (2x2 MFMA tiles of
// 32x32). Operand lane layout of the 32x32x16 MFMA: lane l holds row (l & 31)
// of the A operand and column (l & 31) of the B operand, k elements
// 8*(l >> 5) .. +7 of the 16-wide step; output element e of lane l is row
// 8*(e >> 2) + 4*(l >> 5) + (e & 3), column l & 31. With A = K and B = Q^T
// the tile is S^T, so each lane owns runs of 4 consecutive keys of one query
// row: contiguous in the row-major score matrix.
constexpr int kMfmaBlock = 128;

// LDS of the matrix-core score kernel, 32 KB so that three workgroups fit a CU
// (their registers allow three). Unpadded rows (the DMA copies below write
// consecutive bytes) with XOR-swizzled 16-byte chunks, chosen so that every
// access pattern below touches 16 distinct bank groups per 16 lanes.
//
// Operands: per 64-wide k chunk, the workgroup's 128 Q rows and 128 K rows,
// 128 bytes each, copied global -> LDS by global_load_lds_dwordx4 (a
// wavefront writes 1 KB of consecutive LDS: eight rows). Chunk c of row r sits
// at position c ^ ((r >> 1) & 7): a fragment read takes 16 consecutive rows at
// one chunk, and rows r, r + 1 share a 256-byte bank line.
//
// Epilogue: each wavefront's 64x64 fp32 block in two passes of 32 rows x 256
// bytes, chunk c of row r at c ^ (r & 15); written 16 rows x one chunk per 16
// lanes, read back one row (16 chunks) per 16 lanes.
constexpr int kChunkK = 64;
constexpr int kRowBytes = kChunkK * 2;
constexpr int kOperandBytes = 2 * kMfmaBlock * kRowBytes;  // Q then K: 32 KB
constexpr int kStageBytes = 4 * 32 * 256;                  // 32 rows x 64 fp32 per wavefront: 32 KB
constexpr int kQkLdsBytes = kOperandBytes > kStageBytes ? kOperandBytes : kStageBytes;

typedef __attribute__((address_space(3))) unsigned char qk_lds_u8;
typedef __attribute__((address_space(3))) qk_u32x4 qk_lds_u32x4;

// One 16-byte global -> LDS copy per lane; `dst` is the wavefront's LDS base
// (lane L writes dst + 16 L).
__device__ __forceinline__ void dma16(const void* src, qk_lds_u8* dst) {
    __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}
__device__ __forceinline__ qk_u32x4 lds_read16(const qk_lds_u8* p) { return *(const qk_lds_u32x4*)p; }
typedef float qk_f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) qk_f32x4 qk_lds_f32x4;
typedef __attribute__((address_space(3))) float qk_lds_f32;
__device__ __forceinline__ void lds_write_f4(qk_lds_u8* p, qk_f32x4 v) { *(qk_lds_f32x4*)p = v; }
__device__ __forceinline__ qk_f32x4 lds_read_f4(const qk_lds_u8* p) { return *(const qk_lds_f32x4*)p; }

template <typename T, bool CAP>
__global__ __launch_bounds__(256) void qk_score_mfma_kernel(QkScoreArgs a) {
    // Scale and bias are rounded separately, as the reference applies them.
#pragma clang fp contract(off)
    __shared__ __attribute__((aligned(16))) unsigned char smem[kQkLdsBytes];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t bt = blockIdx.z;
    const int64_t qb0 = (int64_t)blockIdx.y * kMfmaBlock, kb0 = (int64_t)blockIdx.x * kMfmaBlock;
    const int64_t i0 = qb0 + (wave >> 1) * 64;
    const int64_t j0 = kb0 + (wave & 1) * 64;
    const T* q = (const T*)a.q + bt * a.a_sb;
    const T* k = (const T*)a.k + bt * a.b_sb;
    const int r = lane & 31, half = lane >> 5;
    qk_lds_u8* lds = (qk_lds_u8*)smem;
    // DMA copy of one k-chunk: wavefront w, step u copies rows 32u + 8w .. +7
    // of Q and of K; lane L writes row 32u + 8w + (L >> 3), position L & 7,
    // holding global chunk (L & 7) ^ ((row >> 1) & 7). Rows past M or N and
    // chunks past K read clamped in-range addresses; their values are never used.
    auto copy_chunk = [&](int64_t k0) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int row = 32 * u + 8 * wave + (lane >> 3);
            const int c = (lane & 7) ^ ((row >> 1) & 7);
            const int64_t kc = (k0 + 8 * c < a.K) ? k0 + 8 * c : k0;
            const int64_t qi = min(qb0 + row, a.M - 1), kj = min(kb0 + row, a.N - 1);
            const int base = (32 * u + 8 * wave) * kRowBytes;
            dma16(q + qi * a.a_sm + kc, lds + base);
            dma16(k + kj * a.b_sn + kc, lds + kMfmaBlock * kRowBytes + base);
        }
    };
    // Fragment rows of this lane: Q (B operand) rows and K (A operand) rows.
    int qoff[2], koff[2], qsw[2], ksw[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int qr = (wave >> 1) * 64 + 32 * t + r, kr = (wave & 1) * 64 + 32 * t + r;
        qoff[t] = qr * kRowBytes;
        koff[t] = kMfmaBlock * kRowBytes + kr * kRowBytes;
        qsw[t] = (qr >> 1) & 7;
        ksw[t] = (kr >> 1) & 7;
    }
    qk_f32x16 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[x][y][e] = 0.0f;
    const qk_u32x4 zero = {0u, 0u, 0u, 0u};
    for (int64_t k0 = 0; k0 < a.K; k0 += kChunkK) {
        copy_chunk(k0);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this wavefront's copies have landed
        __syncthreads();                      // ... and every other wavefront's
        const int steps = ((int)min((int64_t)kChunkK, a.K - k0) + 15) / 16;  // 16-wide k steps
        for (int st = 0; st < steps; ++st) {
            const int c = 2 * st + half;                     // 16-byte chunk of this lane
            const bool kin = k0 + 8 * c < a.K;               // K is a multiple of 8
            qk_u32x4 qa[2], kb[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                qa[t] = kin ? lds_read16(lds + qoff[t] + 16 * (c ^ qsw[t])) : zero;
                kb[t] = kin ? lds_read16(lds + koff[t] + 16 * (c ^ ksw[t])) : zero;
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = QkMfma<T>::run(kb[y], qa[x], acc[x][y]);
        }
        __syncthreads();  // the next chunk (or the epilogue) overwrites the operands
    }
    // acc[x][y] holds the transposed tile: lane column r is query i0+32x+r and
    // elements 4g..4g+3 are the four consecutive keys j0+32y+8g+4*half+0..3.
    // The block goes through LDS (two passes of 32 rows) so that the global
    // stores and bias loads are full 256-byte row segments: 16 lanes per row,
    // four rows per instruction.
    qk_lds_u8* st = lds + wave * 32 * 256;  // this wavefront's 32-row pass buffer
    const int col = 4 * (lane & 15);
    const int64_t jb = j0 + col;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        // pass x: rows 32x .. 32x+31 of the wavefront's block
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int chunk = 8 * y + 2 * g + half;  // keys 32y + 8g + 4 half .. +3
                lds_write_f4(st + r * 256 + 16 * (chunk ^ (r & 15)),
                             qk_f32x4{acc[x][y][4 * g], acc[x][y][4 * g + 1], acc[x][y][4 * g + 2], acc[x][y][4 * g + 3]});
            }
        __syncthreads();
#pragma unroll 4
        for (int it = 0; it < 8; ++it) {
            const int row = 4 * it + (lane >> 4);
            const int64_t i = i0 + 32 * x + row;
            if (i >= a.M || jb >= a.N) continue;
            const qk_f32x4 raw = lds_read_f4(st + row * 256 + 16 * ((lane & 15) ^ (row & 15)));
            float v[4] = {raw[0], raw[1], raw[2], raw[3]};
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = a.has_scale ? v[u] * a.scale : v[u];
            float* crow = a.c + bt * a.c_sb + i * a.c_sm;
            const float* brow = a.bias != nullptr ? a.bias + bt * a.bias_sb + i * a.bias_sm : nullptr;
            if (a.vec4 && jb + 3 < a.N) {
                if (brow != nullptr) {
                    const float4 b4 = *(const float4*)(brow + jb);
                    v[0] = v[0] + b4.x;
                    v[1] = v[1] + b4.y;
                    v[2] = v[2] + b4.z;
                    v[3] = v[3] + b4.w;
                }
                if (CAP)
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = a.softcap * tanhf(v[u] / a.softcap);
                *(float4*)(crow + jb) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int64_t j = jb + u;
                    if (j >= a.N) break;
                    float w = v[u];
                    if (brow != nullptr) w = w + brow[j * a.bias_sn];
                    if (CAP) w = a.softcap * tanhf(w / a.softcap);
                    crow[j * a.c_sn] = w;
                }
            }
        }
        __syncthreads();  // the next pass reuses the buffer
    }
}

// Post-operations of a row kernel instantiation (the scale is a run-time choice).
enum QkPost { QK_POST_NONE = 0, QK_POST_BIAS = 1, QK_POST_CAP = 2, QK_POST_BIAS_CAP = 3 };

// Score rows, K <= 128: one workgroup per 128-row query block and run of `tpw` 128-key blocks.
// The query block's MFMA fragments stay in registers for the whole run; K
// block t+1 is copied global -> LDS into the second buffer while block t is
// multiplied and written, and the buffer block t was read from then stages
// its epilogue (the same 256-byte row segments as above). 64 KB of LDS, two
// workgroups per CU. A one-block workgroup serialises its copies, MFMAs and
// stores (0.59-0.65 ms for 32 heads x 4096^2 x 128, against 0.35 ms for the
// stores alone); streaming K blocks through two buffers overlaps them.
// Workgroups are numbered so that each XCD (workgroup n runs on XCD n mod 8)
// takes a contiguous range of query blocks, i.e. reads the Q and K of a few
// heads only. Same products and summation order as qk_score_mfma_kernel, so
// the scores are bit-identical. CH = 16-byte chunks per K row in LDS (K <= 8 CH).
//
// A block's bias is requested into registers (32 per lane: one epilogue pass)
// before its products, and the second pass's behind the first one's stores; read
// in the epilogue it stood between each row's LDS read and its store. VEC: scores and bias are read and written as 16
// lanes x 16 bytes per row (aligned rows, N a multiple of 4); else as 64 lanes x
// 4 bytes, whole 256-byte row pieces as well. Measured (us, one-block kernel ->
// this): bf16 32 tiles 2048^2 x 128 with a shared bias 209 -> 169 (3.5 TB/s), with
// a bias per tile, 16 tiles, 148 -> 110 (4.9 TB/s), with a soft-cap 200 -> 169; 30
// tiles 1001 x 1003 x 64, shared bias 69 -> 47, no bias 55 -> 33. A shared bias
// with the tiles of an XCD one after another (the order of the other calls):
// 182.
constexpr int kRowBufBytes = 32 * 1024;   // one K block (128 rows x 16 CH bytes), or the epilogue staging

template <int CH>
__device__ __forceinline__ int row_swz(int row) {
    // chunk position XOR: 16 consecutive rows of a fragment read hit 16 distinct 16-byte bank groups
    return CH == 16 ? (row & 15) : CH == 8 ? ((row >> 1) & 7) : ((row >> 2) & 3);
}

template <typename T, int CH, int POST, bool VEC>
__global__ __launch_bounds__(256, 2) void qk_score_mfma_rows_kernel(QkScoreArgs a, int64_t nqb, int64_t npieces,
                                                                    int tpw) {
#pragma clang fp contract(off)
    __shared__ __attribute__((aligned(16))) unsigned char smem[2 * kRowBufBytes];
    constexpr int RB = CH * 16;    // LDS bytes per K row
    constexpr int RPI = 64 / CH;   // K rows per wavefront copy instruction (1 KB of LDS)
    constexpr int STEPS = CH / 2;  // 16-wide k steps
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, half = lane >> 5;
    const int64_t total = gridDim.x, n = blockIdx.x, per = total / 8;
    const int64_t id = n < 8 * per ? (n % 8) * per + n / 8 : n;
    int64_t piece = id % npieces, qb = (id / npieces) % nqb, bt = id / (npieces * nqb);
    if ((POST & QK_POST_BIAS) != 0 && a.bias_sb == 0 && (a.batch & 7) == 0) {
        // A bias that all tiles share: an XCD's tiles (n mod 8 again) run side by
        // side, so that its L2 serves a bias block to all of them
        bt = n % a.batch;
        piece = (n / a.batch) % npieces;
        qb = n / (a.batch * npieces);
    }
    const int64_t nkb = (a.N + kMfmaBlock - 1) / kMfmaBlock;
    const int64_t kb_begin = piece * tpw;
    const int64_t kb_end = min(nkb, kb_begin + tpw);
    const T* q = (const T*)a.q + bt * a.a_sb;
    const T* k = (const T*)a.k + bt * a.b_sb;
    qk_lds_u8* lds = (qk_lds_u8*)smem;
    const qk_u32x4 zero = {0u, 0u, 0u, 0u};
    const int64_t i0 = qb * kMfmaBlock + (wave >> 1) * 64;   // the wavefront's 64 query rows
    // B-operand fragments of the wavefront's query rows (rows past M clamped, chunks past K zero)
    qk_u32x4 qf[2][STEPS];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int64_t qr = min(i0 + 32 * x + r, a.M - 1);
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            const int c = 2 * st + half;
            qf[x][st] = 8 * c < a.K ? *(const qk_u32x4*)(q + qr * a.a_sm + 8 * c) : zero;
        }
    }
    // K block kb -> LDS buffer buf: wavefront w, step u copies rows (4u + w) RPI .. +RPI-1; lane L
    // writes row (4u + w) RPI + L / CH, position L % CH, holding global chunk (L % CH) ^ row_swz(row).
    // Rows past N and chunks past K read clamped in-range addresses; their values are never used.
    // Lane offsets are 32-bit from the block's base (the launcher checks 128 b_sn fits).
    const int bsn = (int)a.b_sn;
    auto copy_k = [&](int64_t kb, int buf) {
        const T* kblk = k + kb * kMfmaBlock * a.b_sn;
        const int lim = (int)min((int64_t)kMfmaBlock - 1, a.N - 1 - kb * kMfmaBlock);
#pragma unroll
        for (int u = 0; u < CH / 2; ++u) {
            const int slot = 4 * u + wave;
            const int row = slot * RPI + lane / CH;
            const int c = (lane % CH) ^ row_swz<CH>(row);
            const int kc = 8 * c < a.K ? 8 * c : 0;
            dma16(kblk + (min(row, lim) * bsn + kc), lds + buf * kRowBufBytes + slot * 1024);
        }
    };
    int koff[2], ksw[2];
#pragma unroll
    for (int y = 0; y < 2; ++y) {
        const int kr = (wave & 1) * 64 + 32 * y + r;
        koff[y] = kr * RB;
        ksw[y] = row_swz<CH>(kr);
    }
    copy_k(kb_begin, 0);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the first K block and the Q fragments
    __syncthreads();
    for (int64_t kb = kb_begin; kb < kb_end; ++kb) {
        const int buf = (int)((kb - kb_begin) & 1);
        if (kb + 1 < kb_end) copy_k(kb + 1, buf ^ 1);
        qk_lds_u8* kl = lds + buf * kRowBufBytes;
        const int64_t j0 = kb * kMfmaBlock + (wave & 1) * 64;
        // Bias of rows 32 x .. +31 of the wavefront's block; rows and columns past
        // the end repeat the last one. (The row and lane are hidden from the compiler,
        // which would otherwise keep every row's address over the K blocks and spill.)
        [[maybe_unused]] float bias[32];
        auto load_bias = [&](int x) {
            int ln = lane, row0 = (int)min(i0 + 32 * x, a.M - 1);
            int left = (int)(a.M - 1 - row0);
            asm volatile("" : "+v"(ln), "+s"(left));
            const float* bb = a.bias + bt * a.bias_sb + row0 * a.bias_sm;
            if constexpr (VEC) {
                bb += min(j0 + 4 * (ln & 15), a.N - 4);
#pragma unroll
                for (int it = 0; it < 8; ++it) {
                    const qk_f32x4 v = *(const qk_f32x4*)(bb + min(4 * it + (ln >> 4), left) * a.bias_sm);
#pragma unroll
                    for (int u = 0; u < 4; ++u) bias[4 * it + u] = v[u];
                }
            } else {
                bb += min(j0 + ln, a.N - 1) * a.bias_sn;
#pragma unroll
                for (int it = 0; it < 32; ++it) {
                    bias[it] = *bb;
                    bb += it < left ? a.bias_sm : 0;
                }
            }
        };
        if constexpr ((POST & QK_POST_BIAS) != 0) load_bias(0);
        qk_f32x16 acc[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[x][y][e] = 0.0f;
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            const int c = 2 * st + half;
            const bool kin = 8 * c < a.K;
            qk_u32x4 kf[2];
#pragma unroll
            for (int y = 0; y < 2; ++y) kf[y] = kin ? lds_read16(kl + koff[y] + 16 * (c ^ ksw[y])) : zero;
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = QkMfma<T>::run(kf[y], qf[x][st], acc[x][y]);
        }
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): K block kb+1 has landed
        __syncthreads();                      // ... for every wavefront; buffer `kl` is free for staging
        // Epilogue through a 32-row buffer of this wavefront (the block of K is no
        // longer read), 32-bit lane offsets from the wavefront's block (the launcher
        // checks that 64 rows and 64 columns of strides fit).
        qk_lds_u8* stg = kl + wave * 32 * 256;
        float* cw = a.c + bt * a.c_sb + i0 * a.c_sm + j0 * a.c_sn;
        int csm = (int)a.c_sm;
        const int csn = (int)a.c_sn;
        if constexpr ((POST & QK_POST_BIAS) != 0) asm volatile("" : "+s"(csm));  // (as above)
        auto post = [&](float v, float b) {
#pragma clang fp contract(off)  // (a lambda's body does not take the function's pragma)
            if (a.has_scale) v = v * a.scale;
            if constexpr ((POST & QK_POST_BIAS) != 0) v = v + b;
            if constexpr ((POST & QK_POST_CAP) != 0) v = a.softcap * tanhf(v / a.softcap);
            return v;
        };
        // (with registers held for the bias every index into them must be constant)
        constexpr bool BIASED = (POST & QK_POST_BIAS) != 0;
#pragma unroll
        for (int x = 0; x < 2; ++x) {
#pragma unroll
            for (int y = 0; y < 2; ++y)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int chunk = 8 * y + 2 * g + half;
                    lds_write_f4(stg + r * 256 + 16 * (chunk ^ (r & 15)),
                                 qk_f32x4{acc[x][y][4 * g], acc[x][y][4 * g + 1], acc[x][y][4 * g + 2],
                                          acc[x][y][4 * g + 3]});
                }
            // (the buffer is the wavefront's own and its LDS operations stay in order)
            asm volatile("" ::: "memory");
            if constexpr (VEC) {
                const int col = 4 * (lane & 15);
                auto rows4 = [&](int it) {
                    const int row = 4 * it + (lane >> 4);
                    const int rr = 32 * x + row;  // row in the wavefront's block
                    if (i0 + rr >= a.M || j0 + col >= a.N) return;
                    const qk_f32x4 raw = lds_read_f4(stg + row * 256 + 16 * ((lane & 15) ^ (row & 15)));
                    qk_f32x4 v;
#pragma unroll
                    for (int u = 0; u < 4; ++u) v[u] = post(raw[u], BIASED ? bias[4 * it + u] : 0.0f);
                    *(qk_f32x4*)(cw + (rr * csm + col)) = v;
                };
                // without a bias, two rows of stores per unrolled step: more would hoist every row's
                // address out of the K-block loop and leave too few registers for two wavefronts per SIMD
                if constexpr (BIASED) {
#pragma unroll
                    for (int it = 0; it < 8; ++it) rows4(it);
                } else {
#pragma unroll 2
                    for (int it = 0; it < 8; ++it) rows4(it);
                }
            } else {
                // Eight rows at a time are read before the first is stored: a row that is
                // read under its own bounds check waits for its LDS read alone (9 tiles 230 x
                // 110 x 128 9.8 us so, 7.7 now). Rows past the end hold products that are not
                // stored.
                const int rows = (int)min((int64_t)32, a.M - i0 - 32 * x);  // uniform
                const bool in_col = j0 + lane < a.N;
                auto rows8 = [&](int r0) {
                    if (r0 >= rows) return;
                    float v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        v[u] = *(const qk_lds_f32*)(stg + (r0 + u) * 256 + 16 * ((lane >> 2) ^ ((r0 + u) & 15)) + 4 * (lane & 3));
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = post(v[u], BIASED ? bias[r0 + u] : 0.0f);
                    if (!in_col) return;
                    float* cr = cw + ((32 * x + r0) * csm + lane * csn);
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (r0 + u < rows) cr[u * csm] = v[u];
                };
                if constexpr (BIASED) {
#pragma unroll
                    for (int r0 = 0; r0 < 32; r0 += 8) rows8(r0);
                } else {
#pragma unroll 1
                    for (int r0 = 0; r0 < 32; r0 += 8) rows8(r0);
                }
            }
            if constexpr (BIASED) {
                if (x == 0) load_bias(1);
            }
            asm volatile("" ::: "memory");  // the next pass reuses the buffer
        }
        __syncthreads();  // the next K block's copy reuses the buffers
    }
}

// K blocks per workgroup of the row kernel: runs of 4, shorter where that would
// leave fewer than one round of workgroups (two per CU on 256 CUs), longer
// beyond 4096 workgroups. Measured on 32 heads x D 128: 1024^2 0.029 ms with 4
// (0.033 with 2, 0.040 with 1 or 8), 2048^2 0.124 ms with 4 (0.164 with 8 or
// 16), 4096^2 0.463-0.465 ms with 8 or 16 (0.513 with 32).
inline int64_t rows_blocks_per_workgroup(int64_t tiles, int64_t nkb) {
    int64_t tpw = tiles / 4096;
    if (tpw < 4) tpw = std::min<int64_t>(4, std::max<int64_t>(1, tiles / 512));
    return std::min(tpw, nkb);
}

// Soft-capped calls are bound by the vector ALU, so the time is that of the
// busiest CU: rounds of two runs of blocks (row kernel) or of three blocks
// (one-block kernel, whose third workgroup per CU hides less else). Where the
// runs leave more of their last round empty, the one-block kernel is faster.
// Measured, one-block / row kernel (us): 11 tiles 924 x 988 x 32, 704 blocks, 17.4 /
// 20.2; 63 tiles 1122 x 48 x 128 with a bias, 567 blocks, 18.8 / 24.8; 35 tiles 645 x
// 776 x 64, 1470 blocks, 31.7 / 37.0; against 56 tiles 241 x 1092 x 16 with a bias,
// 1008 blocks, 29.5 / 24.0; 12 tiles 1363 x 372 x 64, 396 blocks, 15.3 / 14.3. (Without
// 16-byte rows the row kernel is faster throughout.)
inline bool block_kernel_fills_better(int64_t batch, int64_t nqb, int64_t nkb) {
    const int64_t blocks = batch * nqb * nkb, tpw = rows_blocks_per_workgroup(blocks, nkb);
    const int64_t runs = batch * nqb * ((nkb + tpw - 1) / tpw);
    const int64_t run_rounds = (runs + 2 * kComputeUnits - 1) / (2 * kComputeUnits);
    const int64_t block_rounds = (blocks + 3 * kComputeUnits - 1) / (3 * kComputeUnits);
    return 3 * block_rounds < 2 * tpw * run_rounds;
}

template <typename T, int CH, int POST>
void launch_rows_post(const QkScoreArgs& x, bool vec, int64_t nqb, int64_t npieces, int tpw, hipStream_t s) {
    const dim3 grid((unsigned)(x.batch * nqb * npieces));
    if (vec) hipLaunchKernelGGL((qk_score_mfma_rows_kernel<T, CH, POST, true>), grid, dim3(256), 0, s, x, nqb, npieces, tpw);
    else hipLaunchKernelGGL((qk_score_mfma_rows_kernel<T, CH, POST, false>), grid, dim3(256), 0, s, x, nqb, npieces, tpw);
}
template <typename T, int CH>
void launch_rows_ch(const QkScoreArgs& x, bool vec, int64_t nqb, int64_t npieces, int tpw, hipStream_t s) {
    const bool bias = x.bias != nullptr, cap = x.softcap > 0.0f;
    if (bias && cap) launch_rows_post<T, CH, QK_POST_BIAS_CAP>(x, vec, nqb, npieces, tpw, s);
    else if (bias) launch_rows_post<T, CH, QK_POST_BIAS>(x, vec, nqb, npieces, tpw, s);
    else if (cap) launch_rows_post<T, CH, QK_POST_CAP>(x, vec, nqb, npieces, tpw, s);
    else launch_rows_post<T, CH, QK_POST_NONE>(x, vec, nqb, npieces, tpw, s);
}
template <typename T>
hipError_t launch_rows_k(const QkScoreArgs& x, bool vec, int64_t nqb, int64_t npieces, int tpw, hipStream_t s) {
    if (x.K <= 32) launch_rows_ch<T, 4>(x, vec, nqb, npieces, tpw, s);
    else if (x.K <= 64) launch_rows_ch<T, 8>(x, vec, nqb, npieces, tpw, s);
    else launch_rows_ch<T, 16>(x, vec, nqb, npieces, tpw, s);
    return hipGetLastError();
}

}  // namespace

bool qk_score_mfma_supported(const QkScoreArgs& a, int dtype) {
    if (dtype != DT_BF16 && dtype != DT_F16) return false;
    const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    return a.a_sk == 1 && a.b_sk == 1 && a.K % 8 == 0 && a.a_sm % 8 == 0 && a.b_sn % 8 == 0 &&
           a.a_sb % 8 == 0 && a.b_sb % 8 == 0 && al16(a.q) && al16(a.k);
}

hipError_t launch_qk_score_mfma(const QkScoreArgs& a, int dtype, hipStream_t s) {
    if (a.batch <= 0 || a.M <= 0 || a.N <= 0 || a.K <= 0) return hipSuccess;
    if (!qk_score_mfma_supported(a, dtype)) return hipErrorInvalidValue;
    const auto al16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    const bool c_vec = a.c_sn == 1 && a.c_sm % 4 == 0 && a.c_sb % 4 == 0 && al16(a.c);
    const bool b_vec = a.bias == nullptr ||
                       (a.bias_sn == 1 && a.bias_sm % 4 == 0 && a.bias_sb % 4 == 0 && al16(a.bias));
    // K <= 128, lane offsets within 32 bits: the row kernel.
    const int64_t lim31 = int64_t(1) << 31;
    const bool rows = a.K <= 128 && (kMfmaBlock - 1) * a.b_sn + a.K < lim31 &&
                      63 * (a.c_sm + a.c_sn) + 4 < lim31 && a.b_sn >= 0 && a.c_sm >= 0 && a.c_sn >= 0;
    const int64_t nqb = (a.M + kMfmaBlock - 1) / kMfmaBlock, nkb = (a.N + kMfmaBlock - 1) / kMfmaBlock;
    const bool vec = c_vec && b_vec && a.N % 4 == 0;
    if (rows && !(a.softcap > 0.0f && vec && block_kernel_fills_better(a.batch, nqb, nkb))) {
        const int64_t max_grid = kMaxWorkItems / 256;  // workgroups of a launch
        for (int64_t b0 = 0; b0 < a.batch;) {
            QkScoreArgs x = a;
            x.batch = std::min<int64_t>(a.batch - b0, std::max<int64_t>(1, max_grid / (nqb * nkb)));
            x.q = (const char*)a.q + b0 * a.a_sb * 2;
            x.k = (const char*)a.k + b0 * a.b_sb * 2;
            x.c = a.c + b0 * a.c_sb;
            if (a.bias != nullptr) x.bias = a.bias + b0 * a.bias_sb;
            const int64_t tiles = x.batch * nqb * nkb;
            const int64_t tpw = rows_blocks_per_workgroup(tiles, nkb);
            const int64_t npieces = (nkb + tpw - 1) / tpw;
            const hipError_t e = dtype == DT_BF16 ? launch_rows_k<__bf16>(x, vec, nqb, npieces, (int)tpw, s)
                                                  : launch_rows_k<_Float16>(x, vec, nqb, npieces, (int)tpw, s);
            if (e != hipSuccess) return e;
            b0 += x.batch;
        }
        return hipSuccess;
    }
    for (int64_t b0 = 0; b0 < a.batch; b0 += kMaxGridZ) {
        QkScoreArgs x = a;
        x.vec4 = c_vec && b_vec;
        x.batch = std::min<int64_t>(kMaxGridZ, a.batch - b0);
        x.q = (const char*)a.q + b0 * a.a_sb * 2;
        x.k = (const char*)a.k + b0 * a.b_sb * 2;
        x.c = a.c + b0 * a.c_sb;
        if (a.bias != nullptr) x.bias = a.bias + b0 * a.bias_sb;
        const dim3 grid((unsigned)((a.N + kMfmaBlock - 1) / kMfmaBlock),
                        (unsigned)((a.M + kMfmaBlock - 1) / kMfmaBlock), (unsigned)x.batch);
        // The soft-cap epilogue is a separate instantiation: it needs many more
        // registers, which would lower the occupancy of the common case.
        const bool cap = a.softcap > 0.0f;
        if (dtype == DT_BF16) {
            if (cap) hipLaunchKernelGGL((qk_score_mfma_kernel<__bf16, true>), grid, dim3(256), 0, s, x);
            else hipLaunchKernelGGL((qk_score_mfma_kernel<__bf16, false>), grid, dim3(256), 0, s, x);
        } else {
            if (cap) hipLaunchKernelGGL((qk_score_mfma_kernel<_Float16, true>), grid, dim3(256), 0, s, x);
            else hipLaunchKernelGGL((qk_score_mfma_kernel<_Float16, false>), grid, dim3(256), 0, s, x);
        }
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

namespace {
template <int PT>
hipError_t launch_qk_exact(const QkScoreArgs& x, int dtype, hipStream_t s) {
    const dim3 grid((unsigned)((x.N + 16 * PT - 1) / (16 * PT)), (unsigned)((x.M + 16 * PT - 1) / (16 * PT)),
                    (unsigned)x.batch);
    switch (dtype) {
        case DT_F32: hipLaunchKernelGGL((qk_score_kernel<float, PT>), grid, dim3(256), 0, s, x); break;
        case DT_BF16: hipLaunchKernelGGL((qk_score_kernel<__bf16, PT>), grid, dim3(256), 0, s, x); break;
        case DT_F16: hipLaunchKernelGGL((qk_score_kernel<_Float16, PT>), grid, dim3(256), 0, s, x); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
}  // namespace

hipError_t launch_qk_score(const QkScoreArgs& a, int dtype, hipStream_t s) {
    if (a.batch <= 0 || a.M <= 0 || a.N <= 0 || a.K <= 0) return hipSuccess;
    const size_t esz = dtype == DT_F32 ? 4 : 2;
    for (int64_t b0 = 0; b0 < a.batch; b0 += kMaxGridZ) {
        QkScoreArgs x = a;
        x.batch = std::min<int64_t>(kMaxGridZ, a.batch - b0);
        x.q = (const char*)a.q + b0 * a.a_sb * esz;
        x.k = (const char*)a.k + b0 * a.b_sb * esz;
        x.c = a.c + b0 * a.c_sb;
        if (a.bias != nullptr) x.bias = a.bias + b0 * a.bias_sb;
        x.vec4 = a.c_sn == 1 && a.c_sm % 4 == 0 && a.c_sb % 4 == 0 && (reinterpret_cast<uintptr_t>(a.c) & 15u) == 0;
        // 64x64 blocks where they give every CU three or more, for a short k (their
        // prologue and epilogue weigh more; a bias doubles what the epilogue waits for) many
        // more, and where they pad little more than 32x32 ones, which take every other call
        // (us, 32x32 / 64x64: 16 tiles 512^2 x 64, 1024 blocks, 24.4 / 20.3; 15 x 332 x 508 x
        // 128, 720, 30.5 / 27.4; 5 x 753 x 605 x 64, 600, 15.8 / 17.2; 10 x 707 x 538 x 32, 1080,
        // 14.3 / 17.6; 24 x 321 x 1656 x 32, 3744, 41.1 / 36.9; 57 x 317 x 1020 x 16, 4560, 40.2 /
        // 29.6; with a bias 20 x 288 x 797 x 64, 1300, 29.4 / 33.9, 31 x 887 x 896 x 48, 6076,
        // 98.4 / 78.7; 57 x 1193 x 22 x 24, twice the padding, 10.3 / 18.8). 128x128 blocks gained
        // 1 % at 32 tiles 1024^2 x 128 and lost 35 % at 8 tiles 1100^2 x 96.
        const int64_t blocks64 = x.batch * ((x.M + 63) / 64) * ((x.N + 63) / 64);
        const int64_t blocks32 = x.batch * ((x.M + 31) / 32) * ((x.N + 31) / 32);
        const int64_t k = std::min<int64_t>(x.K, 128);
        const bool wide = blocks64 >= 3 * kComputeUnits && blocks64 * k >= (x.bias != nullptr ? 96 * 1024 : 48 * 1024) &&
                          200 * blocks64 <= 63 * blocks32;  // 1.26 times the area
        const hipError_t e = wide ? launch_qk_exact<4>(x, dtype, s) : launch_qk_exact<2>(x, dtype, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Plain strided fp32 tile product (the tile-GEMM seam,
// src/onednn_flash/tile_kernel.cpp:67-86): the score kernel with no post-ops.
hipError_t launch_tile_gemm(const float* a, const float* b, float* c, int m, int n, int k,
                            int64_t asm_, int64_t ask, int64_t bsk, int64_t bsn, int64_t csm,
                            int64_t csn, hipStream_t s) {
    QkScoreArgs x{};
    x.batch = 1;
    x.M = m;
    x.N = n;
    x.K = k;
    x.q = a;
    x.k = b;
    x.c = c;
    x.a_sm = asm_;
    x.a_sk = ask;
    x.b_sk = bsk;
    x.b_sn = bsn;
    x.c_sm = csm;
    x.c_sn = csn;
    return launch_qk_score(x, DT_F32, s);
}

}  // namespace ofh
