// Register-operand main kernel for gfx950: dK, dV and dQ for launches with
// enough tiles to fill the chip with two (D 128) or three (D 64) small
// workgroups per CU.  Same two job roles and row statistics as
// bwd_main_kernel (fa3_bwd_main_kernel.h); what differs is how a workgroup
// is built:
//
//  * 4 waves, each doing everything for its own 32 keys (dKV role) or 32
//    query rows (dQ role): S and dP of 32 streamed rows x 32 resident
//    columns, softmax, and the output products.
//  * P and dS never leave the registers.  With v_mfma_f32_16x16x32 the score
//    accumulators hold, per lane, rows 4 g .. 4 g + 3 of both 16-row blocks
//    of one column; rounded and packed they are the B operand of the output
//    product as it stands, with its 32 k-slots standing for the rows in the
//    order (4 g + 0..3, 16 + 4 g + 0..3) -- and the transposed A operand is
//    simply read in that order.
//  * the streamed tiles go through two LDS stages filled by direct-to-LDS
//    loads; one barrier per 64 streamed rows.
//  * two (D 128) or three (D 64) workgroups share a CU, so one's prologue,
//    epilogue and barriers overlap another's products, and the hardware's
//    dispatch needs no job queue.
//
// What bounds it.  Large launches are limited by power, not by issue slots:
// a long backward clocks at 1.5-1.75 GHz, so energy per product sets the
// time.  Register-only loops of the two MFMA shapes on N(0, 1) data ran at
// 1 635 (32x32x16) and 1 889 TFLOP/s (16x16x32) in fp16, 1 704 and 1 982 in
// bf16: hence 16x16x32 everywhere (the same kernel with 32x32x16: B2 H16
// S8192 D64 full 1 780 us against 1 606, B2 H16 S4096 D128 full 837 against
// 750).  Against bwd_main_kernel a step also moves no P / dS through LDS
// and a streamed tile serves 128 resident rows instead of 64, half the L2
// traffic.  Measured against it (both in turn on one GPU), whole backwards:
// B2 H16 S8192 D64 full 1 984 -> 1 624 us, B2 Hq32 Hkv8 S4096 D128 causal 963
// -> 845, B1 Hq32 Hkv1 S4096 D128 causal 493 -> 442, B2 Hq32 Hkv8 S2048 D128
// BSHD bf16 causal 257 -> 230, B4 H16 S1024 D128 causal bf16 92.6 -> 69.9, B2
// H12 S1664 D64 full 77.8 -> 64.9.
// Small launches are limited by one wave's chain (a wave alone on its SIMD
// runs a 32 x 32 step in ~2 600 cycles, 1 024 of them MFMA), so launches
// with few jobs stay with bwd_main_kernel (reg_plan, fa3_bwd_main.hip).
//
// The operands stay unscaled: exp2(S c - lse2) takes one fma per element,
// for any c, and K or Q is not rounded again (error against fp64 in fp16
// 3.0e-4, 3.7e-4 with scaled operands).
#pragma once

#include "fa3_bwd_main_kernel.h"

namespace fa3 {

// How a launch cuts its jobs: keys of a dKV job = 128 / split_kv, query rows
// of a dQ job = 128 / split_q.  split_kv 0 (causal): the first `halved` of the
// 128-key tiles, the longest, as two 64-key jobs, the others whole.
struct RegPlan {
    bool on = false;  // false: the launch runs bwd_main_kernel,
    bool unscaled = false;  // and its unscaled instantiation at every scale
    int split_kv = 1;
    int split_q = 1;
    int halved = 0;
};

struct RegArgs {
    const _Float16* q;
    const _Float16* k;
    const _Float16* v;
    const _Float16* dout;
    const float* nlse2;   // [B*Hq*S], -LSE log2 e
    const float* ndelta;  // [B*Hq*S], -delta
    void* dq;
    void* dk;  // the outputs, or the head-split plan's fp32 contributions
    void* dv;
    // fp32 instead of 16-bit stores: dkv_f32 with the head split, dq_f32 never
    // (0) -- the branch stays because without it the compiler spills 9 vector
    // registers of the D 128 full-attention kernels.
    int dq_f32, dkv_f32;
    int q_rs, q_hs, kv_rs, kv_hs;  // as in FusedArgs
    int o_rs, o_hs, o_heads;       // dK / dV: row stride, head stride, heads
    int seqlen, heads_q, heads_kv, group;
    int heads;   // query heads a dKV job streams: group / chunks
    int chunks;  // dKV jobs per key tile
    int halved;  // kSplitKv 0: the first `halved` 128-key tiles run as 64-key jobs
    float scale_log2, scale;
    // job map (job_of)
    int n_groups, jobs_per_group, map_radix, xcd_parts, xcd_interleave, xcd_vgroups, xcd_mode;
    FastDiv div_hkv, div_group, div_chunks, div_parts, div_radix, div_jpg, div_groups;
};

namespace {

constexpr int kRegWaves = 4;
constexpr int kRegThreads = kRegWaves * kWave;
template <int D>
struct RegCfg {
    static constexpr int kTileBytes = 64 * D * 2;  // one streamed [64][D] tile
    static constexpr int kRowsBytes = 512;         // -lse2, -delta of 64 rows
    static constexpr int kStageBytes = 2 * kTileBytes + kRowsBytes;
    static constexpr int kLd = kTileBytes / (kRegWaves * 1024);  // loads per wave and tile
    static constexpr int kKs = D / 32;                           // k-steps of S / dP
    static constexpr int kDB = D / 16;                           // 16-column blocks of D
    static constexpr int kBytes = 2 * kStageBytes;
    // LDS operands on their way while one is in use: during the first row
    // block's scores, the second's, and in the output products.  D 128: as
    // many as the registers free at that point allow (4, 3, 6 against 2, 2, 2:
    // -2 % for large launches, -5 % where waves run alone); D 64, three waves
    // per SIMD, is 1.5 % faster with few.
    static constexpr int kAhead0 = D == 128 ? 4 : 2;
    static constexpr int kAhead1 = D == 128 ? 3 : 2;
    static constexpr int kAheadG = D == 128 ? 6 : 2;
    static_assert(kDB * 2 * 1024 * kRegWaves <= kBytes, "the pieces' exchange fits the stages");
};

// 8 fp32 values of one column to a B operand
template <bool kBf16>
__device__ __forceinline__ f16x8 pack8(const float* x) {
    f16x8 r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r[i] = to16<kBf16>(x[i]);
    return r;
}

// D 64: the MFMA phases at raised priority, so that a wave's softmax does not
// hold back another's products (B2 H16 S4096 D64 causal -2.6 %, B2 H12 S1664
// D64 full -1.7 %; D 128, two waves per SIMD, +0.5 to +1 %).
template <int D, int kPrio>
__device__ __forceinline__ void mm_prio() {
    if constexpr (D == 64) __builtin_amdgcn_s_setprio(kPrio);
}

__device__ __forceinline__ void wall() { __builtin_amdgcn_sched_barrier(0); }

// Row-major [rows][D] 16-bit tile with 16-byte chunks XOR-swizzled per row:
// byte offset of a chunk.  Row bits 0, 1 (D 64: bit 1; bit 0 picks half of a
// 256-byte bank line) move the chunk by 4 and 8, bit 2 by 2 and bit 3 by 1,
// so that both reads below touch every bank evenly:
//   ds_read_b128 of 16 rows: the 16 lanes served together (equal lane bit 5
//     and parity of bits 2..4) get 16 distinct chunks;
//   ds_read_b64_tr_b16 of 16 rows x 2 chunks: served 32 lanes (8 rows) at a
//     time, whose 16 chunks are distinct -- with row bits 2 and 3 the other
//     way round (tile_off, made for reads of 4 rows x 4 chunks) rows 4 .. 7
//     meet rows 0 .. 3 on the same banks: 28 % of the LDS cycles were
//     conflicts, now none, and launches 0.4 to 1.1 % faster (B2 Hq32 Hkv8
//     S4096 D128 causal 826 -> 819 us, B2 H16 S4096 D64 causal 217 -> 215).
template <int D>
__device__ __forceinline__ uint32_t reg_swz(int row) {
    const int hi = (((row >> 2) & 1) << 1) | ((row >> 3) & 1);
    return D == 128 ? ((row & 3) << 2) | hi : (((row >> 1) & 1) << 2) | hi;
}
template <int D>
__device__ __forceinline__ uint32_t reg_tile_off(int row, int chunk) {
    return (uint32_t)(row * (D * 2)) + (((uint32_t)chunk ^ reg_swz<D>(row)) & (D / 8 - 1)) * 16;
}

// LDS addresses of one lane's operands: the k-step / column-block part of an
// address is an XOR of a constant, everything else an immediate offset.
template <int D>
struct RegReader {
    uint32_t a, t;
    __device__ __forceinline__ RegReader(int lane, int row0) {
        const int l16 = lane & 15, g = lane >> 4;
        a = reg_tile_off<D>(l16, p1_chunk<D>(0, g));
        t = reg_tile_off<D>(4 * g + (l16 >> 2), (l16 & 3) >> 1) + (l16 & 1) * 8;
        a += row0 * 2 * D;  // (row0 a multiple of 32: no bit of the XORed field)
        t += row0 * 2 * D;
    }
    // (recomputed per use: held, the XORed addresses cost D 128 its registers)
    __device__ __forceinline__ void opaque() {
        if constexpr (D == 128) __asm__ volatile("" : "+v"(a), "+v"(t));
    }
    // A operand of k-step ks (D chunk p1_chunk(ks, g)) of rows 16 m + l16
    __device__ __forceinline__ f16x8 row(const FA3_LDS char* tile, int m, int ks) const {
        return lds_read_b128(tile + 16 * m * 2 * D, a ^ (uint32_t)(16 * ks));
    }
    // transposed A operand: D column 16 db + l16, rows 32 r + 4 g + 0..3 and + 16
    __device__ __forceinline__ f16x8 tr(const FA3_LDS char* tile, int r, int db) const {
        const FA3_LDS char* p = tile + 32 * r * 2 * D;
        const uint32_t o = t ^ (uint32_t)(32 * db);
        return concat4(lds_read_tr4(p, o), lds_read_tr4(p + 16 * 2 * D, o));
    }
};

// Direct-to-LDS copy of a row-major [64][D] tile (row stride rs elements) by
// the 4 waves; one per-lane offset (reg_load_off) serves all of a wave's
// loads: consecutive 1 KiB blocks differ by whole rows and an XOR.
template <int D>
__device__ __forceinline__ uint32_t reg_load_off(int lane, int rs) {
    constexpr int kC = D / 8;  // 16-byte chunks per row
    const int row = lane / kC;
    return (uint32_t)(row * rs * 2) + (reg_tile_off<D>(row, lane % kC) - (uint32_t)(row * D * 2));
}
template <int D>
__device__ __forceinline__ void reg_load_tile(FA3_LDS char* tile, const _Float16* src, uint32_t v,
                                              int w, int rs) {
    constexpr int kLd = RegCfg<D>::kLd, kRows = 512 / D;  // rows per 1 KiB block
#pragma unroll
    for (int j = 0; j < kLd; ++j)
        __builtin_amdgcn_global_load_lds(
            (const void*)((const char*)(src + (size_t)(16 * w + kRows * j) * rs) +
                          (v ^ (reg_swz<D>(kRows * j) * 16))),
            (FA3_LDS void*)(tile + (w * kLd + j) * 1024), 16, 0, 0);
}

// s0[m][n] += X0 B0, s1[m][n] += X1 B1 over D, for the 32 streamed rows 32 r
// .. (blocks m) and the 32 resident columns (blocks n).
template <int D, bool kBf16>
__device__ __forceinline__ void reg_scores(const RegReader<D>& rd, const FA3_LDS char* x0,
                                           const FA3_LDS char* x1, int r,
                                           const f16x8 (&b0)[2][D / 32],
                                           const f16x8 (&b1)[2][D / 32], f32x4 (&s0)[2][2],
                                           f32x4 (&s1)[2][2]) {
    constexpr int kKs = D / 32, kN = 4 * kKs;
    f16x8 f[kN];
    using C = RegCfg<D>;
    // Operand i: tile, row block m and k-step.  D 64 takes both row blocks of
    // a k-step in turn and the resident blocks n forth and back, so that
    // consecutive products differ in one operand only (less switching in the
    // matrix unit's inputs: B2 H16 S8192 D64 full -0.4 %); at D 128 that
    // order keeps both blocks' accumulators live, which its registers do not allow.
    constexpr bool kKsOuter = D == 64;
    auto tile_of = [](int i) { return kKsOuter ? (i >> 1) & 1 : i & 1; };
    auto m_of = [](int i) { return kKsOuter ? i & 1 : (i >> 1) / kKs; };
    auto ks_of = [](int i) { return kKsOuter ? i >> 2 : (i >> 1) % kKs; };
    auto read = [&](int i) {
        f[i] = rd.row(tile_of(i) ? x1 : x0, 2 * r + m_of(i), ks_of(i));
    };
#pragma unroll
    for (int i = 0; i < C::kAhead0; ++i) read(i);
    int done = C::kAhead0;
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        const int m = m_of(i), ks = ks_of(i);
        const int want = i + 1 + (i < kN / 2 - 1 ? C::kAhead0 : C::kAhead1);
        wall();
        if (done < want && done < kN) read(done++);
        wall();
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = kKsOuter ? j ^ (i & 1) : j;
            if (tile_of(i)) s1[m][n] = mfma_16x16x32<kBf16>(f[i], b1[n][ks], s1[m][n]);
            else s0[m][n] = mfma_16x16x32<kBf16>(f[i], b0[n][ks], s0[m][n]);
        }
    }
    wall();
}

// g0[db][n] += X0^T B0 (and g1[db][n] += X1^T B1 when kTwo) over the 32
// streamed rows 32 r ..
template <int D, bool kBf16, bool kTwo>
__device__ __forceinline__ void reg_grads(const RegReader<D>& rd, const FA3_LDS char* x0,
                                          const FA3_LDS char* x1, int r, const f16x8 (&b0)[2],
                                          const f16x8 (&b1)[2], f32x4 (&g0)[D / 16][2],
                                          f32x4 (&g1)[D / 16][2]) {
    constexpr int kN = (kTwo ? 2 : 1) * (D / 16);
    f16x8 f[kN];
    // Operand i: two column blocks of one product, then two of the other, n
    // forth and back: consecutive products differ in one operand only, half
    // as much switching as one block of each in turn (D 128 -0.3 to -0.5 %,
    // D 64 -0.2 to -0.5 %).
    auto second = [](int i) { return kTwo && (i & 2); };
    auto db_of = [](int i) { return kTwo ? ((i >> 2) << 1) | (i & 1) : i; };
    auto read = [&](int i) { f[i] = rd.tr(second(i) ? x1 : x0, r, db_of(i)); };
    constexpr int kA = RegCfg<D>::kAheadG;
#pragma unroll
    for (int i = 0; i < 2; ++i) read(i);
    wall();
#pragma unroll
    for (int i = 2; i < kA; ++i) read(i);
#pragma unroll
    for (int i = 0; i < kN; ++i) {
        wall();
        if (i + kA < kN) read(i + kA);
        wall();
        const int db = db_of(i);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = j ^ (i & 1);
            if (second(i)) g1[db][n] = mfma_16x16x32<kBf16>(f[i], b1[n], g1[db][n]);
            else g0[db][n] = mfma_16x16x32<kBf16>(f[i], b0[n], g0[db][n]);
        }
    }
    wall();
}

// A wave's 32 x 16 NB output block (acc[db][n]: row 16 n + l16, columns 16
// db + 4 g + i) times mul to `out` (element `base`, row stride rs): fp32
// directly, 16-bit through the wave's own NB KiB of LDS at st, so that every
// global store writes whole row segments.
template <int NB, bool kBf16>
__device__ __forceinline__ void reg_store(bool f32, void* out, size_t base, int rs,
                                          const f32x4 (*acc)[2], float mul, int lane,
                                          FA3_LDS char* st) {
    const int l16 = lane & 15, g = lane >> 4;
    if (f32) {
        float* o = (float*)out + base + (size_t)l16 * rs + 4 * g;
#pragma unroll
        for (int db = 0; db < NB; ++db)
#pragma unroll
            for (int n = 0; n < 2; ++n)
                *(f32x4*)(o + (size_t)16 * n * rs + 16 * db) = acc[db][n] * mul;
        return;
    }
#pragma unroll
    for (int db = 0; db < NB; ++db)
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            f16x4 v;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = to16<kBf16>(acc[db][n][e] * mul);
            const uint32_t off =
                NB == 2 ? stage64_off(16 * n + l16, 2 * db + (g >> 1), g & 1)
                        : (uint32_t)(db >> 2) * 4096 +
                              stage128_off(16 * n + l16, 2 * (db & 3) + (g >> 1), g & 1);
            lds_write_b64(st, off, v);
        }
    _Float16* o = (_Float16*)out + base;
    if constexpr (NB == 2) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int r = stage64_row(j, lane), c = lane & 3;
            const f16x8 x = stage_fix(lds_read_b128(st, stage64_chunk(r, c)), r);
            store_out(o + (size_t)r * rs + 8 * c, x);
        }
    } else {
#pragma unroll
        for (int pn = 0; pn < NB / 4; ++pn)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 8 * j + ((lane >> 2) & 7);
                const int c = (lane & 3) | ((lane >> 5) << 2);
                const f16x8 x =
                    stage_fix(lds_read_b128(st + pn * 4096, stage128_chunk(r, c)), r);
                store_out(o + (size_t)r * rs + 64 * pn + 8 * c, x);
            }
    }
}

// Two waves' partial sums meet in LDS: N accumulators out to slot, or in
// from it and added.
template <int N>
__device__ __forceinline__ void reg_put(FA3_LDS char* slot, const f32x4 (*acc)[2], int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int n = 0; n < 2; ++n)
            *(FA3_LDS f32x4*)(slot + (2 * i + n) * 1024 + lane * 16) = acc[i][n];
}
template <int N>
__device__ __forceinline__ void reg_add(const FA3_LDS char* slot, f32x4 (*acc)[2], int lane) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int n = 0; n < 2; ++n)
            acc[i][n] += *(const FA3_LDS f32x4*)(slot + (2 * i + n) * 1024 + lane * 16);
}

// Key tile kt (128 / kSplit keys) of KV head hkv in batch b, streaming the
// query tiles of `heads` query heads from h0 on; out head ho.
template <int D, bool kCausal, bool kBf16, int kSplit, bool kDebug, typename A>
__device__ __forceinline__ void reg_dkv(const A& a, int b, int hkv, int kt, int h0, int ho,
                                        FA3_LDS char* smem) {
    using C = RegCfg<D>;
    constexpr int kKb = kRegWaves / kSplit;  // 32-key blocks of the job
    const int tid = opaque_tid();
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kb = w & (kKb - 1), rs = w / kKb;
    const int l16 = lane & 15, g4 = lane >> 4;
    const int S = a.seqlen;
    const int key0 = (kt * kKb + kb) * 32;
    const int qa = kCausal ? (kt * kKb) >> 1 : 0, qb = S / 64;
    const int n_it = a.heads * (qb - qa);

    int ld_h = 0;
    size_t ld_e = q_elem<D>(a, b, h0, (qb - 1) * 64);
    size_t ld_row = ((size_t)b * a.heads_q + h0) * S + (qb - 1) * 64;
    const size_t step_e = (size_t)64 * a.q_rs;
    auto issue = [&](FA3_LDS char* st) {
        const int ln = opaque_tid() & 63;
        const uint32_t off = reg_load_off<D>(ln, a.q_rs);
        reg_load_tile<D>(st, a.q + ld_e, off, w, a.q_rs);
        reg_load_tile<D>(st + C::kTileBytes, a.dout + ld_e, off, w, a.q_rs);
        if (w < 2)
            __builtin_amdgcn_global_load_lds(
                (const void*)((w == 0 ? a.nlse2 : a.ndelta) + ld_row + ln),
                (FA3_LDS void*)(st + 2 * C::kTileBytes + 256 * w), 4, 0, 0);
        ld_e += (size_t)a.q_hs;
        ld_row += (size_t)S;
        if (++ld_h == a.heads) {
            ld_h = 0;
            ld_e -= (size_t)a.heads * a.q_hs + step_e;
            ld_row -= (size_t)a.heads * S + 64;
        }
    };
    FA3_LDS char* s0 = smem;
    FA3_LDS char* s1 = smem + C::kStageBytes;
    issue(s0);
    // resident B operands: K and V of keys key0 + 16 n + l16
    f16x8 kf[2][C::kKs], vf[2][C::kKs];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const size_t e = kv_elem<D>(a, b, hkv, key0 + 16 * n + l16);
#pragma unroll
        for (int s = 0; s < C::kKs; ++s) {
            kf[n][s] = *(const f16x8*)(a.k + e + 8 * p1_chunk<D>(s, g4));
            vf[n][s] = *(const f16x8*)(a.v + e + 8 * p1_chunk<D>(s, g4));
        }
    }
    f32x4 av[C::kDB][2], ak[C::kDB][2];
#pragma unroll
    for (int i = 0; i < C::kDB; ++i) {
        av[i][0] = av[i][1] = f32x4{};
        ak[i][0] = ak[i][1] = f32x4{};
    }
    const int rsub = 32 * rs;  // this wave's rows of a stage: all (kSplit 1), or 32 from here
    const RegReader<D> rd0(lane, rsub);
    const float c = a.scale_log2;
    int row0 = (qb - 1) * 64 + rsub - key0;  // this wave's first row of the stage relative to
    int head = 0;                            // its first key; the stage's head

    auto sub = [&](const FA3_LDS char* st, int r) {
        RegReader<D> rd = rd0;
        rd.opaque();
        const FA3_LDS char* tq = st;
        const FA3_LDS char* td = st + C::kTileBytes;
        const FA3_LDS f32x4* rows =
            (const FA3_LDS f32x4*)(st + 2 * C::kTileBytes + 4 * rsub + 128 * r) +
            ((opaque_tid() & 63) >> 4);
        debug_sync<kDebug>();
        if (!kCausal || row0 + 32 * r >= 0) {
            // [m][n]: rows 16 m + 4 g4 + i, keys 16 n + l16
            f32x4 s[2][2], dp[2][2], nl[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                dp[m][0] = dp[m][1] = rows[16 + 4 * m];
                s[m][0] = s[m][1] = f32x4{};
            }
            mm_prio<D, 1>();
            reg_scores<D, kBf16>(rd, tq, td, r, kf, vf, s, dp);
            mm_prio<D, 0>();
            nl[0] = rows[0];
            nl[1] = rows[4];
            float p[2][8], ds[2][8];  // [n][4 m + i]
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int m = j >> 2, i = j & 3;
                    p[n][j] = fast_exp2(__builtin_fmaf(s[m][n][i], c, nl[m][i]));
                    ds[n][j] = p[n][j] * dp[m][n][i];
                }
            if (kCausal && row0 + 32 * r < 32) {  // the diagonal block
                const int ln = opaque_tid() & 63, l16 = ln & 15, g4 = ln >> 4;  // (keeps this a branch)
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (16 * n + l16 > 16 * (j >> 2) + 4 * g4 + (j & 3)) {
                            p[n][j] = 0.f;
                            ds[n][j] = 0.f;
                        }
            }
            const f16x8 bp[2] = {pack8<kBf16>(p[0]), pack8<kBf16>(p[1])};
            const f16x8 bs[2] = {pack8<kBf16>(ds[0]), pack8<kBf16>(ds[1])};
            mm_prio<D, 1>();
            reg_grads<D, kBf16, true>(rd, td, tq, r, bp, bs, av, ak);
        }
        debug_sync<kDebug>();
    };
    int it = 0;
    auto stage = [&](FA3_LDS char* __restrict__ ld, const FA3_LDS char* __restrict__ st) {
        wait_vm_lgkm0<0>();
        barrier();
        if (++it < n_it) issue(ld);
        sub(st, 0);
        if constexpr (kSplit == 1) sub(st, 1);
        if (kCausal) {
            if (++head == a.heads) {  // next query tile
                head = 0;
                row0 -= 64;
            }
        }
    };
    for (;;) {
        stage(s1, s0);
        if (it >= n_it) break;
        stage(s0, s1);
        if (it >= n_it) break;
    }
    wait_vm_lgkm0<0>();
    barrier();  // every wave is done with the stages: they take the outputs
    const size_t base = (size_t)b * a.o_heads * S * D + (size_t)ho * a.o_hs + (size_t)key0 * a.o_rs;
    if constexpr (kSplit == 1) {
        FA3_LDS char* stg = smem + w * C::kDB * 1024;
        reg_store<C::kDB, kBf16>(a.dkv_f32, a.dv, base, a.o_rs, av, 1.f, lane, stg);
        reg_store<C::kDB, kBf16>(a.dkv_f32, a.dk, base, a.o_rs, ak, a.scale, lane, stg);
    } else {
        // the two waves of a key block swap halves: rs 0 sums and writes dV, rs 1 dK
        FA3_LDS char* mine = smem + w * C::kDB * 2048;
        FA3_LDS char* other = smem + (kb + kKb * (1 - rs)) * C::kDB * 2048;
        if (rs == 0) reg_put<C::kDB>(mine, ak, lane);
        else reg_put<C::kDB>(mine, av, lane);
        wait_vm_lgkm0<0>();
        barrier();
        if (rs == 0) {
            reg_add<C::kDB>(other, av, lane);
            reg_store<C::kDB, kBf16>(a.dkv_f32, a.dv, base, a.o_rs, av, 1.f, lane, other);
        } else {
            reg_add<C::kDB>(other, ak, lane);
            reg_store<C::kDB, kBf16>(a.dkv_f32, a.dk, base, a.o_rs, ak, a.scale, lane, other);
        }
    }
}

// Query tile qt (128 / kSplit rows) of query head hq (KV head hkv) in batch b.
template <int D, bool kCausal, bool kBf16, int kSplit, bool kDebug, typename A>
__device__ __forceinline__ void reg_dq(const A& a, int b, int hq, int hkv, int qt,
                                       FA3_LDS char* smem) {
    using C = RegCfg<D>;
    constexpr int kQb = kRegWaves / kSplit;  // 32-row blocks of the job
    const int tid = opaque_tid();
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int qi = w & (kQb - 1), rs = w / kQb;
    const int l16 = lane & 15, g4 = lane >> 4;
    const int S = a.seqlen;
    const int q0 = (qt * kQb + qi) * 32;
    const int n_it = kCausal ? ((qt + 1) * kQb + 1) >> 1 : S / 64;

    const _Float16* kp = a.k + kv_elem<D>(a, b, hkv, 0);
    const _Float16* vp = a.v + kv_elem<D>(a, b, hkv, 0);
    const size_t step_e = (size_t)64 * a.kv_rs;
    auto issue = [&](FA3_LDS char* st) {
        const uint32_t off = reg_load_off<D>(opaque_tid() & 63, a.kv_rs);
        reg_load_tile<D>(st, kp, off, w, a.kv_rs);
        reg_load_tile<D>(st + C::kTileBytes, vp, off, w, a.kv_rs);
        kp += step_e;
        vp += step_e;
    };
    FA3_LDS char* s0 = smem;
    FA3_LDS char* s1 = smem + C::kStageBytes;
    issue(s0);
    // resident B operands: Q and dO of rows q0 + 16 n + l16
    f16x8 qf[2][C::kKs], df[2][C::kKs];
    float nl[2];
    f32x4 nd[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
        const size_t e = q_elem<D>(a, b, hq, q0 + 16 * n + l16);
#pragma unroll
        for (int s = 0; s < C::kKs; ++s) {
            qf[n][s] = *(const f16x8*)(a.q + e + 8 * p1_chunk<D>(s, g4));
            df[n][s] = *(const f16x8*)(a.dout + e + 8 * p1_chunk<D>(s, g4));
        }
        const size_t row = ((size_t)b * a.heads_q + hq) * S + q0 + 16 * n + l16;
        nl[n] = a.nlse2[row];
        const float x = a.ndelta[row];
        nd[n] = f32x4{x, x, x, x};
    }
    f32x4 acc[C::kDB][2];
#pragma unroll
    for (int i = 0; i < C::kDB; ++i) acc[i][0] = acc[i][1] = f32x4{};
    const int rsub = 32 * rs;  // as in reg_dkv, of the streamed keys
    const RegReader<D> rd0(lane, rsub);
    const float c = a.scale_log2;
    int k0 = rsub - q0;  // this wave's first key of the stage relative to its first row

    auto sub = [&](const FA3_LDS char* st, int r) {
        RegReader<D> rd = rd0;
        rd.opaque();
        const FA3_LDS char* tk = st;
        const FA3_LDS char* tv = st + C::kTileBytes;
        debug_sync<kDebug>();
        if (!kCausal || k0 + 32 * r <= 0) {
            // [m][n]: keys 16 m + 4 g4 + i, rows 16 n + l16
            f32x4 s[2][2], dp[2][2];
#pragma unroll
            for (int m = 0; m < 2; ++m)
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    s[m][n] = f32x4{};
                    dp[m][n] = nd[n];
                }
            mm_prio<D, 1>();
            reg_scores<D, kBf16>(rd, tk, tv, r, qf, df, s, dp);
            mm_prio<D, 0>();
            float ds[2][8];
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int m = j >> 2, i = j & 3;
                    ds[n][j] = fast_exp2(__builtin_fmaf(s[m][n][i], c, nl[n])) * dp[m][n][i];
                }
            if (kCausal && k0 + 32 * r == 0) {  // the diagonal block
                const int ln = opaque_tid() & 63, l16 = ln & 15, g4 = ln >> 4;  // (keeps this a branch)
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int j = 0; j < 8; ++j)
                        if (16 * (j >> 2) + 4 * g4 + (j & 3) > 16 * n + l16) ds[n][j] = 0.f;
            }
            const f16x8 bs[2] = {pack8<kBf16>(ds[0]), pack8<kBf16>(ds[1])};
            mm_prio<D, 1>();
            reg_grads<D, kBf16, false>(rd, tk, tk, r, bs, bs, acc, acc);
        }
        debug_sync<kDebug>();
    };
    int it = 0;
    auto stage = [&](FA3_LDS char* __restrict__ ld, const FA3_LDS char* __restrict__ st) {
        wait_vm_lgkm0<0>();
        barrier();
        if (++it < n_it) issue(ld);
        sub(st, 0);
        if constexpr (kSplit == 1) sub(st, 1);
        if (kCausal) k0 += 64;
    };
    for (;;) {
        stage(s1, s0);
        if (it >= n_it) break;
        stage(s0, s1);
        if (it >= n_it) break;
    }
    wait_vm_lgkm0<0>();
    barrier();
    const size_t base = q_elem<D>(a, b, hq, q0);
    if constexpr (kSplit == 1) {
        reg_store<C::kDB, kBf16>(a.dq_f32, a.dq, base, a.q_rs, acc, a.scale, lane,
                                 smem + w * C::kDB * 1024);
    } else {
        // each of the two waves of a row block sums and writes half of the columns
        constexpr int kH = C::kDB / 2;
        FA3_LDS char* mine = smem + w * kH * 2048;
        FA3_LDS char* other = smem + (qi + kQb * (1 - rs)) * kH * 2048;
        if (rs == 0) reg_put<kH>(mine, acc + kH, lane);
        else reg_put<kH>(mine, acc, lane);
        wait_vm_lgkm0<0>();
        barrier();
        if (rs == 0) {
            reg_add<kH>(other, acc, lane);
            reg_store<kH, kBf16>(a.dq_f32, a.dq, base, a.q_rs, acc, a.scale, lane, other);
        } else {
            reg_add<kH>(other, acc + kH, lane);
            reg_store<kH, kBf16>(a.dq_f32, a.dq, base + D / 2, a.q_rs, acc + kH, a.scale, lane, other);
        }
    }
}

template <int D, bool kDebug>
__device__ __forceinline__ void reg_poison(FA3_LDS char* smem) {
    if constexpr (kDebug) {
        const f16x8 nan = __builtin_bit_cast(f16x8, u32x4{~0u, ~0u, ~0u, ~0u});
        for (int i = threadIdx.x * 16; i < RegCfg<D>::kBytes; i += kRegThreads * 16)
            lds_write_b128(smem, i, nan);
        debug_sync<true>();
    }
}

template <int D, bool kCausal, bool kBf16, int kSplitKv, int kSplitQ, bool kDebug>
__global__ __launch_bounds__(kRegThreads, D == 64 ? 3 : 2) void bwd_reg_kernel(RegArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem_raw[RegCfg<D>::kBytes];
    FA3_LDS char* smem = (FA3_LDS char*)smem_raw;
    reg_poison<D, kDebug>(smem);
    const int id = blockIdx.x;
    int g, pos;
    job_of(a, id, g, pos);
    const int b = fdiv(a.div_hkv, g), hkv = g - b * a.heads_kv;
    const int QT = a.seqlen / 128, QTq = a.seqlen / (128 / kSplitQ);
    // 64-key tiles in front, 128-key tiles behind them
    const int n64 = kSplitKv == 2 ? 2 * QT : kSplitKv == 0 ? 2 * a.halved : 0;
    const int QTk = kSplitKv == 0 ? QT + a.halved : n64 > 0 ? n64 : QT;
    // the dKV jobs first, by key tile (causal: longest first), one per chunk
    // of query heads; then the dQ jobs, latest query tile first
    int level, slot;  // slot < chunks: dKV, else the dQ job of query head slot - chunks
    const int n_dkv = a.chunks * QTk;
    if (pos < n_dkv) {
        level = fdiv(a.div_chunks, pos);
        slot = pos - level * a.chunks;
    } else {
        const int r = pos - n_dkv;
        level = fdiv(a.div_group, r);
        slot = a.chunks + r - level * a.group;
    }
    const int h0 = hkv * a.group + slot * a.heads, ho = hkv * a.chunks + slot;
    if (slot < a.chunks) {
        if constexpr (kSplitKv == 0) {
            // (the arguments re-read from the argument segment: held across
            // the roles' code, they spill scalar registers)
            typedef __attribute__((address_space(4))) const RegArgs KReg;
            KReg* ap = (KReg*)__builtin_amdgcn_kernarg_segment_ptr();
            __asm__ volatile("" : "+s"(ap));
            if (level < n64) reg_dkv<D, kCausal, kBf16, 2, kDebug>(*ap, b, hkv, level, h0, ho, smem);
            else
                reg_dkv<D, kCausal, kBf16, 1, kDebug>(*ap, b, hkv, level - n64 / 2, h0, ho, smem);
        } else {
            reg_dkv<D, kCausal, kBf16, kSplitKv, kDebug>(a, b, hkv, level, h0, ho, smem);
        }
    } else
        reg_dq<D, kCausal, kBf16, kSplitQ, kDebug>(a, b, hkv * a.group + slot - a.chunks, hkv,
                                                   QTq - 1 - level, smem);
}

template <bool kDebug>
void launch_reg_kernel(const RegArgs& a, RegPlan plan, int head_dim, bool causal, bool bf16,
                       hipStream_t stream) {
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(a.n_groups * a.jobs_per_group), dim3(kRegThreads), 0,
                           stream, a);
    };
    auto pick = [&](auto d, auto cz, auto bf) {
        constexpr int kD = decltype(d)::value;
        constexpr bool kC = decltype(cz)::value, kB = decltype(bf)::value;
        if constexpr (kD == 64) {
            if (plan.split_q == 2) return go(bwd_reg_kernel<kD, kC, kB, 2, 2, kDebug>);
        }
        if constexpr (kC) go(bwd_reg_kernel<kD, kC, kB, 0, 1, kDebug>);
        else if (plan.split_kv == 1) go(bwd_reg_kernel<kD, kC, kB, 1, 1, kDebug>);
        else go(bwd_reg_kernel<kD, kC, kB, 2, 1, kDebug>);
    };
    auto types = [&](auto d) {
        using T = std::true_type;
        using F = std::false_type;
        if (causal) bf16 ? pick(d, T{}, T{}) : pick(d, T{}, F{});
        else bf16 ? pick(d, F{}, T{}) : pick(d, F{}, F{});
    };
    if (head_dim == 128) types(std::integral_constant<int, 128>{});
    else types(std::integral_constant<int, 64>{});
}

}  // namespace

// The race-check instantiations (fa3_bwd_main_debug.hip).
void launch_reg_race_check(const RegArgs& a, RegPlan plan, int head_dim, bool causal, bool bf16,
                           hipStream_t stream);

}  // namespace fa3
