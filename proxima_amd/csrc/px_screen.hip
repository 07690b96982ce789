// px_screen.hip -- screening of FlatIndex searches on the fp16 matrix cores, gfx950.
//
// Replaces the fp32 scans of crates/core/src/flat.rs:106-148's per-query full scan where rows
// or queries are not exact in fp16. Every result still comes from the fp32 rows in the
// reference's arithmetic (distance.rs:3-39); the screen only rules rows out, and only those
// it can prove to be too far:
//
//   * The index keeps a copy of its rows rounded to fp16 (scaled by one power of two), and the
//     largest rounding residual ||x - x~|| and norm ||x|| over its rows. A batch's queries are
//     rounded alike, with ||q - q~|| of each.
//   * The scan's key of a row, ||x||^2 - 2 q~.x~ (L2) or -q~.x~ (IP), then differs from the
//     reference's key (less ||q||^2, which is the same for all rows) by at most err(q):
//     Cauchy-Schwarz on the residuals, plus worst-case bounds of the fp32 sums' rounding in
//     the scan, the norms and the reference itself (screen_queries_kernel).
//   * If A is the k-th smallest scan key, k rows have reference keys at or below A + err, so a
//     row whose scan key is past A + 2 err is not among the best k. The select
//     (flat_collect_select_kernel) recomputes the key of every row up to there and takes the
//     best k of them; a query whose collected rows do not reach that far goes round again.
//
// So the results are those of a scan of every row in the reference's arithmetic; how tight
// the fp16 keys are only decides how many rows are recomputed (1M x 128 N(0,1), k = 10: err
// is 0.1 on keys whose spread is 32, and 3% more rows than k are).
//
// The fp32 scans are bound by the fp32 MFMA rate (157 TFLOP/s); the fp16 matrix cores do
// sixteen times that. A scan, ms (kernel trace; before: the fp32 lists or collect scan):
//   1M x 128 uniform, 2,000 queries, k = 10           0.47 (1,090 TFLOP/s)   before 4.43
//   100k x 384, 1,000 queries, k = 10                 0.098 (780 TFLOP/s)    before 0.75
//   200k x 768, 500 queries, k = 20                   0.157 (980 TFLOP/s)    before 1.41
//   200k of 2M x 384 filtered, 4,096 queries, k = 100 0.68 (930 TFLOP/s)     before 5.38
//   500k x 100 (128 padded), 4,999 queries, k = 100   0.67                   before 4.95
#include "px_device.h"
#include "px_host.h"
#include "px_kernels.h"
#include "px_scan_common.h"

#include <float.h>
#include <limits.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

namespace px {

namespace {

constexpr int kWaves = 8;
constexpr int kSlots = 64 * kWaves;            // query slots a workgroup (QB = 2)
static_assert(kSlots == kScreenBlockSlots, "screen_batch's slots");
constexpr int kTile = 32;                      // rows a tile: one MFMA block
constexpr int kTiles = kScreenRows / kTile;    // tiles a row group (4)
constexpr int kRowBytes = kChunk * 2;          // a staged chunk of a row: 128 fp16
// LDS row pitch: 16 bytes more, so that sixteen consecutive rows' same 16-byte piece fall in
// sixteen different bank groups (conflict-free b128 reads of the A operands)
constexpr int kPitch = kRowBytes + 16;
constexpr int kBufs = 3;                       // LDS stage buffers
constexpr int kNormSlots = 4;                  // row groups whose norms LDS holds
constexpr int kScreenWideSlots = 256;          // most queries that a workgroup each selects

// Largest of three / two scan sums as one v_max3_f32 / v_max_f32: fmaxf of MFMA results costs
// two canonicalising instructions more (IEEE maxNum); the sums are finite here.
__device__ __forceinline__ float max3_of(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float max_of(float a, float b) {
    float r;
    asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// The scan. One workgroup = 8 waves = 512 query slots x one split of the rows; a wave holds
// 64 queries as two 32-query B operands of v_mfma_f32_32x32x16_f16, one 128-dim chunk of them
// at a time (64 VGPRs; with several chunks, MULTI, each fragment's registers take the next
// chunk's as soon as its MFMAs have read them), and the sums of a group of 128 rows x 64
// queries (128 VGPRs), so that each 16-byte A operand read from LDS feeds two MFMAs and a
// chunk of queries read from L2 feeds 128 rows. A stage is one chunk of one row group.
//
// Sums start from -||x||^2 / 2 (L2; zero for IP), so that they end as D = key / f with
// f = -2 (L2) or -1 (IP), times the power of two both operands are scaled by; a row passes
// where D is at or above its query's threshold / f.
//
// Pipeline: three LDS stage buffers, the loads of stage s + 2 held in registers during stage
// s, no barrier per stage (stage_wait / stage_publish, px_scan_common.h). The two waves of a
// SIMD drift apart, so that one wave's tests run beside the other's MFMAs.
//
// MIN: no thresholds; the smallest key of every group of group_tiles tiles of a lane (16 rows
// of each) goes to minima[query][2 x group + h]. Their r-th smallest bounds the r-th
// smallest key of the sample from above (r different rows), at a 16th to a 64th of the
// writes, and of the ladder's work, that every sampled key would take.
//
// QB = 1 (batches of at most 256 queries, one query tile): 32 queries a wave, 256 slots. Such a
// scan is bound by HBM, and with one stage's loads in flight by their latency: the registers
// of the second query block hold another two stages' (1M x 128, one query: 60 us = 4.2 TB/s,
// with them 42 us = 6.1 TB/s; 5,000 x 128, 16 queries: 13 and 8.8 us).
template <bool L2, bool FILT, bool MIN, bool MULTI, int QB>
__global__ __launch_bounds__(512) void flat_screen_kernel(ScreenArgs a) {
    constexpr int SL = 32 * QB * kWaves;         // query slots a workgroup
    constexpr int PD = QB == 1 ? 2 : 1;          // stages whose loads are held in registers
    constexpr int kF4PerRow = kRowBytes / 16;    // 16-byte pieces a staged row (16)
    constexpr int kRowStep = 512 / kF4PerRow;    // rows between a thread's loads (32)
    constexpr int NG = kChunk / 16;              // dim groups a chunk (8)
    constexpr float kF = L2 ? -2.0f : -1.0f;     // key = kF * D
    static_assert(kScreenRows / kRowStep == 4 && NG == 8, "four staged pieces a thread");
    __shared__ __attribute__((aligned(16))) char tile[kBufs][kScreenRows * kPitch];
    __shared__ __attribute__((aligned(16))) float tnorm[kNormSlots][kScreenRows];
    __shared__ int committed[8];  // per wave: the last stage it has committed
    __shared__ int wants[8];      // per wave: whether a row can pass for one of its queries
    // rows each lane has appended for its two queries: in LDS, as registers they spilled
    __shared__ int counts[MIN ? 1 : QB][MIN ? 1 : 512];

    const int tid = threadIdx.x;
    const int wave = tid >> 6, lane = tid & 63, j = lane & 31, h = lane >> 5;
    const int qtiles = gridDim.x / a.splits;
    // the last (partial) query tile, whose workgroups run fastest, starts first
    const int qt = qtiles - 1 - (int)(blockIdx.x / a.splits), split = blockIdx.x % a.splits;
    const int slot0 = qt * SL + wave * 32 * QB + j;  // block 1: slot0 + 32
    const int row0 = (int)((int64_t)split * a.rows_per_split);
    const int row1 = (int)min(a.n_eff, (int64_t)row0 + a.rows_per_split);
    PX_DCHECK(a.dbg, kDbgScreen, row0 < row1 && (int64_t)qtiles * a.splits == (int64_t)gridDim.x);
    const float kInf = __int_as_float(0x7f800000);
    const int ngroups = (row1 - row0 + kScreenRows - 1) / kScreenRows;  // >= 1
    const int C = MULTI ? a.chunks : 1;
    const int nstages = ngroups * C;
    const int cc = tid % kF4PerRow;   // this thread's 16-byte piece of a staged row
    const int rr0 = tid / kF4PerRow;  // its first row of a stage
    // D carries the scale (a power of two); in scalar registers
    auto uniform = [](float v) __attribute__((always_inline)) {
        return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
    };
    const float scale = uniform(a.scale[0]);
    const float unscale = uniform(a.scale[1]) * kF;  // key = unscale * D
    auto opaque = [](int v) __attribute__((always_inline)) {
        asm volatile("" : "+v"(v));
        return v;
    };

    // ---- per-query state, [query block]
    // Padding slots: a NaN, which no D passes. (Not +inf: after a wait that gave up, D may come
    // of norms never written, +inf among them, and a slot past nq has no region to append to.)
    const float kNothing = __int_as_float(0x7fc00000);
    float nct[QB];  // the threshold as a D value: a row passes at or above it
    auto query_of = [&](int qb) __attribute__((always_inline)) {
        const int slot = opaque(slot0 + 32 * qb);
        return a.qlist ? a.qlist[slot < a.nq ? slot : 0] : (slot < a.nq ? slot : 0);
    };
    if constexpr (!MIN) {
        bool want = false;
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
            nct[qb] = kNothing;
            if (slot0 + 32 * qb < a.nq)
                nct[qb] = from_total_key(a.thr_key[query_of(qb)]) * (1.0f / kF) * scale;
            want |= nct[qb] < kInf;
        }
        if (__ballot(want) && lane == 0) wants[wave] = 1;
        else if (lane == 0) wants[wave] = 0;
    }

    // ---- staging: every load unconditional, positions past the split's end clamped to its
    // last row (their sums are not used). Positions fit 32 bits, unsigned: at most 2^31 + 511.
    // Unfiltered row ids are formed where they are used; a filter's are loaded a stage ahead.
    const unsigned last = (unsigned)row1 - 1, stride = (unsigned)a.stride;
    unsigned rid[4], pid = 0;
    auto row_of = [&](unsigned pos) __attribute__((always_inline)) {
        const unsigned p = min(pos, last) * stride;
        const unsigned v = FILT ? (unsigned)a.rowidx[p] : p;
        PX_DCHECK(a.dbg, kDbgScreen, v < (unsigned)a.rows);
        return v;
    };
    auto group_ids = [&](int rg) __attribute__((always_inline)) {
        const unsigned t0 = (unsigned)row0 + (unsigned)rg * kScreenRows;
#pragma unroll
        for (int u = 0; u < 4; ++u) rid[u] = row_of(t0 + rr0 + u * kRowStep);
        if (L2) pid = row_of(t0 + (tid & (kScreenRows - 1)));
    };
    int fc = 0, frg = 0;  // chunk and row group the next fetch loads
    // stage s's loads are held in set s % PD (every index is a constant where it is used)
    float4 pf[PD][4];
    float pn[PD] = {};
    const unsigned dsb = (unsigned)a.ds * 2;  // bytes of a row
    using Set0 = std::integral_constant<int, 0>;
    using Set1 = std::integral_constant<int, PD - 1>;
    auto fetch = [&](auto set_tag) __attribute__((always_inline)) {
        constexpr int S = decltype(set_tag)::value;
        if (!FILT) group_ids(frg);
        const char* base = reinterpret_cast<const char*>(a.xs) + (MULTI ? fc * kRowBytes : 0);
        auto load = [&](unsigned r) __attribute__((always_inline)) {
            return *reinterpret_cast<const float4*>(base + ((uint64_t)r * dsb + cc * 16));
        };
#pragma unroll
        for (int u = 0; u < 4; ++u) pf[S][u] = load(rid[u]);
        if (L2 && (!MULTI || fc == 0)) pn[S] = a.norms[pid];
    };
    auto advance = [&]() __attribute__((always_inline)) {
        if (!MULTI || ++fc == C) {
            fc = 0;
            ++frg;
            if (FILT) group_ids(frg);
        }
    };
    auto commit = [&](auto set_tag, int buf, int c, int rg) __attribute__((always_inline)) {
        constexpr int S = decltype(set_tag)::value;
        char* tb = tile[buf] + rr0 * kPitch + cc * 16;
#pragma unroll
        for (int u = 0; u < 4; ++u)
            *reinterpret_cast<float4*>(tb + u * kRowStep * kPitch) = pf[S][u];
        if (L2 && (!MULTI || c == 0) && tid < kScreenRows)
            tnorm[rg & (kNormSlots - 1)][tid] = -0.5f * pn[S] * scale;
    };
    // One stage's loads and commit, PD == 2. A wait for a load is one for all before it, so a
    // filter's ids of the stage after are loaded before this one's rows, and rows after what
    // the stage's MFMAs loaded (issue at a stage's end): nothing waits for the newest rows.
    auto issue = [&](auto set_tag) __attribute__((always_inline)) {
        const bool next = !MULTI || fc == C - 1;
        if constexpr (FILT) {
            unsigned nid[4], np = 0;
            if (next) {
                const unsigned t0 = (unsigned)row0 + (unsigned)(frg + 1) * kScreenRows;
#pragma unroll
                for (int u = 0; u < 4; ++u) nid[u] = row_of(t0 + rr0 + u * kRowStep);
                if (L2) np = row_of(t0 + (tid & (kScreenRows - 1)));
            }
            fetch(set_tag);
            if (next) {
#pragma unroll
                for (int u = 0; u < 4; ++u) rid[u] = nid[u];
                pid = np;
            }
        } else {
            fetch(set_tag);
        }
        fc = next ? 0 : fc + 1;
        frg += next;
    };
    int sc = 0, sg = 0;  // chunk and row group the next commit writes (PD == 2)
    auto settle = [&](auto set_tag, int buf) __attribute__((always_inline)) {
        commit(set_tag, buf, sc, sg);
        const bool next = !MULTI || sc == C - 1;
        sc = next ? 0 : sc + 1;
        sg += next;
    };
    group_ids(0);
    if constexpr (PD == 1) {
        fetch(Set0{});
        commit(Set0{}, 0, 0, 0);
        advance();
        fetch(Set0{});
        commit(Set0{}, 1, fc, frg);
        advance();
    } else {
        issue(Set0{});
        issue(Set1{});
        settle(Set0{}, 0);
        issue(Set0{});
        settle(Set1{}, 1);
        issue(Set1{});
    }
    using P0 = std::integral_constant<int, 0>;
    using P1 = std::integral_constant<int, 1>;
    if (tid < 8) committed[tid] = 1;
    __syncthreads();
    // no query of the workgroup that a row can pass for (the ladder gave them all up): done
    if constexpr (!MIN) {
        int any = 0;
#pragma unroll
        for (int w = 0; w < 8; ++w) any |= wants[w];
        if (!any) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
                if (slot0 + 32 * qb < a.nq)
                    a.cand_count[((int64_t)(slot0 + 32 * qb) * a.splits + split) * 2 + h] = 0;
            return;
        }
    }

    // Stage sync: at the end of stage s a wave waits until every wave has committed stage
    // s + 1 before it reads that stage and writes stage s + 2, whose buffer held stage s - 1
    // (a wave commits s + 1 only after all its reads of s - 1; a norm slot is reused four row
    // groups, at least four stages, later). A wait that gives up is reported (a.spin_fail).
    const unsigned caddr = (unsigned)(uintptr_t)(committed + (lane & 7));
    auto wait_committed = [&](int ct) __attribute__((always_inline)) {
        if (stage_wait(caddr, ct, a.spin_limit) >= a.spin_limit && lane == 0)
            atomicOr(a.spin_fail, 1);
    };

    // a wave whose 64 query slots are all padding only helps stage the rows
    if (qt * SL + wave * 32 * QB >= a.nq) {
        int wb = 2;
        auto stage = [&](auto p_tag, int s) __attribute__((always_inline)) {
            const int pc = fc, prg = frg;
            if constexpr (PD == 1) {
                fetch(Set0{});
                advance();
            }
            wait_committed(s + 1);
            if constexpr (PD == 1) commit(Set0{}, wb, pc, prg);
            else settle(p_tag, wb);
            stage_publish(committed, wave, lane, s + 2);
            if constexpr (PD == 2) issue(p_tag);
            wb = wb == kBufs - 1 ? 0 : wb + 1;
        };
        for (int i = 0; i < nstages >> 1; ++i) {
            stage(P0{}, 2 * i);
            stage(P1{}, 2 * i + 1);
        }
        if (nstages & 1) stage(P0{}, nstages - 1);
        return;
    }

    if constexpr (!MIN) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) counts[qb][tid] = 0;
    }
    float vmax[QB];
#pragma unroll
    for (int qb = 0; qb < QB; ++qb) vmax[qb] = -kInf;
    // The queries lie in fragment order (ScreenArgs::qs), so that a wave's load is 1 KB in one
    // piece: as rows, its 64 lanes touched 32 cache lines for 32 bytes of each, and those
    // loads, not the matrix units, set the pace of several-chunk scans. Buffer loads: a scalar
    // descriptor and offset and one lane offset take no 64-bit address registers.
    const auto qrsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<unsigned short*>(a.qs), 0,
        (int)((unsigned)screen_query_slots(a.nq) * dsb), 0x00027000);
    const int qblock = __builtin_amdgcn_readfirstlane(qt * (SL / 32) + wave * QB);
    const int qb_bytes = (int)(a.ds * 64);  // a block of 32 queries
    const unsigned qlane = (unsigned)lane * 16;
    auto query_frag = [&](int chunk, int qb, int g) __attribute__((always_inline)) {
        return __builtin_bit_cast(
            f16x8, __builtin_amdgcn_raw_buffer_load_b128(
                       qrsrc, qlane, (qblock + qb) * qb_bytes + chunk * (NG * 1024) + g * 1024, 0));
    };
    f16x8 bq[QB][NG];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) bq[qb][g] = query_frag(0, qb, g);
    // (in registers here: a wait for them inside the loop would be one for its row loads too)
    if constexpr (PD == 2) {
#pragma unroll
        for (int g = 0; g < NG; ++g) asm volatile("" : "+v"(bq[0][g]));
    }
    // one row at or above its query's threshold: appended to the region of (slot, split, h);
    // past the region's capacity the count still grows (the select sees the overflow)
    auto append = [&](int qb, float d, int pos) __attribute__((always_inline)) {
        if (d >= nct[qb] && pos < row1) {
            PX_DCHECK(a.dbg, kDbgScreen, slot0 + 32 * qb < a.nq && pos >= row0);
            const int n = counts[qb][tid];
            counts[qb][tid] = n + 1;
            if (n < a.cap) {
                const int64_t at =
                    (((int64_t)opaque(slot0 + 32 * qb) * a.splits + split) * 2 + h) * a.cap + n;
                a.cand_keys[at] = unscale * d;
                a.cand_pos[at] = pos;
            }
        }
    };

    f32x16 acc[kTiles][QB];
    int rb = 0, wb = 2, s = 0;  // LDS buffers read and written next, stage
    int mt = 0;                 // MIN: tiles of the current minimum's group
    auto begin = [&](int rg) __attribute__((always_inline)) {
        // starts of the row group's sums, in the MFMA result's layout (register x: row
        // mfma_row(x, h), four contiguous rows a 4-register group); the lane offset is opaque
        // so that each block's copy is its own LDS read rather than sixteen register copies
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
                if constexpr (L2) {
                    const float* tn =
                        tnorm[rg & (kNormSlots - 1)] + t * kTile + opaque(4 * h);
#pragma unroll
                    for (int m = 0; m < 4; ++m) {
                        const float4 v = *reinterpret_cast<const float4*>(tn + 8 * m);
                        acc[t][qb][4 * m + 0] = v.x;
                        acc[t][qb][4 * m + 1] = v.y;
                        acc[t][qb][4 * m + 2] = v.z;
                        acc[t][qb][4 * m + 3] = v.w;
                    }
                } else {
#pragma unroll
                    for (int x = 0; x < 16; ++x) acc[t][qb][x] = 0.f;
                }
            }
        }
    };
    auto stage = [&](auto p_tag, int c) __attribute__((always_inline)) {
        const int pc = fc, prg = frg;
        if constexpr (PD == 1) {
            fetch(Set0{});
            advance();
        }
        // the queries' next chunk (after the row group's last: chunk 0)
        const int qn = MULTI && c + 1 != C ? c + 1 : 0;
        const char* ta = tile[rb] + j * kPitch + h * 16;
        // A operands three reads ahead: read i is dim group i / 4 of tile i % 4
        auto a_of = [&](int i) __attribute__((always_inline)) {
            return *reinterpret_cast<const f16x8*>(ta + (i & 3) * kTile * kPitch +
                                                   (i >> 2) * 32);
        };
        f16x8 x[4] = {a_of(0), a_of(1), a_of(2), f16x8{}};
#pragma unroll
        for (int i = 0; i < NG * kTiles; ++i) {
            const int g = i >> 2, t = i & 3;
            if (i + 3 < NG * kTiles) x[(i + 3) & 3] = a_of(i + 3);
#pragma unroll
            for (int qb = 0; qb < QB; ++qb)
                acc[t][qb] = mfma16(x[i & 3], bq[qb][g], acc[t][qb]);
            if (MULTI && t == 3) {
#pragma unroll
                for (int qb = 0; qb < QB; ++qb) bq[qb][g] = query_frag(qn, qb, g);
            }
            // as written: the scheduler otherwise sinks the A reads to their MFMAs and
            // the query loads to the stage's end, and every one is waited for
            __builtin_amdgcn_sched_barrier(0);
        }
        // the commit stays after the MFMAs (hoisted, it would wait for the loads there)
        __builtin_amdgcn_sched_barrier(0);
        wait_committed(s + 1);
        pair_priority(__hip_atomic_load(committed + (wave ^ 4), __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_WORKGROUP),
                      s + 1);
        if constexpr (PD == 1) commit(Set0{}, wb, pc, prg);
        else settle(p_tag, wb);
        stage_publish(committed, wave, lane, s + 2);
        if constexpr (PD == 2) issue(p_tag);
        rb = rb == kBufs - 1 ? 0 : rb + 1;
        wb = wb == kBufs - 1 ? 0 : wb + 1;
        ++s;
    };
    auto finish = [&](int rg) __attribute__((always_inline)) {
        const int pt = row0 + rg * kScreenRows;
#pragma unroll
        for (int t = 0; t < kTiles; ++t) {
#pragma unroll
            for (int qb = 0; qb < QB; ++qb) {
                const f32x16& v = acc[t][qb];
                float m[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    m[u] = max_of(max3_of(v[4 * u], v[4 * u + 1], v[4 * u + 2]), v[4 * u + 3]);
                const float mm = max_of(max3_of(m[0], m[1], m[2]), m[3]);
                if constexpr (MIN) {
                    vmax[qb] = max_of(vmax[qb], mm);
                } else if (__builtin_expect(__ballot(mm >= nct[qb]) != 0, 0)) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (__ballot(m[u] >= nct[qb])) {
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                append(qb, v[4 * u + e], pt + t * kTile + mfma_row(4 * u + e, h));
                        }
                    }
                }
            }
            if constexpr (MIN) {
                // (splits and samples are whole numbers of groups: none is partial)
                if (++mt == a.group_tiles) {
                    const int gi = ((pt >> 5) + t) / a.group_tiles;
                    PX_DCHECK(a.dbg, kDbgScreen, 2 * gi + 1 < a.min_ld);
#pragma unroll
                    for (int qb = 0; qb < QB; ++qb) {
                        if (slot0 + 32 * qb < a.nq)
                            a.minima[(int64_t)query_of(qb) * a.min_ld + 2 * gi + h] =
                                unscale * vmax[qb];
                        vmax[qb] = -kInf;
                    }
                    mt = 0;
                }
            }
        }
    };
    if constexpr (PD == 1) {
        for (int rg = 0; rg < ngroups; ++rg) {
            begin(rg);
            for (int c = 0; c < C; ++c) stage(P0{}, c);
            finish(rg);
        }
    } else {  // by stages: their parity names the register set
        int rg = 0, c = 0;
        auto step = [&](auto p_tag) __attribute__((always_inline)) {
            if (!MULTI || c == 0) begin(rg);
            stage(p_tag, c);
            if (!MULTI || ++c == C) {
                finish(rg);
                c = 0;
                ++rg;
            }
        };
        // (no exit between the two: the compiler would take one set's loads for the newest
        // in both, and wait for all)
        for (int i = 0; i < nstages >> 1; ++i) {
            step(P0{});
            step(P1{});
        }
        if (nstages & 1) step(P0{});
    }
    if constexpr (!MIN) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb)
            if (slot0 + 32 * qb < a.nq)
                a.cand_count[((int64_t)(slot0 + 32 * qb) * a.splits + split) * 2 + h] =
                    counts[qb][tid];
    }
}

template <bool MIN, int QB>
void launch_screen_t(const ScreenArgs& a, hipStream_t s) {
    constexpr int SL = 32 * QB * kWaves;
    const int64_t qtiles = (a.nq + SL - 1) / SL;
    const dim3 grid((unsigned)(qtiles * a.splits)), block(512);
    const bool filt = a.rowidx != nullptr, multi = a.chunks > 1;
#define PX_SCREEN(L2, FILT, MULTI) \
    hipLaunchKernelGGL((flat_screen_kernel<L2, FILT, MIN, MULTI, QB>), grid, block, 0, s, a)
    if (a.metric == 0) {
        if (filt) {
            if (multi) PX_SCREEN(true, true, true);
            else PX_SCREEN(true, true, false);
        } else if (multi) PX_SCREEN(true, false, true);
        else PX_SCREEN(true, false, false);
    } else {
        if (filt) {
            if (multi) PX_SCREEN(false, true, true);
            else PX_SCREEN(false, true, false);
        } else if (multi) PX_SCREEN(false, false, true);
        else PX_SCREEN(false, false, false);
    }
#undef PX_SCREEN
}
template <bool MIN>
void launch_screen_q(const ScreenArgs& a, hipStream_t s) {
    if (a.nq <= 32 * kWaves) launch_screen_t<MIN, 1>(a, s);
    else launch_screen_t<MIN, 2>(a, s);
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) v = fmaxf(v, __shfl_xor(v, m));
    return v;
}

// v 2^e in fp16, magnitudes below its smallest normal as zero (no MFMA input depends on
// subnormal handling)
__device__ __forceinline__ _Float16 to_screen(float v, float s) {
    const float w = v * s;
    return fabsf(w) < 0x1p-14f ? (_Float16)0.f : (_Float16)w;
}

// |v|, +inf for a NaN (which fmaxf would drop)
__device__ __forceinline__ float magnitude(float v) {
    const float m = fabsf(v);
    return m <= FLT_MAX ? m : __int_as_float(0x7f800000);
}

// largest |x| of each workgroup's share of count floats (count % 4 == 0, x 16-byte aligned)
__global__ __launch_bounds__(256) void abs_max_kernel(const float4* x, int64_t count4, float* out,
                                                      int* words) {
    if (words && blockIdx.x == 0 && threadIdx.x < 2) words[threadIdx.x] = 0;
    __shared__ float wm[4];
    float m = 0.f;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count4;
         i += (int64_t)gridDim.x * 256) {
        const float4 v = x[i];
        m = fmaxf(m, fmaxf(fmaxf(magnitude(v.x), magnitude(v.y)),
                           fmaxf(magnitude(v.z), magnitude(v.w))));
    }
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) wm[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = fmaxf(fmaxf(wm[0], wm[1]), fmaxf(wm[2], wm[3]));
}

// One wave a row: its fp16 copy (zero pad columns), and the largest squared norm and squared
// residual of all rows (max2: float bits, which order as ints where nothing is negative). The
// residual is taken of the scaled row, whose values lie where squares are fp32 numbers.
__global__ __launch_bounds__(256) void screen_rows_kernel(const float* x, int64_t rows, int dp,
                                                          int ds, float s, unsigned short* out,
                                                          int* max2) {
    __shared__ float wn[4], wr[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float n_max = 0.f, r_max = 0.f;
    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < rows; r += (int64_t)gridDim.x * 4) {
        const float* xr = x + r * dp;
        unsigned short* o = out + r * ds;
        float n2 = 0.f, r2 = 0.f;
        for (int c = lane * 2; c < ds; c += 128) {
            const float2 v = c < dp ? *reinterpret_cast<const float2*>(xr + c) : float2{0.f, 0.f};
            const _Float16 h0 = to_screen(v.x, s), h1 = to_screen(v.y, s);
            const float d0 = v.x * s - (float)h0, d1 = v.y * s - (float)h1;
            n2 += v.x * v.x + v.y * v.y;
            r2 += d0 * d0 + d1 * d1;
            *reinterpret_cast<ushort2*>(o + c) = make_ushort2(__builtin_bit_cast(unsigned short, h0),
                                                              __builtin_bit_cast(unsigned short, h1));
        }
        n_max = fmaxf(n_max, wave_sum(n2));
        r_max = fmaxf(r_max, wave_sum(r2));
    }
    if (lane == 0) {
        wn[wave] = n_max;
        wr[wave] = r_max;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(max2, __float_as_int(fmaxf(fmaxf(wn[0], wn[1]), fmaxf(wn[2], wn[3]))));
        atomicMax(max2 + 1, __float_as_int(fmaxf(fmaxf(wr[0], wr[1]), fmaxf(wr[2], wr[3]))));
    }
}

// screen_rows_kernel of the rows that PQ codes stand for (dim / m dims of a subspace's
// centroid each), and their squared norms.
__global__ __launch_bounds__(256) void screen_codes_kernel(const uint8_t* codes, int64_t rows,
                                                           int dim, int ds, int m, int ks,
                                                           const float* books, float s,
                                                           unsigned short* out, float* norms,
                                                           int* max2) {
    __shared__ float wn[4], wr[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, dsub = dim / m;
    float n_max = 0.f, r_max = 0.f;
    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < rows; r += (int64_t)gridDim.x * 4) {
        const uint8_t* cr = codes + r * m;
        float n2 = 0.f, r2 = 0.f;
        for (int c = lane; c < ds; c += 64) {
            float v = 0.f;
            if (c < dim) {
                const int sub = c / dsub;
                v = books[((int64_t)sub * ks + cr[sub]) * dsub + (c - sub * dsub)];
            }
            const _Float16 hv = to_screen(v, s);
            const float d = v * s - (float)hv;
            n2 += v * v;
            r2 += d * d;
            out[r * ds + c] = __builtin_bit_cast(unsigned short, hv);
        }
        n2 = wave_sum(n2);
        if (lane == 0) norms[r] = n2;
        n_max = fmaxf(n_max, n2);
        r_max = fmaxf(r_max, wave_sum(r2));
    }
    if (lane == 0) {
        wn[wave] = n_max;
        wr[wave] = r_max;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(max2, __float_as_int(fmaxf(fmaxf(wn[0], wn[1]), fmaxf(wn[2], wn[3]))));
        atomicMax(max2 + 1, __float_as_int(fmaxf(fmaxf(wr[0], wr[1]), fmaxf(wr[2], wr[3]))));
    }
}

// 64 columns a workgroup, four groups of rows: a few microseconds once an add.
__global__ __launch_bounds__(256) void screen_spread_kernel(const unsigned short* xs, int64_t rows,
                                                            int ds, float* parts) {
    __shared__ float sums[4][64], squares[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t n = min(rows, (int64_t)256);
    const unsigned short* x = xs + (int64_t)blockIdx.x * 64 + lane;
    float m = 0.f, v2 = 0.f;
#pragma unroll 8
    for (int64_t i = wave; i < n; i += 4) {
        // (i rows / n, not i times a whole step: rows of one kind may lie at every third)
        const float v = (float)__builtin_bit_cast(_Float16, x[i * rows / n * ds]);
        m += v;
        v2 += v * v;
    }
    sums[wave][lane] = m;
    squares[wave][lane] = v2;
    __syncthreads();
    if (wave != 0) return;
    const float inv = 1.0f / (float)n;
    m = inv * (sums[0][lane] + sums[1][lane] + sums[2][lane] + sums[3][lane]);
    v2 = inv * (squares[0][lane] + squares[1][lane] + squares[2][lane] + squares[3][lane]);
    m = wave_sum(m * m);
    v2 = wave_sum(v2);
    if (lane == 0) {
        parts[2 * blockIdx.x] = m;
        parts[2 * blockIdx.x + 1] = v2;
    }
}

// One wave a query: its fp16 copy, scaled by 2^eq with the batch's largest magnitude (max_abs,
// or the maximum of parts) in [2^9, 2^10), and err(q), the bound on |scan key - reference key| over
// all rows of the index (X, dX: its largest norm and residual; D: dims summed). With u =
// 2^-24, every sum of D products being off by at most 2 D u times the sum of the magnitudes
// (2 u an addition: the matrix cores' rounding is not assumed to be to nearest), and the
// start of a sum counted with its terms:
//   L2: 2 (||q|| dX + dq (X + dX))  +  2 * 2 D u (X^2 / 2 + ||q|| X)  (the scan)
//       + D u X^2  (the norms)  +  R u (||q|| + X)^2  (the reference's own sums, R terms)
//   IP: ||q|| dX + dq (X + dX)  +  2 D u ||q|| X  +  R u ||q|| X
// with 1% on top for the rounding of these figures and of key + err. ||q|| and dq are summed of
// the scaled query, whose largest magnitude is about 2^9: what fp32 loses of its squares (values
// below 2^-75) is far within the terms in u (of queries near 2^-60 as they are, the squared
// residuals were all zero, and the nearest row could be ruled out). Where the scales of rows
// and queries are too far apart for one product to carry both, or a figure overflows, err is
// +inf, which no query finishes with. Workgroup 0 writes scale: 2^(ex + eq) and its inverse.
struct QueryScale {
    float s, inv_s;
    bool ok;
    int eq;
};
__device__ __forceinline__ QueryScale query_scale(float m, int ex) {
    int eq = m > 0.f && m <= FLT_MAX ? 9 - ilogbf(m) : ex;
    const bool ok = m == 0.f || (m >= 0x1p-60f && m <= 0x1p60f && abs(eq - ex) <= 40);
    if (!ok) eq = ex;
    return {ldexpf(1.f, eq), ldexpf(1.f, -eq), ok, eq};
}
__global__ __launch_bounds__(256) void screen_queries_kernel(ScreenQueryArgs a) {
    const int lane = threadIdx.x & 63;
    float m = a.max_abs;
    if (a.parts) {
        m = 0.f;
        for (int i = lane; i < a.parts_n; i += 64) m = fmaxf(m, a.parts[i]);
        m = wave_max(m);
    }
    const QueryScale qs = query_scale(m, a.ex);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        a.scale[0] = ldexpf(1.f, a.ex + qs.eq);
        a.scale[1] = ldexpf(1.f, -(a.ex + qs.eq));
        if (a.words) {
            if (!a.parts) a.words[0] = a.words[1] = 0;
            else if (m > FLT_MAX) a.words[1] = 1;
        }
    }
    // slot sl holds query q; padding slots are zeros
    const int64_t sl = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (sl >= screen_query_slots(a.nq)) return;  // whole waves; no barrier below
    const bool live = sl < a.nq;
    const int64_t q = !live ? 0 : a.qlist ? a.qlist[sl] : sl;
    const float* x = a.queries + q * a.pitch;
    unsigned short* o = a.qs + (sl >> 5) * 32 * a.ds + (sl & 31) * 8;
    float n2 = 0.f, r2 = 0.f;
    for (int c = lane * 2; c < a.ds; c += 128) {
        const float v0 = live && c < a.dim ? x[c] : 0.f;
        const float v1 = live && c + 1 < a.dim ? x[c + 1] : 0.f;
        if (a.padded && live && c < a.dp)
            *reinterpret_cast<float2*>(a.padded + q * a.dp + c) = float2{v0, v1};
        const _Float16 h0 = qs.ok ? to_screen(v0, qs.s) : (_Float16)0.f;
        const _Float16 h1 = qs.ok ? to_screen(v1, qs.s) : (_Float16)0.f;
        const float w0 = v0 * qs.s, w1 = v1 * qs.s;
        const float d0 = w0 - (float)h0, d1 = w1 - (float)h1;
        n2 += w0 * w0 + w1 * w1;
        r2 += d0 * d0 + d1 * d1;
        // fragment order: 16-dim group c / 16, half (c / 8) % 2, query, dim c % 8
        *reinterpret_cast<ushort2*>(o + (c >> 3) * 256 + (c & 7)) = make_ushort2(
            __builtin_bit_cast(unsigned short, h0), __builtin_bit_cast(unsigned short, h1));
    }
    if (!live) return;
    n2 = wave_sum(n2);
    r2 = wave_sum(r2);
    if (lane == 0) {
        const float u = 0x1p-24f, D = (float)a.ds, X = a.x_norm, dX = a.x_res;
        const float qn = sqrtf(n2) * qs.inv_s, dq = sqrtf(r2) * qs.inv_s;
        const float rep = qn * dX + dq * (X + dX), ref = a.ref_terms * u;
        const float e = a.metric == 0 ? 2.f * rep + 4.f * D * u * (0.5f * X * X + qn * X) +
                                            D * u * X * X + ref * (qn + X) * (qn + X)
                                      : rep + 2.f * D * u * qn * X + ref * qn * X;
        a.err[q] = qs.ok && e < FLT_MAX * 0.25f ? 1.01f * e : __int_as_float(0x7f800000);
    }
}

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// LDS bytes of a query's select: candidates (8 bytes each), rows to re-rank, a histogram and
// the regions' offsets.
__host__ __device__ inline int screen_select_pitch(int lc, int regions) {
    return (lc * 12 + 1024 + (regions + 1) * 4 + 15) / 16 * 16;
}

// The select of a screened first round (flat_collect_select_kernel's rules for err), one wave a
// query: its candidates in LDS (LC at most; more is an overflow), the k-th smallest scan key
// by a radix select, everything up to twice the bound past it re-ranked in the reference's
// arithmetic by eight lanes each, and each result's place by counting those before it. WAVES =
// 1: four queries a workgroup, nothing waits for another wave (a workgroup a query spent its
// time at some sixty barriers of sorts: 10,000 queries, k = 10, 180 candidates 245 us, this 87;
// 4,999, k = 100, 370 candidates 228, this 150). WAVES = 16: a workgroup a query, all of whose
// waves re-rank (128 rows at once), for batches that leave the chip idle otherwise (three
// ADC queries, k = 50: one wave each 31 us, this 21).
template <int LC, int WAVES>
__global__ __launch_bounds__(WAVES == 1 ? 256 : 64 * WAVES) void screen_select_kernel(
    CollectSelectArgs a) {
    constexpr int PER = LC / 64;
    constexpr bool WIDE = WAVES > 1;
    extern __shared__ __attribute__((aligned(16))) char lds[];  // screen_select_lds
    __shared__ int s_m;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (a.status_host && blockIdx.x == 0 && threadIdx.x < 2)
        a.status_host[a.queries_n + threadIdx.x] = a.words[threadIdx.x];
    const int gave_up = *a.spin_fail;  // (looked at before the first write)
    const int b = WIDE ? blockIdx.x : blockIdx.x * 4 + wave;
    if (b >= a.slots) return;  // whole waves, and where WIDE whole workgroups
    const int pitch = screen_select_pitch(LC, a.regions);
    char* base = lds + (WIDE ? 0 : wave * pitch);
    unsigned long long* cand = reinterpret_cast<unsigned long long*>(base);
    int* list = reinterpret_cast<int*>(base + LC * 8);
    unsigned* hist = reinterpret_cast<unsigned*>(base + LC * 12);
    int* off = reinterpret_cast<int*>(base + LC * 12 + 1024);
    const int q = a.qlist ? a.qlist[b] : b;
    auto finish = [&](int status) __attribute__((always_inline)) {
        if (lane == 0) {
            a.status[q] = status;
            if (a.status_host) a.status_host[q] = status;
        }
    };
    // one wave: the rows to re-rank to list, and their number; -1: the query is not finished
    auto rows_to_rank = [&]() __attribute__((always_inline)) -> int {
        const float err = a.err[q];
        const float kInf = __int_as_float(0x7f800000);
        // offsets of the regions' stored candidates (all counts loaded before the first is
        // waited for)
        const int* cnt = a.cand_count + (int64_t)b * a.regions;
        int cv[kMaxCollectRegions / 64];
#pragma unroll
        for (int u = 0; u < kMaxCollectRegions / 64; ++u)
            cv[u] = lane + 64 * u < a.regions ? cnt[lane + 64 * u] : 0;
        int total = 0, held = 0;
        bool over = false;
#pragma unroll
        for (int u = 0; u < kMaxCollectRegions / 64; ++u) {
            const int r = lane + 64 * u, c = cv[u];
            if (64 * u >= a.regions) break;
            over |= __ballot(c > a.cap) != 0;
            const int st = min(c, a.cap);
            int incl = st, all = c;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(incl, o);
                if (lane >= o) incl += v;
                all += __shfl_xor(all, o);
            }
            if (r < a.regions) off[r] = min(held + incl - st, LC);
            held += __shfl(incl, 63);
            total += all;
        }
        over |= held > LC;
        held = min(held, LC);
        wave_lds_fence();
        if (gave_up) return -1;
        if (!over && total < a.kk) {
            // too few: the next, looser rung; past the last, or with no bound (which let no
            // row pass), the query cannot be screened
            const int r = a.rung[q] + 1;
            const bool more = r < kRungs && err < kInf;
            if (lane == 0 && more) {
                a.thr_key[q] = a.ladder_key[(int64_t)q * kRungs + r];
                a.rung[q] = r;
            }
            finish(more ? 1 : 2);
            return -1;
        }
        if (held < a.kk) {  // too many, but too few held: again, with larger regions
            finish(1);
            return -1;
        }
        // candidate lane + 64 u: its key (order-preserving unsigned form) and position: the
        // last region whose offset is at or below its number holds it
        unsigned ck[PER];
        int cp[PER];
        int steps = 0;
        while ((1 << steps) < a.regions) ++steps;
        const float* rk = a.cand_keys + (int64_t)b * a.regions * a.cap;
        const int* rp = a.cand_pos + (int64_t)b * a.regions * a.cap;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            ck[u] = 0xffffffffu;
            cp[u] = 0;
            const int i = lane + 64 * u;
            if (64 * u < held) {  // uniform
                int r = 0;
                for (int s = steps - 1; s >= 0; --s) {
                    const int r2 = r + (1 << s);
                    if (r2 < a.regions && off[r2] <= i) r = r2;
                }
                if (i < held) {
                    const int64_t at = (int64_t)r * a.cap + (i - off[r]);
                    PX_DCHECK(a.dbg, kDbgScreen, i - off[r] < a.cap);
                    ck[u] = (unsigned)total_key(rk[at]) ^ 0x80000000u;
                    cp[u] = rp[at];
                }
            }
        }
        // the kk-th smallest key: four 8-bit digits, most significant first
        unsigned pre = 0, need = (unsigned)a.kk;
        for (int pass = 0; pass < 4; ++pass) {
            const int shift = 24 - 8 * pass;
            *reinterpret_cast<uint4*>(hist + 4 * lane) = uint4{0, 0, 0, 0};
            wave_lds_fence();
#pragma unroll
            for (int u = 0; u < PER; ++u)
                if (lane + 64 * u < held && (pass == 0 || (ck[u] >> (shift + 8)) == pre))
                    atomicAdd(&hist[(ck[u] >> shift) & 0xffu], 1u);
            wave_lds_fence();
            const uint4 h = *reinterpret_cast<const uint4*>(hist + 4 * lane);
            const unsigned c[4] = {h.x, h.y, h.z, h.w};
            const unsigned sum = c[0] + c[1] + c[2] + c[3];
            unsigned incl = sum;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const unsigned v = __shfl_up(incl, o);
                if (lane >= o) incl += v;
            }
            unsigned before = incl - sum, below = 0;
            int digit = -1;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (digit < 0 && before + c[e] >= need) {
                    digit = 4 * lane + e;
                    below = before;
                }
                before += c[e];
            }
            // (need is at most the keys under the prefix: some lane has the digit)
            const int src = __builtin_ctzll(__ballot(digit >= 0));
            pre = (pre << 8) | (unsigned)__shfl(digit, src);
            need -= __shfl(below, src);
            wave_lds_fence();
        }
        const float cut = from_total_key((int)(pre ^ 0x80000000u)) + 2.f * err;
        const float thr = from_total_key(a.thr_key[q]);
        if (over || cut > thr) {
            // rows that may count were not collected: again, up to there
            if (lane == 0) a.thr_key[q] = total_key(over ? fminf(cut, thr) : cut);
            finish(1);
            return -1;
        }
        // the rows at or below the cut
        const unsigned cutk = (unsigned)total_key(cut) ^ 0x80000000u;
        int m = 0;
#pragma unroll
        for (int u = 0; u < PER; ++u) {
            const bool in = lane + 64 * u < held && ck[u] <= cutk;
            const unsigned long long mask = __ballot(in);
            if (in) list[m + __popcll(mask & ((1ull << lane) - 1ull))] = cp[u];
            m += __popcll(mask);
        }
        return m;
    };
    auto sync = [&]() __attribute__((always_inline)) {
        if constexpr (WIDE) __syncthreads();
        else wave_lds_fence();
    };
    int m = 0;
    if (!WIDE || wave == 0) m = rows_to_rank();
    if constexpr (WIDE) {
        if (threadIdx.x == 0) s_m = m;
        __syncthreads();
        m = s_m;
    }
    if (m < 0) return;  // (all of the workgroup's waves where they share the query)
    sync();
    // their keys in the reference's arithmetic, eight lanes a row: entry x is (key, id) as one
    // number that orders as they do
    const float* qv = a.queries + (int64_t)q * a.dp;
    const int tid = WIDE ? threadIdx.x : lane, gl = lane & 7;
    for (int x = tid >> 3; x < m; x += 8 * WAVES) {
        int id = list[x];
        if (a.rowidx) id = a.rowidx[id];
        float kv;
        if (a.corpus) {
            const float* xv = a.corpus + (int64_t)id * a.dp;
            kv = a.metric == 0 ? ref_key_g8(qv, xv, a.dim, true, gl)
                               : -ref_key_g8(qv, xv, a.dim, false, gl);
        } else {
            kv = ref_adc_g8(qv, a.books, a.codes + (int64_t)id * a.m, a.m, a.ks, a.dim / a.m,
                            a.metric == 0, gl);
        }
        if (gl == 0)
            cand[x] = (unsigned long long)((unsigned)total_key(kv) ^ 0x80000000u) << 32 |
                      (unsigned)id;
    }
    sync();
    for (int x = tid; x < m; x += 64 * WAVES) {
        const unsigned long long e = cand[x];
        int rank = 0;
        for (int y = 0; y < m; ++y) rank += cand[y] < e;
        if (rank >= a.k) continue;
        const float kv = from_total_key((int)((unsigned)(e >> 32) ^ 0x80000000u));
        a.out_ids[(int64_t)q * a.k + rank] = (int64_t)(unsigned)e;
        a.out_dists[(int64_t)q * a.k + rank] =
            a.raw_keys ? kv : (a.metric == 0 ? sqrtf(kv) : -kv);
    }
    if (!WIDE || wave == 0) finish(0);
}

// queries qlist[i] to dst[i] (rows of dp floats) ...
__global__ __launch_bounds__(256) void gather_queries_kernel(const float* q, const int* qlist,
                                                             int64_t n, int dp, float* dst) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n * dp) return;
    const int64_t r = e / dp;
    dst[e] = q[(int64_t)qlist[r] * dp + (e - r * dp)];
}
// ... and their results back
__global__ __launch_bounds__(256) void scatter_results_kernel(const int64_t* ids, const float* d,
                                                              const int* qlist, int64_t n, int k,
                                                              int64_t* out_ids, float* out_d) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= n * k) return;
    const int64_t r = e / k, o = (int64_t)qlist[r] * k + (e - r * k);
    out_ids[o] = ids[e];
    out_d[o] = d[e];
}

}  // namespace

int flat_screen_queries_per_block() { return kSlots; }

hipError_t launch_flat_screen(const ScreenArgs& a0, hipStream_t s) {
    ScreenArgs a = a0;
    if (a.spin_limit <= 0) a.spin_limit = kSpinLimit;
    const bool min = a.minima != nullptr;
    if (a.nq <= 0 || a.splits <= 0 || a.rows_per_split % kScreenRows != 0 || !a.spin_fail ||
        a.ds != a.chunks * kChunk || a.stride < 1 || !screen_batch_fits(a.nq, a.ds) ||
        (int64_t)a.splits * a.rows_per_split < a.n_eff ||
        (int64_t)(a.splits - 1) * a.rows_per_split >= a.n_eff)
        return hipErrorInvalidValue;
    if (min && (a.group_tiles < 1 || a.n_eff % kScreenRows != 0 ||
                a.n_eff % (kTile * a.group_tiles) != 0 ||
                a.rows_per_split % (kTile * a.group_tiles) != 0 ||
                a.n_eff / (kTile / 2 * a.group_tiles) > a.min_ld))
        return hipErrorInvalidValue;
    if (min) launch_screen_q<true>(a, s);
    else launch_screen_q<false>(a, s);
    return hipGetLastError();
}

hipError_t launch_abs_max(const float* x, int64_t count, float* parts, int* parts_n, int* words,
                          hipStream_t s) {
    if (count % 4 != 0 || ((uintptr_t)x & 15) != 0) return hipErrorInvalidValue;
    const int64_t blocks = std::max<int64_t>(
        1, std::min<int64_t>((count / 4 + 1023) / 1024, kAbsMaxParts));
    *parts_n = (int)blocks;
    hipLaunchKernelGGL(abs_max_kernel, dim3((unsigned)blocks), dim3(256), 0, s,
                       reinterpret_cast<const float4*>(x), count / 4, parts, words);
    return hipGetLastError();
}

hipError_t launch_screen_rows(const float* x, int64_t rows, int dp, int ds, int e,
                              unsigned short* out, int* max2, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((rows + 3) / 4, 8192);
    hipLaunchKernelGGL(screen_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, rows, dp,
                       ds, ldexpf(1.f, e), out, max2);
    return hipGetLastError();
}

hipError_t launch_screen_codes(const uint8_t* codes, int64_t rows, int dim, int ds, int m, int ks,
                               const float* books, int e, unsigned short* out, float* norms,
                               int* max2, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    const int64_t blocks = std::min<int64_t>((rows + 3) / 4, 8192);
    hipLaunchKernelGGL(screen_codes_kernel, dim3((unsigned)blocks), dim3(256), 0, s, codes, rows,
                       dim, ds, m, ks, books, ldexpf(1.f, e), out, norms, max2);
    return hipGetLastError();
}

hipError_t launch_screen_spread(const unsigned short* xs, int64_t rows, int ds, float* parts,
                                int* parts_n, hipStream_t s) {
    if (rows <= 0 || ds % 64 != 0) return hipErrorInvalidValue;
    // (past 16,384 dims the first of them stand for all)
    const int blocks = std::min(ds / 64, kAbsMaxParts / 2);
    *parts_n = 2 * blocks;
    hipLaunchKernelGGL(screen_spread_kernel, dim3((unsigned)blocks), dim3(256), 0, s, xs, rows, ds,
                       parts);
    return hipGetLastError();
}

hipError_t launch_screen_queries(const ScreenQueryArgs& a, hipStream_t s) {
    if (a.nq <= 0) return hipSuccess;
    if (a.dim > a.dp || a.dp > a.ds || (a.padded && (a.dp % 2 != 0 || a.qlist)))
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(screen_queries_kernel, dim3((unsigned)(screen_query_slots(a.nq) / 4)), dim3(256),
                       0, s, a);
    return hipGetLastError();
}

hipError_t launch_screen_select(const CollectSelectArgs& a, int lc, hipStream_t s) {
    if (a.slots <= 0 || !a.err || !a.spin_fail || a.kk > lc || a.regions > kMaxCollectRegions ||
        (lc != 512 && lc != 1024))
        return hipErrorInvalidValue;
    // one wave a query fills the chip with enough queries (us, one wave against sixteen: 1
    // query, k = 10: 18 / 16; 3 ADC queries, k = 50: 31 / 21; 500 of 768 dims, k = 20: 51 / 53;
    // 1,000 of 384, k = 10: 22 / 59)
    const bool wide = a.slots <= kScreenWideSlots ||
                      screen_select_pitch(lc, a.regions) * 4 > 65536;
    const dim3 grid((unsigned)(wide ? a.slots : (a.slots + 3) / 4)), block(wide ? 1024 : 256);
    const size_t lds = (size_t)screen_select_pitch(lc, a.regions) * (wide ? 1 : 4);
#define PX_SELECT(LC, WAVES) \
    hipLaunchKernelGGL((screen_select_kernel<LC, WAVES>), grid, block, lds, s, a)
    if (wide) {
        if (lc == 512) PX_SELECT(512, 16);
        else PX_SELECT(1024, 16);
    } else {
        if (lc == 512) PX_SELECT(512, 1);
        else PX_SELECT(1024, 1);
    }
#undef PX_SELECT
    return hipGetLastError();
}

hipError_t launch_gather_queries(const float* q, const int* qlist, int64_t n, int dp, float* dst,
                                 hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(gather_queries_kernel, dim3((unsigned)((n * dp + 255) / 256)), dim3(256), 0,
                       s, q, qlist, n, dp, dst);
    return hipGetLastError();
}

hipError_t launch_scatter_results(const int64_t* ids, const float* d, const int* qlist, int64_t n,
                                  int k, int64_t* out_ids, float* out_d, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(scatter_results_kernel, dim3((unsigned)((n * k + 255) / 256)), dim3(256), 0,
                       s, ids, d, qlist, n, k, out_ids, out_d);
    return hipGetLastError();
}

}  // namespace px
