// ============================================================================
//  batch_rq.hip — k_batch_rq: batched scoring with the queries held in registers,
//  for batches of up to 1023 queries (64, 128 or 256 per workgroup, one corpus pass each).
//
//  A query tile of 256 fp16 queries x d does not fit in LDS (384 KiB at d = 768), but
//  it fits in the register files of one CU: each of the four waves (one per SIMD, the
//  whole 512-register file) holds 16 QT queries as MFMA A fragments for the whole kernel
//  (NS x QT fragments of 16 bytes per lane: 384 registers at d = 768 and QT = 4). Only
//  the corpus moves: 16-row tiles stream from HBM straight into LDS
//  (global_load_lds_dwordx4, each wave loading a quarter of every tile, whole rows
//  contiguous), four tile buffers deep, and all four waves read every tile's B fragments
//  from LDS. Each corpus row is read from HBM once per workgroup's 64 QT queries, and the
//  CU takes in nothing else.
//
//  Tile layout in LDS: row r's 16-byte piece p sits in slot r * P + (p ^ (r & 15)),
//  P = d / 8 pieces per row. A B-fragment read (lanes 16 g .. 16 g + 15: rows 0 .. 15,
//  the same piece) then touches 16 distinct 16-byte bank groups.
//
//  Scores: the same MFMA, operands and k order as k_batch_scan (queries the A operand,
//  rows the B operand, k-steps 0 .. NS - 1 accumulated in order from zero), so every raw
//  score is bit-identical to that kernel's, and so is every fused score. Selection: every
//  product is tested in the MFMA layout (a lane holds one row's scores for 4 QT queries)
//  against its query's bound (a floor from the sampled pass of launch_batch_topk, then its K-th
//  best), between the MFMAs of the next tile; the few that reach it are fused, exactly as
//  k_batch_scan does, and offered to their query's list of K keys. Output: K keys per (query,
//  row range), or over few rows every row's score (BatchArgs::scores), as k_batch_merge reads them.
//
//  What bounds it (1M rows, d = 768, 256 queries of one time): the pass takes 375 us, 360 us with
//  the selection switched off, against 160 us of MFMAs alone and 260 us of row loads alone: the
//  matrix cores' issue and the loads' share one wave per SIMD. 450 us before: the test ran after
//  a tile's MFMAs, the tile loads were issued in one block before them, and a tile with a pair
//  went through LDS into sorted lists. 128 queries over 100K rows: 183 -> 70 us (half of that the
//  selection: rows of one recent episode reach the bounds of many queries at once).
//
//  Reference analogue: wmma_mma_similarity_kernel / wmma_similarity_kernel
//  (src/wmma_similarity.cu:55-138), which score one query and are never called.
// ============================================================================
#include "device.hpp"

#include <cfloat>

namespace mars {
namespace {

constexpr int kRWaves = 4;     // one per SIMD; each holds QT 16-query MFMA tiles
constexpr int kRThreads = kRWaves * 64;
constexpr int kRRows = 16;     // corpus rows per tile
constexpr int kRBuf = 4;       // tile buffers: see the main loop
constexpr int kRAhead = 4;     // B fragment registers: k-steps read 3 ahead
constexpr int kRMeet = 2;      // the k-step before which the waves meet
constexpr int kRqSparse = 6;   // at most this many lanes with one pair each: the pairs one at a time

template <int NS, int K, int QT>
struct RqLds {
    u32x4 tile[kRBuf][kRRows * NS * 4];          // 16 rows x d / 8 pieces, swizzled
    uint32_t side[kRBuf][kRWaves][64];           // per wave: lanes 0-15 the rows' timestamps, 16-31 modalities
    alignas(16) float stage[kRWaves][kRRows][16 * QT + 1];   // per-wave score tile (+1: bank spread)
    float wrow[kRWaves][kRRows];                 // per wave: the tile rows' weights (or timestamps)
    uint64_t list[kRWaves][K][16 * QT];          // per wave: its queries' best keys, in no order
    alignas(16) float floorv[kRWaves][16 * QT];  // per wave: its queries' bounds (-inf: none)
    float scale[kRWaves][16 * QT];               // per wave: its queries' 1 / A_q (k_batch_rq)
    alignas(16) float tqv[kRWaves][16 * QT];     // per wave: its queries' times
};

// s_waitcnt immediates (gfx9 encoding: vmcnt[3:0] and [15:14], expcnt[6:4], lgkmcnt[11:8])
constexpr int rq_wait_vm(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
constexpr int kRqWaitLgkm0 = 15 | (3 << 14) | (7 << 4);

// Orders this wave's LDS writes before its later LDS reads (the score stage is private
// to one wave).
__device__ inline void rq_wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// One 16-byte (or 4-byte) piece per lane from global memory straight into LDS: lane l
// writes lds + l * bytes.
__device__ __attribute__((always_inline)) inline void dma16(const void* g, u32x4* lds) {
    __builtin_amdgcn_global_load_lds(g, lds, 16, 0, 0);
}
__device__ __attribute__((always_inline)) inline void dma4(const void* g, uint32_t* lds) {
    __builtin_amdgcn_global_load_lds(g, lds, 4, 0, 0);
}

// Workgroups per query group of a launch that keeps every row's score: one tile each, at most 256 in all.
__host__ __device__ inline int rq_all_wgs(const BatchArgs& a) {
    const int wgq = a.q <= 64 ? 64 : a.q <= 128 ? 128 : 256, groups = (a.q + wgq - 1) / wgq;
    const int64_t tiles = (a.n + kRRows - 1) / kRRows, most = 256 / groups > 1 ? 256 / groups : 1;
    return int(tiles < most ? tiles : most);
}

// QT: 16-query MFMA tiles per wave (1, 2 or 4: 64, 128 or 256 queries per workgroup). MODE: the
// full pass keeps the best K keys per query and range; the sampled pass of launch_batch_topk
// keeps K row-class maxima instead; kRqAll writes every row's score (BatchArgs::scores).
constexpr int kRqFull = 0, kRqSample = 1, kRqAll = 2;
template <int NS, int K, int QT, int MODE>
__global__ __launch_bounds__(kRThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
void k_batch_rq(BatchArgs a) {
    __shared__ __attribute__((aligned(16))) RqLds<NS, K, QT> sh;
    static_assert(sizeof(sh) <= 160 * 1024, "LDS");
    constexpr bool FULL = MODE == kRqFull, ALL = MODE == kRqAll;
    constexpr int WQ = 16 * QT;                  // queries per wave
    constexpr int P = NS * 4;                    // 16-byte pieces per row
    constexpr int kLd = NS / 4;                  // tile loads per wave (64 slots each)
    static_assert(NS % 4 == 0 && P % 16 == 0, "tile layout");
    const int tid = int(threadIdx.x), lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = lane & 15, kg = lane >> 4;
    constexpr int d = NS * 32;
    // every row's score: the tiles are dealt out evenly, wg_rows per workgroup
    const int n_wg = ALL ? rq_all_wgs(a) : a.n_rranges;           // workgroups per query group
    const int wg_rows = int((a.n + kRRows * n_wg - 1) / (kRRows * n_wg)) * kRRows;
    const int r_id = int(blockIdx.x) % n_wg;
    const int g = int(blockIdx.x) / n_wg;                                         // the workgroup's group of 64 QT queries
    const int wq0 = (g * kRWaves + wave) * WQ;                    // this wave's first query
    // rows and tiles in 32 bits (the launch checks that the row numbers fit)
    const int r0 = int(int64_t(r_id) * (ALL ? wg_rows : a.range_stride > 0 ? a.range_stride : a.rows_per_range));
    const int64_t rows = ALL ? wg_rows : a.rows_per_range;
    const int r1 = int(a.n < r0 + rows ? a.n : r0 + rows);
    const int ntiles = r1 > r0 ? (r1 - r0 + kRRows - 1) / kRRows : 0;

    // This lane's slots of a tile: load j of the wave fills slots s = (wave kLd + j) 64 +
    // lane, i.e. slot s % P of row s / P, which holds piece (s % P) ^ (row & 15). Two slots per
    // register: row << 8 | piece.
    uint32_t lin2[(kLd + 1) / 2];
    static_assert(P <= 256, "8-bit pieces");
#pragma unroll
    for (int j = 0; j < kLd; ++j) {
        const int s = (wave * kLd + j) * 64 + lane;
        const uint32_t o = uint32_t((s / P) << 8 | ((s % P) ^ ((s / P) & 15)));
        lin2[j / 2] = j % 2 ? lin2[j / 2] | o << 16 : o;
    }
    // lanes 0-15 load the rows' timestamps, 16-31 their modalities
    const char* const side_base = lane >= 16 && lane < 32 ? reinterpret_cast<const char*>(a.mods) : reinterpret_cast<const char*>(a.ts);
    // Load j of tile tt (kLd: the side data) into buffer b. Tiles past the last load the last one
    // again, so every iteration issues the same loads and the wait counts stay exact; rows past
    // the range's end are clamped to its last. Branch-free, so that it fits between MFMAs.
    auto issue_piece = [&](int tt, int b, int j) {
        tt = tt < ntiles ? tt : ntiles - 1;
        const int base = r0 + tt * kRRows;
        const uint32_t last = uint32_t(r1 - 1 - base < kRRows - 1 ? r1 - 1 - base : kRRows - 1);
        if (j == kLd) {
            const uint32_t r = uint32_t(lane & 15) < last ? uint32_t(lane & 15) : last;
            dma4(side_base + int64_t(base + int(r)) * 4, &sh.side[b][wave][0]);
            return;
        }
        const uint32_t o = (lin2[j / 2] >> (16 * (j % 2))) & 0xFFFFu;
        const uint32_t r = (o >> 8) < last ? (o >> 8) : last;
        dma16(uniform_ptr(reinterpret_cast<const char*>(a.emb16 + int64_t(base) * d)) + (r * uint32_t(d * 2) + (o & 0xFFu) * 16u),
              &sh.tile[b][(wave * kLd + j) * 64]);
    };
    if (ntiles > 0) {
#pragma unroll
        for (int b = 0; b < kRBuf - 1; ++b)
#pragma unroll
            for (int j = 0; j <= kLd; ++j) issue_piece(b, b, j);
    }

    // The wave's WQ queries as A fragments: af[qt][ks] = query wq0 + qt*16 + m,
    // halves ks*32 + kg*8 .. +7 (zero past the batch).
    f16x8 af[QT][NS];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int qrow = wq0 + qt * 16 + m;
        const bool ok = qrow < a.q;
        const u32x4* qp = reinterpret_cast<const u32x4*>(a.qh + int64_t(ok ? qrow : 0) * d + kg * 8);
#pragma unroll
        for (int ks = 0; ks < NS; ++ks) {
            const u32x4 v = ok ? qp[ks * 4] : u32x4{0u, 0u, 0u, 0u};
            af[qt][ks] = __builtin_bit_cast(f16x8, v);
        }
    }

    // lane j < WQ owns query wq0 + j
    const int myq = wq0 + lane;
    const bool qvalid = lane < WQ && myq < a.q;
    const bool wave_live = wq0 < a.q;            // uniform: the wave has queries to score
    if (lane < WQ) sh.tqv[wave][lane] = qvalid ? a.tq[myq] : 0.0f;
    const bool uni = a.uniform_tq != 0;
    const float tq0 = a.tq[0];
    const bool plain = myq >= a.q_plain;          // neighbour search: dot product only
    // Sampled pass: the maxima (query qt*16 + 4*kg + v, rows m mod 16).
    float mx[4 * QT];
#pragma unroll
    for (int i = 0; i < 4 * QT; ++i) mx[i] = -INFINITY;
    // Full pass: lane j keeps its query's best keys in LDS, unordered (the merge takes any order),
    // so a key costs one store until K are held, and a search of the 16 for the new worst one after
    // that. (The registers hold the queries and one tile's products; sorted lists there, 32
    // registers at K = 16, left no room to test a tile during the next one's MFMAs.)
    uint32_t own = 0u;                           // ord32 of the bound: max(floor, the worst of K keys' score)
    uint32_t cnt = 0u;                           // keys held; K + slot of the worst one once K are
    if (FULL && a.floor_keys != nullptr && qvalid) {
        const uint64_t fk = a.floor_keys[int64_t(myq) * a.floor_k + a.floor_k - 1];
        if (fk != kEmptyKey) own = ord32(key_score(fk));
    }

    // The test's weight of a row and bound of a query. One query time: the row's own weight, and the
    // test compares the score itself. Per-query times: w(q, row) = exp(-lambda max(0, tq - ts)) <=
    // A_q B_row with A_q = exp(-lambda (tq - tmin)), B_row = min(exp(lambda (ts - tmin)), exp(40))
    // (tmin the wave's earliest time; equal where ts <= tq), so a row reaches the query's bound f > 0
    // only if x B_row >= f / A_q, up to rounding. Where the wave's times span more than exp(40):
    // w <= exp(-lambda max(0, tmin - ts)); with a time that is not finite: w <= 1; lambda < 0: NaN,
    // which passes everything. (Testing x itself against f passed most positive products when
    // decay separates the rows: 100 queries of mixed times over 100K rows, full pass 130 us.)
    float tmin = INFINITY, lam_b = 0.0f;
    bool clamp_b = true;
    if (FULL && !uni) {
        const float tq = sh.tqv[wave][lane & (WQ - 1)];
        const bool fused = qvalid && !plain;
        float tmax = -INFINITY;
        if (fused) { tmin = tq; tmax = tq; }
#pragma unroll
        for (int x = 32; x >= 1; x >>= 1) {
            tmin = fminf(tmin, __shfl_xor(tmin, x));
            tmax = fmaxf(tmax, __shfl_xor(tmax, x));
        }
        tmin = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(tmin)));
        tmax = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(tmax)));
        float scale = 1.0f;
        if (__ballot(fused && !(fabsf(tq) < INFINITY)) == 0) {
            lam_b = a.lambda;
            clamp_b = !(a.lambda * (tmax - tmin) <= 40.0f);
            if (!clamp_b) scale = expf(a.lambda * (tq - tmin));
        }
        if (!(a.lambda >= 0.0f)) lam_b = __builtin_nanf("");
        if (lane < WQ) sh.scale[wave][lane] = fused ? scale : 0.0f;        // 0: the bound as it is
    }
    // Rounding: 1e-4 (publish) covers the exponents' (arguments up to 100, 2 ulp), 1e-25 a weight
    // that underflowed (A_q >= exp(-40)); products of fp16 rows (|x| < 4e12) times B_row don't overflow.
    auto row_weight = [&](float ts) {
        if (uni) return a.lambda != 0.0f ? expf(-a.lambda * fmaxf(0.0f, tq0 - ts)) : 1.0f;
        if (lam_b == 0.0f) return 1.0f;
        const float age = tmin - ts;
        const float w = expf(-lam_b * (clamp_b ? fmaxf(0.0f, age) : age)) + 1e-25f;
        return w > 2.4e17f ? 2.4e17f : w;
    };
    // the bound of this lane's query, as the test takes it; past the batch +inf. Per-query times: a
    // bound <= 0 lets every unfiltered row pass (x B_row is no bound of a negative score).
    auto publish = [&]() {
        float f = own != 0u ? ord32_inv(own) : -INFINITY;
        if (!uni) {
            const float sc = sh.scale[wave][lane];
            if (sc > 0.0f) {
                if (f > 1e-30f) f = fminf(f * sc * (1.0f - 1e-4f), FLT_MAX);
                else if (f > -1e38f) f = -1e38f;
            }
        }
        sh.floorv[wave][lane] = qvalid ? f : INFINITY;
    };
    if (FULL && lane < WQ) publish();
    // a row's key for this lane's query, whose score is not below the query's bound
    auto offer = [&](uint64_t key) {
        uint32_t at = cnt;
        if (cnt >= K) {
            at = cnt - K;
            if (!(key < sh.list[wave][at][lane])) return;
        }
        sh.list[wave][at][lane] = key;
        if (cnt < K && ++cnt < K) return;
        uint64_t worst = 0;
#pragma unroll
        for (int j = 0; j < K; ++j) {
            const uint64_t e = sh.list[wave][j][lane];
            cnt = e >= worst ? uint32_t(K + j) : cnt;
            worst = e >= worst ? e : worst;
        }
        const uint32_t o = ord32(key_score(worst));
        if (o > own) {
            own = o;
            publish();
        }
    };

    // B-fragment slots: k-step ks reads piece 4 ks + kg of row m, i.e. slot
    // m P + ((4 ks + kg) ^ m) = m P + 16 (ks / 4) + ((4 (ks % 4)) ^ kg ^ m)
    // (m P is a multiple of 16: one register, the k-step's part is an xor).
    const int boff = m * P + (kg ^ m);
    auto bfrag = [&](int b, int ks) {
        return __builtin_bit_cast(f16x8, sh.tile[b][(boff ^ (4 * (ks & 3))) + 16 * (ks >> 2)]);
    };
    // this lane's first query, relative to the first neighbour search; laundered, so that the
    // 4 QT values derived from it are computed where they are used rather than held across the loop
    auto first_rel = [&]() {
        int qrel = wq0 + 4 * kg - a.q_plain;
        asm volatile("" : "+v"(qrel));
        return qrel;
    };

    // The tile under test: its products, and of this lane's row (m) the test's weight and offset
    // (a filtered row: 0 and -FLT_MAX), the weight (or timestamp) the score takes, the filter flag.
    // Element e of the test is in the MFMA layout: C[query qt*16 + 4*kg + v][row m], e = 4 qt + v;
    // the row passes unless x weight + offset < the query's bound (NaN passes). A wave of both
    // global queries and neighbour searches (whose score is x) takes every tile to select_tile.
    f32x4 tacc[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) tacc[qt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float tw = 0.0f, tb = 0.0f, tsc = 0.0f;
    bool tkeep = false;
    const bool all_plain = wq0 >= a.q_plain, mixed = !all_plain && wq0 + WQ > a.q_plain;
    auto bounds = [&](int qt) { return *reinterpret_cast<const f32x4*>(&sh.floorv[wave][qt * 16 + 4 * kg]); };

    // The tile under test at row t0 may have pairs that reach their bounds: offers those rows.
    auto select_tile = [&](int t0) {
        const int nr = r1 - t0 < kRRows ? r1 - t0 : kRRows;
        const int qrel = first_rel();
        uint32_t hb = 0u;                        // bit e: this lane's row reaches element e's query
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            const f32x4 fl = bounds(qt);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float x = tacc[qt][v];
                float sv = fmaf(x, tw, tb);
                sv = (qrel + qt * 16 + v >= 0) ? x : sv;
                hb |= uint32_t(!(sv < fl[v])) << (4 * qt + v);
            }
        }
        hb = m < nr ? hb : 0u;
        const uint64_t hl = __ballot(hb != 0u);
        if (hl == 0) return;
        // The fused score of a row for this lane's query: dot * w (k_batch_scan's arithmetic),
        // filtered rows -FLT_MAX, neighbour searches the plain dot. wj: the row's weight at the
        // one query time, else its timestamp.
        auto fuse = [&](float x, float wj, bool keep) {
            float sv = x;
            if (uni) sv = x * wj;
            else if (a.lambda != 0.0f) sv = x * expf(-a.lambda * fmaxf(0.0f, sh.tqv[wave][lane & (WQ - 1)] - wj));
            sv = keep ? sv : -FLT_MAX;
            return plain ? x : sv;
        };
        const uint32_t keepm = uint32_t(__ballot(tkeep && lane < kRRows));
        // the query's own row (a neighbour search of a corpus row), relative to the tile
        int32_t self_t = -1;
        if (a.self_base >= 0 && plain) {
            const int64_t rel = a.self_base + (myq - a.q_plain) - t0;
            self_t = rel >= 0 && rel < kRRows ? int32_t(rel) : -1;
        }
        // The rows of this lane's query: bit e of lane (m, kg) is row m of query (e / 4)*16 + 4*kg
        // + e % 4. A few lanes with one pair each: pair by pair, the score going by readlane; else
        // the products transposed through LDS and one row per lane and round.
        uint64_t ln = hl;
        uint32_t pass = 0u;
        float hx = 0.0f;
        const int be = hb != 0u ? __builtin_ctz(hb) : 0;
        const bool sparse = __popcll(hl) <= kRqSparse && __ballot((hb & (hb - 1u)) != 0u) == 0;
        if (sparse) {
#pragma unroll
            for (int e = 0; e < 4 * QT; ++e) hx = be == e ? tacc[e >> 2][e & 3] : hx;
        } else {
            const int my_e = 4 * (lane >> 4) + (lane & 3), my_kg = (lane >> 2) & 3;
            if (lane < kRRows) sh.wrow[wave][lane] = tsc;
#pragma unroll
            for (int e = 0; e < 4 * QT; ++e) {
                sh.stage[wave][m][(e >> 2) * 16 + 4 * kg + (e & 3)] = tacc[e >> 2][e & 3];
                const uint64_t mk = __ballot((hb >> e) & 1u);
                const uint32_t h = my_kg >= 2 ? uint32_t(mk >> 32) : uint32_t(mk);
                pass = my_e == e ? (h >> (16 * (my_kg & 1))) & 0xFFFFu : pass;
            }
            rq_wave_lds_sync();
            if (!qvalid) pass = 0u;
            if (self_t >= 0) pass &= ~(1u << self_t);
        }
        for (;;) {
            int j = 0;
            float x = 0.0f, wj = 0.0f;
            bool mine = false;
            if (sparse) {
                if (ln == 0) break;
                const int L = __builtin_ctzll(ln);
                ln &= ln - 1;
                const int e1 = __builtin_amdgcn_readlane(be, L);
                j = L & 15;
                x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(hx), L));
                wj = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(tsc), j));
                mine = lane == (e1 >> 2) * 16 + 4 * (L >> 4) + (e1 & 3) && qvalid && j != self_t;
            } else {
                if (__ballot(pass != 0u) == 0) break;
                mine = pass != 0u;
                if (mine) {
                    j = __builtin_ctz(pass);
                    pass &= pass - 1u;
                    x = sh.stage[wave][j][lane];
                    wj = sh.wrow[wave][j];
                }
            }
            if (mine) {
                const float sv = fuse(x, wj, (keepm >> j) & 1u);
                if (ord32(sv) >= own) offer(make_key(sv, uint32_t(t0 + j)));
            }
        }
        rq_wave_lds_sync();
    };

    // The main loop is one stream of k-steps over all tiles: the fragments of a tile's first k-steps
    // are read during the tile before, so the matrix cores run on. Before k-step kRMeet of tile i a
    // wave waits for its loads of tile i + 1 and meets the others: then tile i + 1 is whole, and
    // every wave is done with tile i - 1, whose buffer takes the loads of tile i + 3, spread over
    // tile i's k-steps (all at once, they wait for the address unit with the matrix core idle).
    // Between the MFMAs (groups of one and a few vector operations, which fit beside it) goes the
    // test of tile i - 1's products (the first tile tests zeros nobody reads).
    constexpr int kLdStep = (NS - kRMeet) / (kLd + 1);
    static_assert(NS % kRAhead == 0 && kLdStep >= 1 && kRBuf == 4, "the k-step ring and the loads' places");
    f16x8 bf[kRAhead];
    auto meet = [&](int tiles_in_flight) {
        if (tiles_in_flight == 2) __builtin_amdgcn_s_waitcnt(rq_wait_vm(2 * (kLd + 1)));
        else __builtin_amdgcn_s_waitcnt(rq_wait_vm(kLd + 1));
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (ntiles > 0) {
        __builtin_amdgcn_s_waitcnt(kRqWaitLgkm0);
        meet(2);
        if (wave_live) {
#pragma unroll
            for (int j = 0; j < kRAhead - 1; ++j) bf[j] = bfrag(0, j);
        }
    }
    int b = 0;
    // (the full pass's last iteration has no tile of its own: it tests the last tile)
    for (int i = 0; i < ntiles + (FULL ? 1 : 0); ++i) {
        const int t0 = r0 + i * kRRows;
        uint64_t hits = ~0ull;                   // lanes whose row reached a bound in the tile under test
        f32x4 acc[QT] = {};
        float sts = 0.0f;
        bool keep_m = false;
        if (i < ntiles) {
            const int bn = (b + kRBuf - 1) & (kRBuf - 1), b1 = (b + 1) & (kRBuf - 1);
            if (wave_live) {
                // row m of the tile: timestamp, filter flag
                sts = __uint_as_float(sh.side[b][wave][m]);
                keep_m = a.mod_filter < 0 || int32_t(sh.side[b][wave][16 + m]) == a.mod_filter;
                if constexpr (FULL) hits = mixed ? ~0ull : 0ull;
                f32x4 fl{}, fn{};
                if constexpr (FULL) fn = bounds(0);
#pragma unroll
                for (int ks = 0; ks < NS; ++ks) {
                    if (ks == kRMeet) meet(1);
                    const int ka = ks + kRAhead - 1;
                    bf[ka % kRAhead] = ka < NS ? bfrag(b, ka) : bfrag(b1, ka - NS);
#pragma unroll
                    for (int qt = 0; qt < QT; ++qt)
                        acc[qt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[qt][ks], bf[ks % kRAhead],
                                                                         ks == 0 ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[qt], 0, 0, 0);
                    if (ks >= kRMeet && (ks - kRMeet) % kLdStep == 0 && (ks - kRMeet) / kLdStep <= kLd)
                        issue_piece(i + kRBuf - 1, bn, (ks - kRMeet) / kLdStep);
                    if constexpr (FULL) {
#pragma unroll
                        for (int e = ks * 4 * QT / NS; e < (ks + 1) * 4 * QT / NS; ++e) {
                            if ((e & 3) == 0) {
                                fl = fn;
                                if (e / 4 + 1 < QT) fn = bounds(e / 4 + 1);
                            }
                            hits |= __ballot(!(fmaf(tacc[e >> 2][e & 3], tw, tb) < fl[e & 3]));
                        }
                    }
#pragma unroll
                    for (int qt = 0; qt < QT; ++qt) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);       // one MFMA
                        __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);       // three vector operations
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
                meet(1);
#pragma unroll
                for (int j = 0; j <= kLd; ++j) issue_piece(i + kRBuf - 1, bn, j);
            }
            b = b1;
        }
        if constexpr (!FULL) {
            if (wave_live) {
                const int nr = r1 - t0 < kRRows ? r1 - t0 : kRRows;
                const int qrel = first_rel();
                const float w_m = row_weight(sts);
                // the row's fused score (the selection's operations, so the same bits) for each
                // of the lane's queries; self: the neighbour search whose own row this is
                const int64_t self64 = a.self_base >= 0 ? t0 + m - a.self_base : -1;
                const int self = self64 >= 0 && self64 < a.q ? int(self64) : -1;
#pragma unroll
                for (int qt = 0; qt < QT; ++qt) {
                    const f32x4 tqv = *reinterpret_cast<const f32x4*>(&sh.tqv[wave][qt * 16 + 4 * kg]);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float x = acc[qt][v];
                        const int qi = qrel + qt * 16 + v;
                        float sv = x;
                        if (uni) sv = x * w_m;
                        else if (a.lambda != 0.0f) sv = x * expf(-a.lambda * fmaxf(0.0f, tqv[v] - sts));
                        sv = keep_m ? sv : -FLT_MAX;
                        sv = qi >= 0 ? x : sv;
                        __builtin_amdgcn_sched_barrier(0);       // one score at a time: no registers for more
                        const bool in = m < nr && !(qi >= 0 && qi == self);
                        if constexpr (!ALL) {
                            mx[4 * qt + v] = in ? fmaxf(mx[4 * qt + v], sv) : mx[4 * qt + v];
                        } else {
                            // row t0 + m is score m of range (t0 + m) / 16 (the query's own row among
                            // them; rows past the last are not written)
                            const int q = qi + a.q_plain;
                            if (q < a.q && m < nr)
                                reinterpret_cast<float*>(a.part)[((int64_t(q / 64) * a.n_rranges + t0 / kRRows) * 64 + q % 64) * kRRows + m] = sv;
                        }
                    }
                }
            }
        } else {
            if (wave_live && i > 0 && hits != 0) select_tile(t0 - kRRows);
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) tacc[qt] = acc[qt];
            tw = row_weight(sts);
            tsc = uni ? tw : sts;
            tkeep = keep_m;
            tb = keep_m || all_plain ? 0.0f : -FLT_MAX;
            tw = all_plain ? 1.0f : keep_m ? tw : 0.0f;
        }
    }
    // the last iterations' loads (clamped tiles nobody reads) must land before the
    // workgroup ends and its LDS is handed to another
    __builtin_amdgcn_s_waitcnt(rq_wait_vm(0));
    if constexpr (MODE == kRqSample) {
        // K distinct rows' scores per query and range: the maxima of the 16 row classes, or (K = 8)
        // of the class pairs m, m + 8; keyed with the class (only the score is used). A class without
        // a score above -inf (no rows, or NaN alone, which ranks below -inf) is no row to count.
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int qi = wq0 + qt * 16 + 4 * kg + v;
                float x = mx[4 * qt + v];
                if constexpr (K == 8) x = fmaxf(x, xor_lanef<8>(x));
                if (qi < a.q && m < K)
                    a.part[((int64_t(qi / 64) * a.n_rranges + r_id) * 64 + qi % 64) * K + m] =
                        x > -INFINITY ? make_key(x, uint32_t(r0) + uint32_t(m)) : kEmptyKey;
            }
    } else if constexpr (FULL) {
        if (qvalid) {
            uint64_t* out = a.part + ((int64_t(myq / 64) * a.n_rranges + r_id) * 64 + myq % 64) * K;
#pragma unroll
            for (int j = 0; j < K; ++j) out[j] = uint32_t(j) < cnt ? sh.list[wave][j][lane] : kEmptyKey;
        }
    }
}

template <int NS, int K, int QT>
int launch_rq_q(const BatchArgs& a, hipStream_t s) {
    constexpr int wgq = kRWaves * 16 * QT;       // queries per workgroup
    const unsigned grid = unsigned((a.scores ? rq_all_wgs(a) : a.n_rranges) * ((a.q + wgq - 1) / wgq));
    if constexpr (K == 16) {
        if (a.scores) {
            MARS_LAUNCH((k_batch_rq<NS, K, QT, kRqAll>), dim3(grid), dim3(kRThreads), 0, s, a);
            return MARS_OK;
        }
    }
    if (a.sample_pass)
        MARS_LAUNCH((k_batch_rq<NS, K, QT, kRqSample>), dim3(grid), dim3(kRThreads), 0, s, a);
    else
        MARS_LAUNCH((k_batch_rq<NS, K, QT, kRqFull>), dim3(grid), dim3(kRThreads), 0, s, a);
    return MARS_OK;
}

template <int NS, int K>
int launch_rq_t(const BatchArgs& a, hipStream_t s) {
    switch (batch_rq_tiles(a.q)) {
        case 1: return launch_rq_q<NS, K, 1>(a, s);
        case 2: return launch_rq_q<NS, K, 2>(a, s);
        default: return launch_rq_q<NS, K, 4>(a, s);
    }
}

template <int K>
int launch_rq_k(const BatchArgs& a, hipStream_t s) {
    switch (a.d / 32) {
        case 8: return launch_rq_t<8, K>(a, s);
        case 12: return launch_rq_t<12, K>(a, s);
        case 16: return launch_rq_t<16, K>(a, s);
        case 24: return launch_rq_t<24, K>(a, s);
        default: return set_error(MARS_ERR_UNSUPPORTED, "batched scoring: embedding_dim %d not in {256,384,512,768}", a.d);
    }
}

}  // namespace

int launch_batch_rq(const BatchArgs& a, hipStream_t s) {
    MARS_CHECK(a.k >= 1 && a.k <= 16, MARS_ERR_UNSUPPORTED, "batched scoring keeps at most 16 per query (asked %d)",
               a.k);
    MARS_CHECK(a.n <= INT32_MAX - 64, MARS_ERR_CAPACITY, "batched scoring: %lld rows", (long long)a.n);
    MARS_CHECK(a.n_qblocks == (a.q + 63) / 64, MARS_ERR_INVALID, "batched scoring: %d query blocks for %d queries",
               a.n_qblocks, a.q);
    return a.k <= 8 && !a.scores ? launch_rq_k<8>(a, s) : launch_rq_k<16>(a, s);
}

}  // namespace mars
