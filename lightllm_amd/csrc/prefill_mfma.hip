// MFMA paged prefill attention (see prefill_mfma.h for the design).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

#include "prefill_mfma.h"

namespace llkv {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
// Native vector for staged K/V rows (HIP's uint4 struct is copied with memcpy,
// which keeps the staging registers in scratch memory).
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

template <typename T> struct Mfma;

template <> struct Mfma<_Float16> {
    typedef f16x8 vec;
    __device__ static inline f32x4 mma(const uint4& a, const uint4& b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                     __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
    __device__ static inline uint32_t pack2(float x, float y) { return pack_h2(x, y); }
    static constexpr uint32_t kOnes = 0x3C003C00u;   // two halves of 1.0
};

template <> struct Mfma<bf16_t> {
    typedef bf16x8 vec;
    __device__ static inline f32x4 mma(const uint4& a, const uint4& b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                      __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    __device__ static inline f32x16 mma32(const uint4& a, const uint4& b, f32x16 c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    __device__ static inline uint32_t pack2(float x, float y) { return pack_b2(x, y); }
    static constexpr uint32_t kOnes = 0x3F803F80u;   // two bfloat16 1.0
};

constexpr int BQ = 128;   // query rows per work-group

// Key-chunk partial rows are fp32 for every pool type.  fp16 rows (half the
// merge's traffic, 2-3 us on configuration 4) added a rounding of each chunk's
// normalised row, which chunks of opposite sign amplify in the merged output:
// seeded ragged batches over 4k-key prefixes went past the fp16 bound.
constexpr int WQ = 32;    // query rows per wave (two 16-column MFMA tiles)
constexpr int BN = 64;    // keys per tile (four pages)

// Unit u = (sequence n, query block qb): its query rows [q_lo, q_lo + BQ) of
// the sequence's P new tokens (starting at row q0 of q) over L keys, and its
// key tiles (the causal extent of the rows).  Query blocks are numbered from
// the last, so that in a sequence the longest unit comes first.
struct UnitInfo {
    int q0, P, L, kvo, hist, tiles;
};

// Sequence n's first q row, new tokens P, keys L, and (contiguous K/V) the
// element offset of its first K/V row.  Paged: rows cu_q[n] .. cu_q[n+1],
// L = seq_lens[n] capped at the table's extent.  Contiguous (first prefill):
// q rows from offsets[n] (a row start), P = token_cumsum[n + 1] - token_cumsum[n],
// L = num_tokens[n].
// hist: keys before query row 0's own position, so that causal query row i
// sees keys j <= hist + i (L - P for a chunk on a cached prefix; 0 for a first
// prefill entry, whose query and key counts may differ).
__device__ inline void seq_geom(const MfmaPrefillArgs& a, int n, int& q0, int& P, int& L, int& kvo,
                                int& hist) {
    if (a.contig) {
        q0 = a.q_off[n] / a.q_row;
        P = max(a.tcum[n + 1] - a.tcum[n], 0);
        L = max(a.ntok[n], 0);
        kvo = a.kv_off[n];
        hist = 0;
    } else {
        q0 = a.cu_q[n];
        P = a.cu_q[n + 1] - q0;
        const int l = a.lens[n];
        const int cap = a.max_blocks * kPage;
        L = l < 0 ? 0 : (l > cap ? cap : l);
        kvo = 0;
        hist = L - P;
    }
}

__device__ inline UnitInfo unit_info(const MfmaPrefillArgs& a, int u) {
    const int n = u / a.qblocks;
    const int qb = a.qblocks - 1 - (u % a.qblocks);
    UnitInfo r;
    seq_geom(a, n, r.q0, r.P, r.L, r.kvo, r.hist);
    const int q_lo = qb * BQ;
    if (q_lo >= r.P) {
        r.tiles = -1;   // no query rows: no work
        return r;
    }
    int kend = a.causal ? r.hist + min(q_lo + BQ, r.P) : r.L;
    kend = kend < 0 ? 0 : (kend > r.L ? r.L : kend);
    r.tiles = (kend + BN - 1) / BN;
    return r;
}

// The launch's items, from the actual lengths (up to kRankUnits units): the
// units that have query rows, where the launch has room for partials cut into
// equal chunks of at most `limit` tiles, and ranked by tiles per chunk
// (descending, ties by index).  Every work-group derives the same items from the
// same lengths; item y is the y-th chunk in that order.
//
// limit: no unit is cut unless the longest has cut_margin tiles more than a
// compute unit's share of the launch (sum of tiles x Hq / CUs): partials and merge
// cost that much (cut_margin(); cutting from the share on took 12/2/128 fp16 chunks of
// 2, 1062, 23, 309, 808, 4 and 1496 rows from 42.7 to 52.9 us).
// Otherwise the longest is cut into the fewest equal chunks of at most that share or
// kMinChunkTiles, the greater, and the others to the same size.  With one
// work-group per CU a second round waits for the first: there the limit is the
// first up to 7/4 of the share at which the items run in one round (761 fp32 rows
// on 1031, 16/8/256: 17 items per head 340 us, 16 items 277), or else 7/4 of it
// (16/8/256 fp16 chunks of 1 .. 1121 rows 102 us cut at the share, 76 uncut).
// The launched items and the partial slots bound the limit too: a cut unit of t
// tiles has ceil(t / limit) < t / limit + 1 chunks, at most 2 t / limit, so
// sum / limit <= extra items suffices, and for the slots either of
// 2 sum / limit <= slots and sum / limit <= slots - units.  (The first alone cut
// one unit of 54 tiles for 32/32/96 heads into four chunks of 14 where seven of 8
// run in 24 us instead of 29.)
//
// pick_item leaves in LDS each unit's lengths, so that the chosen unit costs no
// second global round trip; every thread of the work-group calls it (it contains
// barriers).
constexpr int kRankUnits = 1024;
constexpr int kMinChunkTiles = 8;
constexpr int kFitUnits = 256;   // units up to which a limit that fits one round is looked for (0.4 us per 64)
constexpr int kKeyTiles = (1 << 19) - 1;   // the ranking's key: 19 bits of tiles, 12 of chunks

struct Item {
    int unit, ci, chunks, part;   // part: partial slot of chunk 0 (chunks > 1)
};

// Sum over aligned groups of 8 lanes.
__device__ inline int group8_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, kDppQuadXor1, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, kDppQuadXor2, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, kDppRowHalfMirror, 0xF, 0xF, false);
    return v;
}

__device__ inline bool pick_item(const MfmaPrefillArgs& a, int y, int* lds, Item& it, UnitInfo& info) {
    __shared__ Item s_item;
    const int U = a.N * a.qblocks;
    if (U > kRankUnits) {   // index order, nothing cut
        if (y >= U) return false;
        it = Item{y, 0, 1, 0};
        info = unit_info(a, y);
        return info.tiles >= 0;
    }
    int* tiles = lds;
    int* key = lds + kRankUnits;   // tiles per chunk (at most kKeyTiles) << 12 | chunks; -1: no rows
    int* q0s = lds + 2 * kRankUnits;
    int* ps = lds + 3 * kRankUnits;
    int* ls = lds + 4 * kRankUnits;
    int* kvos = lds + 5 * kRankUnits;
    const bool cut = a.max_parts > 0;   // uniform
    const int U4 = (U + 3) & ~3;
    for (int u = threadIdx.x; u < U4; u += blockDim.x) {
        UnitInfo r;
        r.tiles = -1;
        if (u < U) {
            r = unit_info(a, u);
            q0s[u] = r.q0;
            ps[u] = r.P;
            ls[u] = r.L;
            kvos[u] = r.kvo;
        }
        tiles[u] = r.tiles;
        key[u] = r.tiles < 0 ? -1 : (min(r.tiles, kKeyTiles) << 12) | 1;
    }
    if (threadIdx.x == 0) s_item.unit = -1;
    __syncthreads();
    if (cut) {
        int sum = 0, longest = 0, units = 0;
        for (int v = threadIdx.x & 63; v < U; v += 64) {   // every wave for itself
            const int t = max(tiles[v], 0);
            sum += t;
            longest = max(longest, t);
            units += tiles[v] >= 0 ? 1 : 0;
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            sum += __shfl_xor(sum, off, 64);
            longest = max(longest, __shfl_xor(longest, off, 64));
            units += __shfl_xor(units, off, 64);
        }
        const int share = (int)(((int64_t)sum * a.Hq + a.n_cus - 1) / a.n_cus);
        if ((int64_t)(longest - a.cut_margin) * a.n_cus > (int64_t)sum * a.Hq) {   // uniform
            const bool one = a.resident < 2 * a.n_cus;
            const int per = one ? (7 * share + 3) / 4 : share;
            const int most = (longest + kMinChunkTiles - 1) / kMinChunkTiles;   // chunks of the longest
            const int k = min((longest + per - 1) / per, most);
            int limit = (longest + k - 1) / k;
            if (one && units * a.Hq <= a.resident && U <= kFitUnits) {   // a lane per limit
                const int l = max(share, (longest + most - 1) / most) + (threadIdx.x & 63);
                const float inv = 1.0f / l;
                int n = 0;
                for (int v = 0; v < U; ++v)
                    n += tiles[v] < 0 ? 0 : max(1, (int)((float)(tiles[v] + l - 1) * inv));
                const uint64_t fits = __builtin_amdgcn_ballot_w64(n * a.Hq <= a.resident && l <= per);
                if (fits != 0) limit = l - (int)(threadIdx.x & 63) + __builtin_ctzll(fits);
            }
            int by_slots = (2 * sum + a.max_parts - 1) / a.max_parts;
            const int spare = a.max_parts - units;
            if (spare > 0) by_slots = min(by_slots, (sum + spare - 1) / spare);
            limit = max(limit, max(by_slots, (sum + a.extra_items - 1) / a.extra_items));
            for (int u = threadIdx.x; u < U; u += blockDim.x) {
                const int t = tiles[u];
                if (t > limit) {
                    const int n = (t + limit - 1) / limit;
                    key[u] = min((t + n - 1) / n, kKeyTiles) << 12 | n;
                }
            }
        }
        __syncthreads();
    }
    // Eight lanes per unit, each over an eighth of the others.
    for (int u0 = 0; u0 < U; u0 += blockDim.x / 8) {
        const int u = u0 + threadIdx.x / 8;
        const int ku = u < U ? key[u] : -1;
        int before = 0, parts = 0;   // chunks of the units ranked before u; those of cut units
        for (int v = 4 * (threadIdx.x & 7); v < U4; v += 32) {
            const int4 kv = *reinterpret_cast<const int4*>(key + v);
            const int k4[4] = {kv.x, kv.y, kv.z, kv.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = (k4[e] > ku) | ((k4[e] == ku) & (v + e < u)) ? k4[e] & 4095 : 0;
                before += n;
                parts += n > 1 ? n : 0;
            }
        }
        before = group8_sum(before);
        parts = group8_sum(parts);
        if (u >= U || (threadIdx.x & 7) != 0) continue;
        const int n = ku < 0 ? 0 : ku & 4095;
        if (y >= before && y < before + n) s_item = Item{u, y - before, n, parts};
        if (cut && blockIdx.x == 0) a.table[u] = make_int2(parts, n);   // for the merge kernel
    }
    __syncthreads();
    // (the same for every lane: scalar registers)
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };
    it = Item{uniform(s_item.unit), uniform(s_item.ci), uniform(s_item.chunks), uniform(s_item.part)};
    if (it.unit < 0) return false;
    info.q0 = uniform(q0s[it.unit]);
    info.P = uniform(ps[it.unit]);
    info.L = uniform(ls[it.unit]);
    info.kvo = uniform(kvos[it.unit]);
    info.tiles = uniform(tiles[it.unit]);
    return true;
}

// Wave priority around the S = K Q^T cluster (s_setprio: issue arbitration
// among the waves of one SIMD, not a queue or stream priority): a wave in its
// matrix phase issues ahead of waves in their softmax.  Measured at head_dim
// 128 (configuration 5: 210 -> 201 us); neutral at head_dim 64, where it is
// off.  Raising the PV cluster as well gained nothing.
#define LLKV_PF_PRIO(on, p)                                \
    do {                                                   \
        if (on) {                                          \
            __builtin_amdgcn_sched_barrier(0);             \
            __builtin_amdgcn_s_setprio(p);                 \
            __builtin_amdgcn_sched_barrier(0);             \
        }                                                  \
    } while (0)

constexpr int kPageWindow = 256;   // page ids staged in LDS at a time

constexpr int kXcds = 8;   // XCDs of an MI355X; work-groups go to them round-robin


// One work-group's work item, from its blockIdx.
//
// Items (pick_item's order: longest first) times Hkv kv-head groups of G q
// heads, which read the same K/V tiles.  The dispatcher hands consecutive
// work-groups to the 8 XCDs in turn, and each XCD has its own L2, so group
// j (item-major) goes to XCD j % 8 with its G heads as that XCD's next G
// work-groups: they run together and share their K/V reads in one L2.
struct Work {
    int hq, kvh, n, ci, part, q0, P, q_lo, L, kvo, hist, kend, t_begin, t_end;
    bool direct;   // one chunk: write the output row itself
};

// False when the work-group has nothing to do (uniform over the work-group;
// it may return before or after the ranking barriers, never between).
__device__ inline bool take_work(const MfmaPrefillArgs& a, int* lds, Work& wk) {
    const int G = a.Hq / a.Hkv;
    // Work-groups b, b + CUs, b + 2 CUs of the first resident set share a CU.
    // When a CU holds two or more, the second set takes its items in reverse,
    // so that the CU holding the longest item of the first set gets the
    // shortest of the second, or none: a grid of more than one set has two whole
    // ones.  (With the reverse of a part of the second set the longest items got
    // the others beside them, and the CUs of the shortest none: 28/4/128 fp16
    // chunks of 1009, 11, 1 and 2 rows 30.4 -> 32.1 us.)
    int bid = blockIdx.x;
    if (a.resident >= 2 * a.n_cus && bid >= a.n_cus && bid < 2 * a.n_cus)
        bid = a.n_cus + (2 * a.n_cus - 1 - bid);
    const int xcd = bid % kXcds, r = bid / kXcds;
    const int j = (r / G) * kXcds + xcd;
    if (j >= a.groups) return false;
    wk.kvh = j % a.Hkv;
    wk.hq = wk.kvh * G + r % G;
    Item it;
    UnitInfo ui;
    if (!pick_item(a, j / a.Hkv, lds, it, ui)) return false;
    wk.n = it.unit / a.qblocks;
    const int qb = a.qblocks - 1 - (it.unit % a.qblocks);
    wk.q0 = ui.q0;
    wk.P = ui.P;
    wk.q_lo = qb * BQ;
    wk.L = ui.L;
    wk.kvo = ui.kvo;
    wk.hist = a.contig ? 0 : ui.L - ui.P;   // as seq_geom (not kept with the ranked units)
    int kend = a.causal ? wk.hist + min(wk.q_lo + BQ, wk.P) : wk.L;
    wk.kend = kend < 0 ? 0 : (kend > wk.L ? wk.L : kend);
    // equal chunks; a unit of no tiles has one, which writes zeros
    const int per = (ui.tiles + it.chunks - 1) / it.chunks;
    wk.ci = it.ci;
    wk.part = it.part + it.ci;
    wk.t_begin = min(it.ci * per, ui.tiles);
    wk.t_end = min(wk.t_begin + per, ui.tiles);
    wk.direct = it.chunks == 1;
    return true;
}

// Query rows beyond the launch's qblocks * BQ (a max_q_len bound below a
// sequence's query count) have no work-group: the top query block's chunk-0
// work-group sets them to NaN for its head, so the broken bound shows in the
// output instead of leaving stale rows.
template <typename T, int D>
__device__ inline void poison_uncovered_rows(const MfmaPrefillArgs& a, const Work& wk) {
    const int covered = a.qblocks * BQ;
    if (wk.ci != 0 || wk.q_lo != covered - BQ || wk.P <= covered) return;
    T* og = reinterpret_cast<T*>(a.out);
    const int n = (wk.P - covered) * D;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int r = covered + i / D;
        og[((int64_t)(wk.q0 + r) * a.Hq + wk.hq) * D + i % D] = Elem<T>::from_f32(__builtin_nanf(""));
    }
}

// Direct-to-LDS load of 16 bytes per lane: lane L's bytes land at LDS address
// lds + 16 L (lds uniform over the wave).  Issued as inline assembly, so that
// the compiler, which cannot tell the two tile buffers apart, does not wait for
// it before every LDS read of the other buffer; the caller waits (vmcnt) before
// the barrier that publishes the tile.  A later load only lengthens the
// compiler's own in-order vmcnt waits.
// la: the LDS byte address (lds_addr), wave-uniform.
__device__ inline uint32_t lds_addr(const void* lds) {
    return __builtin_amdgcn_readfirstlane(
        (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)lds);
}

__device__ inline void dma16(const void* gptr, uint32_t la) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(gptr), "s"(la)
                 : "memory", "m0");
}

// The same with a wave-uniform base (scalar registers) and a 32-bit per-lane
// byte offset (no per-lane 64-bit address arithmetic).
__device__ inline void dma16_s(const void* sbase, uint32_t voff, uint32_t la) {
    const uint64_t b = (uint64_t)(uintptr_t)sbase;
    // (readfirstlane returns int: widen through uint32_t, not by sign extension)
    const uint64_t bs = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) |
                        (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
                 :
                 : "v"(voff), "s"(bs), "s"(la)
                 : "memory", "m0");
}

// Instruction order of the S^T = K Q^T cluster (KS k-steps of 4 K operand
// reads and 8 MFMAs): the reads of k-steps 0 and 1, then each k-step's MFMAs
// followed by the reads of the k-step after next, so that one k-step's LDS
// reads are always in flight behind the MFMAs.
template <int KS, int I = 0>
__device__ inline void qk_schedule() {
    if constexpr (I == 0) __builtin_amdgcn_sched_group_barrier(0x100, KS > 1 ? 8 : 4, 0);   // DS reads
    if constexpr (I < KS) {
        __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);                                 // MFMAs
        if constexpr (I + 2 < KS) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        qk_schedule<KS, I + 1>();
    }
}

// K and V tiles are row-major (key rows of D halves, KPAD apart); V's O^T
// operand is read with transposing LDS reads.  DMA: the tiles are written by
// direct-to-LDS loads in 1 KB blocks, so rows are unpadded and their 16-byte
// chunks XOR-swizzled by row instead.
template <int D, bool DMA>
struct Smem {
    static constexpr int KPAD = DMA ? D : D + 8;   // halves per K / V row (pad: spread LDS banks)
    union {
        struct {
            alignas(16) uint16_t k[2][BN * KPAD];
            alignas(16) uint16_t v[2][BN * KPAD];
        };
        int order[6 * kRankUnits];   // prologue only: unit tiles, ranking keys, q0, P, L, K/V offset
    };
    int pages[kPageWindow];   // page ids [tbase, tbase + kPageWindow) of the sequence
};

// CG: contiguous K/V (first prefill): key j of the sequence is row kvo + j of
// k / v; the staged rows are clamped to the sequence's last, and there is no
// page table.
// head_dim 128: two waves per SIMD (<= 256 registers).
template <typename T, int D, bool CG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 128 ? 2 : 1)))
void prefill_mfma_kernel(MfmaPrefillArgs a) {
    // Direct-to-LDS staging (head_dim 64 / 128): wave w loads page w of the
    // tile (rows 16w .. 16w + 15) of K and of V, RPB rows per 1 KB block.
    constexpr bool kDma = D == 64 || D == 128;
    using SM = Smem<D, kDma>;
    constexpr int KPAD = SM::KPAD;
    constexpr int CPR = D / 8;            // 16-byte chunks per row
    constexpr int RPB = 64 / CPR;         // rows per 1 KB block
    constexpr int BPW = 16 / RPB;         // blocks per wave (one page) per tile
    // Chunk swizzle of tile row r: row bits 0, 1, 3, 4 (the QK^T operand reads
    // rows 8 (c16 / 4) + 4 h + c16 % 4 together, so rows 8 apart must differ).
    auto swz_row = [](int r) { return ((r & 3) | ((r >> 1) & 0xC)) & (CPR - 1); };
    constexpr int KS = D / 32;            // k-steps of the QK^T product
    constexpr int DT = D / 16;            // 16-dim tiles of the output
    constexpr int KCH = BN * D / 8;       // 16-byte K chunks per tile
    constexpr int KCH_T = KCH / 256;      // per thread
    __shared__ SM sm;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave index, known uniform
    const int g = lane >> 4, c16 = lane & 15;
    Work wk;
    if (!take_work(a, sm.order, wk)) return;
    // The ranking's arrays overlay the tile buffers.  Paged launches pass an
    // LDS barrier (stage_pages) before the first tile is written; contiguous
    // K/V has no page window, so every wave's reads of its unit from the
    // ranking must complete here before any wave writes the first tile.
    if constexpr (CG) lds_barrier();
    poison_uncovered_rows<T, D>(a, wk);
    const int hq = wk.hq, kvh = wk.kvh, n = wk.n;
    const int q0 = wk.q0, P = wk.P, q_lo = wk.q_lo, L = wk.L, kend = wk.kend;
    const int t_begin = wk.t_begin, t_end = wk.t_end;
    const bool direct = wk.direct;
    const int last_page = L > 0 ? (L - 1) / kPage : 0;
    const int* bt = a.bt + (int64_t)n * a.max_blocks;
    const T* kg = reinterpret_cast<const T*>(a.k) + (int64_t)kvh * D + (CG ? (int64_t)wk.kvo : 0);
    const T* vg = reinterpret_cast<const T*>(a.v) + (int64_t)kvh * D + (CG ? (int64_t)wk.kvo : 0);

    // ---- Q^T operands (B of S^T = K Q^T), kept in registers; loaded after the
    // page ids so that their latency overlaps the first tile's ------------
    uint4 qop[2][KS];
    const T* qg = reinterpret_cast<const T*>(a.q);
    auto load_q = [&]() {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const int ql = q_lo + w * WQ + nt * 16 + c16;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                if (ql < P)
                    qop[nt][ks] = *reinterpret_cast<const uint4*>(
                        qg + ((int64_t)(q0 + ql) * a.Hq + hq) * D + ks * 32 + g * 8);
                else
                    qop[nt][ks] = make_uint4(0, 0, 0, 0);
            }
        }
    };

    // Absolute position of this lane's two query columns; rows >= P see nothing.
    int qpos[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int ql = q_lo + w * WQ + nt * 16 + c16;
        qpos[nt] = ql < P ? (a.causal ? wk.hist + ql : L - 1) : -1;
    }

    // Smallest query position of the wave's 32 rows (every row valid), for the
    // unmasked fast path of tiles that lie entirely below it.
    const int wq0 = q_lo + w * WQ;
    const int wave_min_pos = (wq0 + WQ <= P) ? (a.causal ? wk.hist + wq0 : L - 1) : -1;

    f32x4 o[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) o[dt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m[2] = {kNegBig, kNegBig};
    // Row sums of P on the MFMA: O^T's extra tile with an all-ones A operand;
    // every element of osum[nt] is the running sum of query column c16.
    f32x4 osum[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    const uint4 ones = make_uint4(Mfma<T>::kOnes, Mfma<T>::kOnes, Mfma<T>::kOnes, Mfma<T>::kOnes);

    // ---- staging: global -> registers -> LDS -----------------------------
    int tbase = 0;   // first page id held in sm.pages
    // V is staged like K (row-major, the same row offsets and page addresses).
    u32x4 kr[KCH_T], vr[KCH_T];
    static_assert(KCH % 256 == 0, "K / V chunks spread evenly over the threads");
    // Per-thread byte offsets inside a page and page slot of each staged row;
    // a load is then base + phys * page_bytes + offset (one 32x32->64 multiply-add).
    // Contiguous K/V: the key within the tile and the byte offset in the row.
    const uint32_t row_bytes = (uint32_t)(a.Hkv * D * sizeof(T));
    const uint32_t page_bytes = row_bytes * kPage;
    const char* kb = reinterpret_cast<const char*>(kg);
    const char* vb = reinterpret_cast<const char*>(vg);
    uint32_t koff[KCH_T];
    int kslot[KCH_T];
#pragma unroll
    for (int j = 0; j < KCH_T; ++j) {
        const int ch = tid + 256 * j;
        const int key = ch / (D / 8), c = ch % (D / 8);
        kslot[j] = CG ? key : key >> 4;
        koff[j] = (CG ? 0u : (uint32_t)(key & 15) * row_bytes) + (uint32_t)c * 16u;
    }
    auto load_tile = [&](int t, u32x4 (&kreg)[KCH_T], u32x4 (&vreg)[KCH_T]) {
        if constexpr (CG) {   // rows past the sequence's last are staged as the last
            const int key0 = t * BN, last = L - 1;
#pragma unroll
            for (int j = 0; j < KCH_T; ++j) {
                const uint64_t off = (uint64_t)min(key0 + kslot[j], last) * row_bytes + koff[j];
                kreg[j] = *reinterpret_cast<const u32x4*>(kb + off);
                vreg[j] = *reinterpret_cast<const u32x4*>(vb + off);
            }
            return;
        }
        // pages past the sequence's last are staged as the last page (valid memory)
        const int* pg = sm.pages + (4 * t - tbase);
#pragma unroll
        for (int j = 0; j < KCH_T; ++j) {
            const uint64_t off = (uint64_t)(uint32_t)max(pg[kslot[j]], 0) * page_bytes + koff[j];
            kreg[j] = *reinterpret_cast<const u32x4*>(kb + off);
            vreg[j] = *reinterpret_cast<const u32x4*>(vb + off);
        }
    };
    auto store_tile = [&](int buf, const u32x4 (&kreg)[KCH_T], const u32x4 (&vreg)[KCH_T]) {
#pragma unroll
        for (int j = 0; j < KCH_T; ++j) {
            const int ch = tid + 256 * j;
            const int key = ch / (D / 8), c = ch % (D / 8);
            *reinterpret_cast<u32x4*>(&sm.k[buf][key * KPAD + c * 8]) = kreg[j];
            *reinterpret_cast<u32x4*>(&sm.v[buf][key * KPAD + c * 8]) = vreg[j];
        }
    };
    // Half-column hc of tile row `row` in LDS: with DMA the 16-byte chunk
    // index is XOR-ed with the row (mod the chunks per row).
    auto scol = [&](int row, int hc) {
        if constexpr (kDma) return (((hc >> 3) ^ swz_row(row)) << 3) | (hc & 7);
        return hc;
    };
    // A operand of O^T = V^T P^T for output dims dt*16 .. +15 and the 32-key
    // half ss: lane (g, c16) holds dim dt*16 + c16 of keys 32 ss + 8 g .. + 7.
    // ds_read_b64_tr_b16 within each 16-lane group: output lane 4a + e gets
    // element e of the 4 halves addressed by lanes a, a + 4, a + 8, a + 12; so
    // lane c16 addresses row (key) c16 / 4, dims 4 (c16 % 4) .. + 3, and each
    // lane receives its dim over 4 consecutive keys (two reads: 8 keys).
    auto v_operand = [&](int buf, int dt, int ss) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        const int r0 = 32 * ss + 8 * g + (c16 >> 2), hc = dt * 16 + 4 * (c16 & 3);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(&sm.v[buf][r0 * KPAD + scol(r0, hc)]));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(&sm.v[buf][(r0 + 4) * KPAD + scol(r0 + 4, hc)]));
        typedef unsigned u32x2v __attribute__((ext_vector_type(2)));
        const u32x2v l2 = __builtin_bit_cast(u32x2v, lo), h2 = __builtin_bit_cast(u32x2v, hi);
        return make_uint4(l2.x, l2.y, h2.x, h2.y);
    };

    // Page ids live in LDS so that no K/V load waits behind a table load.
    auto stage_pages = [&](int base) {
        if constexpr (CG) return;   // no page table
        tbase = base;
        for (int i = tid; i < kPageWindow; i += 256) sm.pages[i] = bt[min(base + i, last_page)];
        lds_barrier();   // the page ids are in LDS; no global load needs to have landed
    };
    // Direct-to-LDS: lane L of block j writes LDS chunk L of rows 16w + j RPB ..,
    // i.e. row 16w + j RPB + L / CPR, chunk position L % CPR, which holds the
    // row's global chunk (L % CPR) ^ swz_row(row).
    uint32_t dma_off[BPW];   // byte offset of the lane's chunk inside its page (paged) / row (CG)
    int dma_row[BPW];        // the lane's row within the wave's page
#pragma unroll
    for (int j = 0; j < BPW; ++j) {
        const int r = j * RPB + lane / CPR;
        const int c = (lane % CPR) ^ swz_row(16 * w + r);
        dma_row[j] = r;
        dma_off[j] = (CG ? 0u : (uint32_t)r * row_bytes) + (uint32_t)c * 16u;
    }
    // LDS byte addresses of the wave's blocks in each buffer, computed once
    // (scalar registers; the loop then only moves them to M0).
    uint32_t lds_k[2][BPW], lds_v[2][BPW];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int j = 0; j < BPW; ++j) {
            const int lrow = 16 * w + j * RPB;
            lds_k[b][j] = lds_addr(&sm.k[b][lrow * KPAD]);
            lds_v[b][j] = lds_addr(&sm.v[b][lrow * KPAD]);
        }
    auto dma_tile = [&](int t, int buf) {
        if constexpr (kDma) {
            if constexpr (CG) {
#pragma unroll
                for (int j = 0; j < BPW; ++j) {   // rows past the sequence's last are staged as the last
                    const int key = min(t * BN + 16 * w + dma_row[j], L - 1);
                    const uint64_t off = (uint64_t)key * row_bytes + dma_off[j];
                    dma16(kb + off, lds_k[buf][j]);
                    dma16(vb + off, lds_v[buf][j]);
                }
            } else {
                // the wave's page: one scalar base per pool, 32-bit lane offsets
                const int phys = __builtin_amdgcn_readfirstlane(max(sm.pages[4 * t + w - tbase], 0));
                const uint64_t pbase = (uint64_t)(uint32_t)phys * page_bytes;
#pragma unroll
                for (int j = 0; j < BPW; ++j) {
                    dma16_s(kb + pbase, dma_off[j], lds_k[buf][j]);
                    dma16_s(vb + pbase, dma_off[j], lds_v[buf][j]);
                }
            }
        }
    };
    if (t_begin < t_end) {
        stage_pages(4 * t_begin);
        load_q();
        if constexpr (kDma) {
            dma_tile(t_begin, 0);
            __builtin_amdgcn_s_waitcnt(0x3F70);   // vmcnt(0): this wave's blocks are in LDS
        } else {
            load_tile(t_begin, kr, vr);
            store_tile(0, kr, vr);
        }
    }
    __syncthreads();

    // One key tile; buf = (t - t_begin) & 1.  The loop below runs it twice per
    // trip with buf as a compile-time constant, so the LDS addresses of both
    // buffers fold into the instructions' offsets.
    auto tile_step = [&](int t, auto bufc) {
        const int buf = static_cast<int>(bufc);
        if (t + 1 < t_end) {
            // tile t+1 covers pages [4(t+1), 4(t+1)+4); restage when they leave the window
            // (uniform branch; every earlier read of sm.pages preceded the last barrier)
            if (4 * (t + 1) + 4 > tbase + kPageWindow) stage_pages(4 * (t + 1));
            if constexpr (kDma) dma_tile(t + 1, buf ^ 1);
            else load_tile(t + 1, kr, vr);
        }
        __builtin_amdgcn_sched_barrier(0);   // next tile's loads issue before this tile's MFMAs
        LLKV_PF_PRIO(D >= 128, 1);

        // ---- S^T = K Q^T over the 64 keys: 4 key tiles x 2 query tiles ----
        // k-step outer: the 8 (key tile, query tile) chains advance together,
        // and the K operands of k-step ks + 1 are read while those of ks feed
        // the matrix core.
        f32x4 s[4][2];
        auto k_operand = [&](int kt, int ks) {
            // A row c16 of key tile kt = 2*ss + h holds key 32*ss + 8*(c16/4) + 4*h + c16%4
            const int krow = 32 * (kt >> 1) + 8 * (c16 >> 2) + 4 * (kt & 1) + (c16 & 3);
            return *reinterpret_cast<const uint4*>(&sm.k[buf][krow * KPAD + scol(krow, ks * 32 + g * 8)]);
        };
        uint4 ka[2][4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) ka[0][kt] = k_operand(kt, 0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            if (ks + 1 < KS) {
#pragma unroll
                for (int kt = 0; kt < 4; ++kt) ka[(ks + 1) & 1][kt] = k_operand(kt, ks + 1);
            }
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
                    s[kt][nt] = Mfma<T>::mma(ka[ks & 1][kt], qop[nt][ks],
                                             ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[kt][nt]);
        }
        if constexpr (kDma) qk_schedule<KS>();

        LLKV_PF_PRIO(D >= 128, 0);
        // ---- mask, online softmax (per query column) ----------------------
        // Scores stay raw (unscaled) until the exponent: p = 2^(s c - m) with
        // c = scale * log2(e) > 0, so the row maximum commutes with the scaling.
        const int key0 = t * BN;
        const float c = a.scale_log2;
        // Every key of the tile visible to every row of the wave (uniform): no mask.
        const bool unmasked = key0 + BN - 1 <= wave_min_pos && key0 + BN <= kend;
        float mx[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            if (!unmasked) {
                // key = key0 + 8g + (32 ss + 4 h + i) is visible iff key <= min(qpos, kend - 1)
                const int r = min(qpos[nt], kend - 1) - key0 - 8 * g;
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (32 * (kt >> 1) + 4 * (kt & 1) + i > r) s[kt][nt][i] = -INFINITY;
            }
            float v = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) v = fmaxf(v, s[kt][nt][i]);
            mx[nt] = v * c;   // this lane's 16 keys only
        }
        // Lazy rescaling: the running max m only moves when some lane's tile
        // max exceeds it by more than 8 (so p <= 2^8 otherwise); then the wave
        // reduces the row maxima over the 4 lanes of each query column and
        // rescales its accumulators once.  Usually only the first tile does, so
        // the common path has no cross-lane traffic.
        bool grow = false;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) grow |= mx[nt] > m[nt] + 8.0f;
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                float v = mx[nt];
                v = fmaxf(v, __shfl_xor(v, 16, 64));
                v = fmaxf(v, __shfl_xor(v, 32, 64));
                const float mnew = fmaxf(m[nt], v);
                const float corr = fast_exp2(m[nt] - mnew);
                m[nt] = mnew;
                osum[nt] *= corr;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[dt][nt] *= corr;
            }
        }
        // ---- P = 2^(S c - m) and O^T += V^T P^T, one 32-key half after the
        // other: the second half's exponentials are interleaved with the first
        // half's MFMAs, so that the VALU and the matrix core work together.
        uint4 pop[2][2];   // P^T operands [k-step = key half][query tile]
        auto softmax_half = [&](int ss) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                float pv[2][4];
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        pv[h][i] = fast_exp2(fmaf(s[2 * ss + h][nt][i], c, -m[nt]));
                pop[ss][nt].x = Mfma<T>::pack2(pv[0][0], pv[0][1]);
                pop[ss][nt].y = Mfma<T>::pack2(pv[0][2], pv[0][3]);
                pop[ss][nt].z = Mfma<T>::pack2(pv[1][0], pv[1][1]);
                pop[ss][nt].w = Mfma<T>::pack2(pv[1][2], pv[1][3]);
            }
        };
        // The first half's MFMAs, each followed by a share of the second half's
        // exponentials; sched_barrier keeps this order (the scheduler would
        // otherwise put all VALU work first).  V^T rows of the second half are
        // read as those of the first are consumed.
        softmax_half(0);
        {
            constexpr int kMf = 2 * DT + 2;   // MFMAs per half
            uint4 va0[DT], va1[DT];
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                va0[dt] = v_operand(buf, dt, 0);
            float pv1[2][2][4];   // [query tile][h][i] of the second half
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < kMf; ++k) {
                if (k < 2 * DT) {
                    const int dt = k >> 1, nt = k & 1;
                    o[dt][nt] = Mfma<T>::mma(va0[dt], pop[0][nt], o[dt][nt]);
                    if (nt == 1)
                        va1[dt] = v_operand(buf, dt, 1);
                } else {
                    const int nt = k - 2 * DT;
                    osum[nt] = Mfma<T>::mma(ones, pop[0][nt], osum[nt]);
                }
#pragma unroll
                for (int e = k * 16 / kMf; e < (k + 1) * 16 / kMf; ++e) {
                    const int nt = e >> 3, h = (e >> 2) & 1, i = e & 3;
                    pv1[nt][h][i] = fast_exp2(fmaf(s[2 + h][nt][i], c, -m[nt]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                pop[1][nt].x = Mfma<T>::pack2(pv1[nt][0][0], pv1[nt][0][1]);
                pop[1][nt].y = Mfma<T>::pack2(pv1[nt][0][2], pv1[nt][0][3]);
                pop[1][nt].z = Mfma<T>::pack2(pv1[nt][1][0], pv1[nt][1][1]);
                pop[1][nt].w = Mfma<T>::pack2(pv1[nt][1][2], pv1[nt][1][3]);
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) o[dt][nt] = Mfma<T>::mma(va1[dt], pop[1][nt], o[dt][nt]);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) osum[nt] = Mfma<T>::mma(ones, pop[1][nt], osum[nt]);
        }

        if constexpr (kDma) {
            if (t + 1 < t_end) __builtin_amdgcn_s_waitcnt(0x3F70);   // vmcnt(0): tile t+1 in LDS
        } else {
            if (t + 1 < t_end) store_tile(buf ^ 1, kr, vr);
        }
        __syncthreads();
    };
    {
        int t = t_begin;
        for (; t + 1 < t_end; t += 2) {
            tile_step(t, std::integral_constant<int, 0>());
            tile_step(t + 1, std::integral_constant<int, 1>());
        }
        if (t < t_end) tile_step(t, std::integral_constant<int, 0>());
    }

    // ---- normalise and write: lane holds dims dt*16 + 4g + i of its query --
    // (one chunk: the output row; several: an fp32 partial row + log2-sum-exp2,
    // -inf for a row that saw no key of this chunk)
    T* og = reinterpret_cast<T*>(a.out);
    const int64_t pidx = (int64_t)wk.part * a.Hq + hq;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const float lt = osum[nt][0];
        const int row = w * WQ + nt * 16 + c16;
        const int ql = q_lo + row;
        if (ql >= P) continue;
        const float inv = lt > 0.f ? 1.0f / lt : 0.f;
        if (direct) {
            T* orow = og + ((int64_t)(q0 + ql) * a.Hq + hq) * D;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                uint2 w2;
                w2.x = Mfma<T>::pack2(o[dt][nt][0] * inv, o[dt][nt][1] * inv);
                w2.y = Mfma<T>::pack2(o[dt][nt][2] * inv, o[dt][nt][3] * inv);
                *reinterpret_cast<uint2*>(orow + dt * 16 + 4 * g) = w2;
            }
        } else {
            float* prow = a.part_o + (pidx * BQ + row) * D;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                *reinterpret_cast<float4*>(prow + dt * 16 + 4 * g) =
                    make_float4(o[dt][nt][0] * inv, o[dt][nt][1] * inv, o[dt][nt][2] * inv,
                                o[dt][nt][3] * inv);
            if (g == 0) a.part_lse[pidx * BQ + row] = lt > 0.f ? m[nt] + fast_log2(lt) : -INFINITY;
        }
    }
}

// fp32 pools: v_mfma_f32_16x16x4f32 for both products, same work mapping,
// chunking and merge as the 16-bit kernel.  Per wave and 64-key tile:
//   S^T = K Q^T   A = K rows from LDS, one 16-byte read feeds four k-steps:
//                 lane (g, c16) holds dims 16kb + 4g .. 16kb + 4g + 3 of key
//                 row c16, and Q^T (registers) holds the same dims of query
//                 c16, so k-step j of block kb contracts dim 16kb + 4g + j.
//                 Accumulator lane (g, c16) holds keys 4g + i of query c16.
//   O^T = V^T P^T the lane's four keys 4g + i of a 16-key tile are exactly the
//                 k-slot g of four k-steps (i = 0..3), so P^T never leaves
//                 registers; A = V^T (transposed while staging) read 16 bytes
//                 (keys 4g .. 4g + 3 of one dim) per four k-steps.
// Softmax row sums are kept per lane (its own keys) and reduced over the four
// lanes of a query column at the end.
// Instantiated for head_dim 256 alone: the smaller head dims run faster on
// prefill_f32_split_kernel, whose two tiles of two planes would take 128 KB of
// LDS here and its operands more registers than a wave has.  One work-group per
// CU, single-buffered tiles (134 KB).
// The S = K Q^T cluster runs at raised wave priority (as in the 16-bit kernel).
template <int D>
struct SmemF32 {
    static constexpr int KPAD = D + 4;    // floats per K row (pad: 16-byte reads of 16 rows hit distinct banks)
    static constexpr int VPAD = BN + 4;   // floats per V^T row
    union {
        struct {
            alignas(16) float k[BN * KPAD];
            alignas(16) float vt[D * VPAD];
        };
        int order[6 * kRankUnits];
    };
    int pages[kPageWindow];
};

template <int D, bool CG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1)))
void prefill_f32_kernel(MfmaPrefillArgs a) {
    typedef SmemF32<D> S;
    constexpr int KPAD = S::KPAD, VPAD = S::VPAD;
    constexpr int KB = D / 16;              // 16-dim blocks of the QK^T product
    constexpr int DT = D / 16;              // 16-dim tiles of the output
    constexpr int KCH_T = BN * D / 4 / 256;          // 16-byte K chunks per thread
    constexpr int VT_N = (BN / 4) * (D / 4);           // V tasks (4 keys x 4 dims) per tile
    constexpr int VT_T = VT_N / 256;                   // per thread
    static_assert(VT_N % 256 == 0, "V tasks spread evenly over the threads");
    __shared__ S sm;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c16 = lane & 15;
    Work wk;
    if (!take_work(a, sm.order, wk)) return;
    // The ranking's arrays overlay the tile buffers.  Paged launches pass an
    // LDS barrier (stage_pages) before the first tile is written; contiguous
    // K/V has no page window, so every wave's reads of its unit from the
    // ranking must complete here before any wave writes the first tile.
    if constexpr (CG) lds_barrier();
    poison_uncovered_rows<float, D>(a, wk);
    const int hq = wk.hq, kvh = wk.kvh, n = wk.n;
    const int q0 = wk.q0, P = wk.P, q_lo = wk.q_lo, L = wk.L, kend = wk.kend;
    const int t_begin = wk.t_begin, t_end = wk.t_end;
    const int last_page = L > 0 ? (L - 1) / kPage : 0;
    const int* bt = a.bt + (int64_t)n * a.max_blocks;

    float4 qop[2][KB];
    const float* qg = reinterpret_cast<const float*>(a.q);
    auto load_q = [&]() {
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const int ql = q_lo + w * WQ + nt * 16 + c16;
#pragma unroll
            for (int kb = 0; kb < KB; ++kb)
                qop[nt][kb] = ql < P ? *reinterpret_cast<const float4*>(
                                           qg + ((int64_t)(q0 + ql) * a.Hq + hq) * D + kb * 16 + g * 4)
                                     : make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };
    int qpos[2];
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        const int ql = q_lo + w * WQ + nt * 16 + c16;
        qpos[nt] = ql < P ? (a.causal ? wk.hist + ql : L - 1) : -1;
    }
    const int wq0 = q_lo + w * WQ;
    const int wave_min_pos = (wq0 + WQ <= P) ? (a.causal ? wk.hist + wq0 : L - 1) : -1;

    f32x4 o[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) o[dt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m[2] = {kNegBig, kNegBig};
    float lsum[2] = {0.f, 0.f};   // this lane's keys only

    int tbase = 0;
    u32x4 kr[KCH_T];
    u32x4 vr[VT_T][4];
    const uint32_t row_bytes = (uint32_t)(a.Hkv * D * sizeof(float));
    const uint32_t page_bytes = row_bytes * kPage;
    const int64_t kv0 = (int64_t)kvh * D + (CG ? (int64_t)wk.kvo : 0);
    const char* kb_ = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.k) + kv0);
    const char* vb_ = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.v) + kv0);
    uint32_t koff[KCH_T], voff[VT_T];
    int kslot[KCH_T], vslot[VT_T];
#pragma unroll
    for (int j = 0; j < KCH_T; ++j) {
        const int ch = tid + 256 * j;
        const int key = ch / (D / 4), c = ch % (D / 4);
        kslot[j] = CG ? key : key >> 4;   // contiguous K/V: the key within the tile
        koff[j] = (CG ? 0u : (uint32_t)(key & 15) * row_bytes) + (uint32_t)c * 16u;
    }
#pragma unroll
    for (int j = 0; j < VT_T; ++j) {
        const int task = tid + 256 * j;
        const int kq = task % (BN / 4), c = task / (BN / 4);   // keys 4kq .. 4kq+3, dims 4c .. 4c+3
        vslot[j] = CG ? 4 * kq : (4 * kq) >> 4;
        voff[j] = (CG ? 0u : (uint32_t)((4 * kq) & 15) * row_bytes) + (uint32_t)c * 16u;
    }
    // Next-tile staging in two halves (K, then V^T), so that only one half's
    // registers are live at a time.
    auto load_k = [&](int t) {
        if constexpr (CG) {   // rows past the sequence's last are staged as the last
#pragma unroll
            for (int j = 0; j < KCH_T; ++j)
                kr[j] = *reinterpret_cast<const u32x4*>(
                    kb_ + (uint64_t)min(t * BN + kslot[j], L - 1) * row_bytes + koff[j]);
            return;
        }
        const int* pg = sm.pages + (4 * t - tbase);
#pragma unroll
        for (int j = 0; j < KCH_T; ++j) {
            const uint64_t phys = (uint32_t)max(pg[kslot[j]], 0);
            kr[j] = *reinterpret_cast<const u32x4*>(kb_ + phys * page_bytes + koff[j]);
        }
    };
    auto load_v = [&](int t) {
        if constexpr (CG) {
#pragma unroll
            for (int j = 0; j < VT_T; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    vr[j][r] = *reinterpret_cast<const u32x4*>(
                        vb_ + (uint64_t)min(t * BN + vslot[j] + r, L - 1) * row_bytes + voff[j]);
            return;
        }
        const int* pg = sm.pages + (4 * t - tbase);
#pragma unroll
        for (int j = 0; j < VT_T; ++j) {
            const uint64_t phys = (uint32_t)max(pg[vslot[j]], 0);
            const char* p = vb_ + phys * page_bytes + voff[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) vr[j][r] = *reinterpret_cast<const u32x4*>(p + r * row_bytes);
        }
    };
    auto store_k = [&]() {
#pragma unroll
        for (int j = 0; j < KCH_T; ++j) {
            const int ch = tid + 256 * j;
            const int key = ch / (D / 4), c = ch % (D / 4);
            *reinterpret_cast<u32x4*>(&sm.k[key * KPAD + c * 4]) = kr[j];
        }
    };
    auto store_v = [&]() {
#pragma unroll
        for (int j = 0; j < VT_T; ++j) {
            const int task = tid + 256 * j;
            const int kq = task % (BN / 4), c = task / (BN / 4);
#pragma unroll
            for (int e = 0; e < 4; ++e)   // 4x4 transpose: V^T row 4c + e, keys 4kq .. 4kq+3
                *reinterpret_cast<u32x4*>(&sm.vt[(4 * c + e) * VPAD + 4 * kq]) =
                    u32x4{vr[j][0][e], vr[j][1][e], vr[j][2][e], vr[j][3][e]};
        }
    };
    auto stage_pages = [&](int base) {
        if constexpr (CG) return;   // no page table
        tbase = base;
        for (int i = tid; i < kPageWindow; i += 256) sm.pages[i] = bt[min(base + i, last_page)];
        lds_barrier();
    };
    if (t_begin < t_end) {
        stage_pages(4 * t_begin);
        load_q();
        load_k(t_begin);
        load_v(t_begin);
        store_k();
        store_v();
    }
    __syncthreads();

    for (int t = t_begin; t < t_end; ++t) {
        const bool next = t + 1 < t_end;   // uniform
        if (next) {
            if (4 * (t + 1) + 4 > tbase + kPageWindow) stage_pages(4 * (t + 1));
            load_k(t + 1);
        }
        __builtin_amdgcn_sched_barrier(0);

        LLKV_PF_PRIO(true, 1);
        // ---- S^T = K Q^T: key tile kt holds keys 16kt .. 16kt+15 ---------
        // The two halves of the head dims accumulate apart and are added at
        // the end: half the rounding steps in each sum, which halves the
        // score's rounding error (it dominates the fp32 output's error).
        f32x4 s[4][2];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            f32x4 hi[2];
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                s[kt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
                hi[nt] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const float4 ka = *reinterpret_cast<const float4*>(
                    &sm.k[(16 * kt + c16) * KPAD + kb * 16 + g * 4]);
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) {
                    f32x4& acc = kb < KB / 2 ? s[kt][nt] : hi[nt];
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.x, qop[nt][kb].x, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.y, qop[nt][kb].y, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.z, qop[nt][kb].z, acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(ka.w, qop[nt][kb].w, acc, 0, 0, 0);
                }
            }
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) s[kt][nt] += hi[nt];
        }
        LLKV_PF_PRIO(true, 0);
        if (next) {
            __syncthreads();   // every wave is done with the K buffer
            store_k();
            load_v(t + 1);
        }

        // ---- mask and online softmax (scores scaled in the exponent) -----
        const int key0 = t * BN;
        const float c = a.scale_log2;
        const bool unmasked = key0 + BN - 1 <= wave_min_pos && key0 + BN <= kend;
        float mx[2];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            if (!unmasked) {
                // key = key0 + 16kt + 4g + i is visible iff key <= min(qpos, kend - 1)
                const int r = min(qpos[nt], kend - 1) - key0 - 4 * g;
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        if (16 * kt + i > r) s[kt][nt][i] = -INFINITY;
            }
            float v = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) v = fmaxf(v, s[kt][nt][i]);
            mx[nt] = v * c;
        }
        bool grow = false;
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) grow |= mx[nt] > m[nt] + 8.0f;
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                float v = mx[nt];
                v = fmaxf(v, __shfl_xor(v, 16, 64));
                v = fmaxf(v, __shfl_xor(v, 32, 64));
                const float mnew = fmaxf(m[nt], v);
                const float corr = fast_exp2(m[nt] - mnew);
                m[nt] = mnew;
                lsum[nt] *= corr;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) o[dt][nt] *= corr;
            }
        }
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = fast_exp2(fmaf(s[kt][nt][i], c, -m[nt]));
                    s[kt][nt][i] = p;
                    lsum[nt] += p;
                }

        // ---- O^T += V^T P^T ------------------------------------------------
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) {
                const float4 va = *reinterpret_cast<const float4*>(
                    &sm.vt[(dt * 16 + c16) * VPAD + 16 * kt + 4 * g]);
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) {
                    o[dt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(va.x, s[kt][nt][0], o[dt][nt], 0, 0, 0);
                    o[dt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(va.y, s[kt][nt][1], o[dt][nt], 0, 0, 0);
                    o[dt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(va.z, s[kt][nt][2], o[dt][nt], 0, 0, 0);
                    o[dt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(va.w, s[kt][nt][3], o[dt][nt], 0, 0, 0);
                }
            }
        }

        if (next) {
            __syncthreads();   // every wave is done with the V^T buffer
            store_v();
        }
        __syncthreads();
    }

    float* og = reinterpret_cast<float*>(a.out);
    const int64_t pidx = (int64_t)wk.part * a.Hq + hq;
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
        float lt = lsum[nt];
        lt += __shfl_xor(lt, 16, 64);
        lt += __shfl_xor(lt, 32, 64);
        const int row = w * WQ + nt * 16 + c16;
        const int ql = q_lo + row;
        if (ql >= P) continue;
        const float inv = lt > 0.f ? 1.0f / lt : 0.f;
        float* dst = wk.direct ? og + ((int64_t)(q0 + ql) * a.Hq + hq) * D
                               : a.part_o + (pidx * BQ + row) * D;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
            *reinterpret_cast<float4*>(dst + dt * 16 + 4 * g) =
                make_float4(o[dt][nt][0] * inv, o[dt][nt][1] * inv, o[dt][nt][2] * inv, o[dt][nt][3] * inv);
        if (!wk.direct && g == 0) a.part_lse[pidx * BQ + row] = lt > 0.f ? m[nt] + fast_log2(lt) : -INFINITY;
    }
}

// fp32 pools at head_dim 64 / 96 / 128: both products on the bf16 matrix
// instructions, every operand as the sum of three bf16 terms x = x1 + x2 + x3
// (x1 = bf16(x), x2 = bf16(x - x1), x3 = x - x1 - x2: 24 bits, what fp32 holds),
// and six of the nine partial products,
//     x y = x3 y1 + x2 y2 + x2 y1 + x1 y3 + x1 y2 + x1 y1
// (x3 y2 + x2 y3 + x3 y3 is below 2^-22 |x y|, 2^-25 on average), summed in fp32.
// The fp32 form on v_mfma_f32_16x16x4_f32 ran at 61 % of that instruction's rate
// (356 us for eight 512-row chunks on prefixes up to 4096, 14/2/64);
// v_mfma_f32_32x32x16_bf16 has 16 times the rate, so the six products cost 0.38
// of its matrix time, and the splits are VALU work that runs beside the MFMAs:
// 218 us there, 313 -> 155 us for 32/8/128 chunks of 512, 300 and 77 rows on
// 1000, 0 and 2000.  Bound by the matrix rate on real data and by VALU issue (two
// waves per SIMD at 256 registers; one at head_dim 96 / 128; Q's third terms are
// read from LDS: 222 -> 218 and 176 -> 155 us).
// Two fp16 terms and three products take 172 and 120 us, but hold 22 bits, and
// fewer below 2^-14 of a scale: a V channel of 1e-6 beside channels of one came
// out 7e-5 off, prompts of five rows 9.2e-8 (this form 5.5e-8, the fp32 form
// 7.1e-8), and finite V of 1e34 overflowed their scales.
//
// Error.  A score sums its products with a second or third term first, over every
// k-step, then x1 y1 (D / 16 roundings at its full size; the fp32 form D / 4).  The
// output and the row sums take a tile's sum in one addition, where the fp32 form
// rounds them 16 times per 64 keys: 5.0e-7 -> 3.0e-7 against 64 bits for 512 rows
// on 4096, 14/2/64, and with the output's products summed in place 5.2e-7 (215 us).
//
// bf16 has the exponents of fp32, so nothing is scaled.  A tile or a Q whose
// largest magnitude is beyond 2^60 (infinities included) or, not being zero, below
// 2^-60 runs on the fp32 matrix instructions: within these bounds no sum of
// products of terms overflows.  In a tile that has larger values, one below 2^-110
// keeps an absolute error of at most 2^-126, the smallest normal number.  A tile
// that does not fit is staged again as plain fp32, high halves in the first plane
// and low halves in the second.
//
// K and V tiles lie in LDS as three planes with the operand layout of the 16-bit
// kernel (V^T by transposing reads), split once per work-group while staging.
constexpr int kTerms = 3, kProducts = 6;
constexpr float kFitMax = 0x1p60f, kFitMin = 0x1p-60f;

// x - float(low / high half of w).
__device__ inline float minus_lo(float x, uint32_t w) { return x - __uint_as_float(w << 16); }
__device__ inline float minus_hi(float x, uint32_t w) { return x - __uint_as_float(w & 0xFFFF0000u); }

// The three bf16 terms of 8 values, two per word.
__device__ inline void split8(const float (&x)[8], uint4 (&t)[kTerms]) {
    uint32_t w[kTerms][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        float a = x[2 * j], b = x[2 * j + 1];
#pragma unroll
        for (int p = 0; p < kTerms; ++p) {
            w[p][j] = pack_b2(a, b);
            a = minus_lo(a, w[p][j]);
            b = minus_hi(b, w[p][j]);
        }
    }
#pragma unroll
    for (int p = 0; p < kTerms; ++p) t[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}

// 8 plain fp32 values in the same place, and element e of them.
__device__ inline void plain8(const float (&x)[8], uint4 (&t)[2]) {
    uint32_t w[2][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t a = __float_as_uint(x[2 * j]), b = __float_as_uint(x[2 * j + 1]);
        w[0][j] = (a >> 16) | (b & 0xFFFF0000u);
        w[1][j] = (a & 0xFFFFu) | (b << 16);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) t[p] = make_uint4(w[p][0], w[p][1], w[p][2], w[p][3]);
}
__device__ inline float plain(const uint4 (&t)[2], int e) {
    const uint32_t h = e < 2 ? t[0].x : (e < 4 ? t[0].y : (e < 6 ? t[0].z : t[0].w));
    const uint32_t l = e < 2 ? t[1].x : (e < 4 ? t[1].y : (e < 6 ? t[1].z : t[1].w));
    return __uint_as_float((e & 1) ? (h & 0xFFFF0000u) | (l >> 16) : (h << 16) | (l & 0xFFFFu));
}

// Uniform over the wave: the largest magnitudes `most` of its lanes do not fit
// the terms.  (A NaN passes as one: it stays NaN in either form.)
__device__ inline bool unfit(float most) {
    return __builtin_amdgcn_ballot_w64(most > kFitMax) != 0 ||
           (__builtin_amdgcn_ballot_w64(most >= kFitMin) == 0 && __builtin_amdgcn_ballot_w64(most > 0.0f) != 0);
}

// f(integral_constant 0), ..., f(integral_constant N - 1).
template <class F, int... I>
__device__ inline void static_for_impl(F f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>()), ...);
}
template <int N, class F>
__device__ inline void static_for(F f) {
    static_for_impl(f, std::make_integer_sequence<int, N>());
}

// The six products in the order of accumulation: term of A, term of B.
constexpr int kProdA[kProducts] = {2, 1, 1, 0, 0, 0};
constexpr int kProdB[kProducts] = {0, 1, 0, 2, 1, 0};

// Order of a score's products over K k-steps: per k-step the first five, then,
// again per k-step, x1 y1.  Their A operands come in 4 K groups (one term of one
// k-step), read kAhead groups before their first product into a ring of kAhead + 1.
template <int K>
struct ScoreChain {
    static constexpr int kLength = kProducts * K, kGroups = 4 * K;
    static constexpr bool small(int i) { return i < 5 * K; }
    static constexpr int step(int i) { return small(i) ? i / 5 : i - 5 * K; }        // k-step of product i
    static constexpr int prod(int i) { return small(i) ? i % 5 : kProducts - 1; }
    static constexpr int group(int i) { return small(i) ? 3 * step(i) + 2 - kProdA[prod(i)] : 3 * K + step(i); }
    static constexpr bool first(int i) { return i == 0 || group(i) != group(i - 1); }
    static constexpr int group_step(int g) { return g < 3 * K ? g / 3 : g - 3 * K; }
    static constexpr int group_term(int g) { return g < 3 * K ? 2 - g % 3 : 0; }
};

// split8 of 2 N values in 4 N steps of three VALU instructions or so, to be
// issued one by one between MFMAs: a 32x32x16 MFMA holds the matrix core for 32
// cycles, in which a wave can issue VALU instructions, but only those that stand
// between it and the next MFMA (issue is in order, and the compiler by itself
// puts all VALU work of a region on one side of its MFMAs).
template <int N>
struct SplitSeq {
    static constexpr int kSteps = 4 * N, kStepsOf8 = 16;
    float x[2 * N];
    uint32_t w[kTerms][N];
    float most;   // largest magnitude (step 0 starts it)
    template <bool FIT>
    __device__ void step(int i) {
        const int j = i >> 2;
        float &a = x[2 * j], &b = x[2 * j + 1];
        switch (i & 3) {
            case 0:
                if constexpr (FIT) {
                    const float ab = fmaxf(fabsf(a), fabsf(b));
                    most = i == 0 ? ab : fmaxf(most, ab);
                }
                w[0][j] = pack_b2(a, b);
                break;
            case 1:
                a = minus_lo(a, w[0][j]);
                b = minus_hi(b, w[0][j]);
                break;
            case 2:
                w[1][j] = pack_b2(a, b);
                a = minus_lo(a, w[1][j]);
                break;
            case 3:
                b = minus_hi(b, w[1][j]);
                w[2][j] = pack_b2(a, b);
                break;
        }
    }
    __device__ uint4 term(int p, int c) const {   // values 8 c .. 8 c + 7
        return make_uint4(w[p][4 * c], w[p][4 * c + 1], w[p][4 * c + 2], w[p][4 * c + 3]);
    }
};

template <int D>
struct SmemSplit {
    static constexpr bool kSwz = (D & (D - 1)) == 0;      // 16-byte chunks XOR-swizzled by row, else rows padded
    static constexpr int PAD = kSwz ? D : D + 8;          // halves per row
    union {
        struct {
            alignas(16) uint16_t k[kTerms][BN * PAD];
            alignas(16) uint16_t v[kTerms][BN * PAD];
        };
        int order[6 * kRankUnits];
    };
    alignas(16) uint4 q3[4][D / 16][64];   // third terms of Q: [wave][k-step][lane]
    int pages[kPageWindow];
    int plain[2][2];   // [K, V][tile parity]: the latest such tile that does not fit the terms
    int plain_q;       // a wave's Q does not fit
};

template <int D, bool CG>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(D == 64 ? 2 : 1)))
void prefill_f32_split_kernel(MfmaPrefillArgs a) {
    typedef SmemSplit<D> S;
    constexpr int PAD = S::PAD;
    constexpr int CPR = D / 8;              // 8-value chunks per row
    constexpr int KS = D / 16;              // k-steps of the QK^T product
    constexpr int DT = D / 32;              // 32-dim tiles of the output
    constexpr int CH_T = BN * CPR / 256;    // chunks per thread and tile
    static_assert(BN * CPR % 256 == 0, "chunks spread evenly over the threads");
    __shared__ S sm;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = lane >> 5, c32 = lane & 31;
    Work wk;
    if (!take_work(a, sm.order, wk)) return;
    if (tid < 5) (&sm.plain[0][0])[tid] = tid < 4 ? -1 : 0;   // (before the barrier of stage_pages / below)
    // Every wave's reads of its unit from the ranking, which overlays the tile
    // buffers, complete before any wave writes the first tile (stage_pages has
    // its own barrier).
    if constexpr (CG) lds_barrier();
    poison_uncovered_rows<float, D>(a, wk);
    const int hq = wk.hq, kvh = wk.kvh, n = wk.n;
    const int q0 = wk.q0, P = wk.P, q_lo = wk.q_lo, L = wk.L, kend = wk.kend;
    const int t_begin = wk.t_begin, t_end = wk.t_end;
    const int last_page = L > 0 ? (L - 1) / kPage : 0;
    const int* bt = a.bt + (int64_t)n * a.max_blocks;

    // Q^T operands: lane (h, c32) holds dims 16 ks + 8 h .. + 7 of query c32.
    const int ql = q_lo + w * WQ + c32;
    uint4 qop[KS][2];   // first and second terms (the third: sm.q3)
    const float* qrow = reinterpret_cast<const float*>(a.q) + ((int64_t)(q0 + ql) * a.Hq + hq) * D + h * 8;
    auto read_q = [&](int ks, float (&x)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = 0.0f;
        if (ql < P) {
            const float4* p = reinterpret_cast<const float4*>(qrow + ks * 16);
            const float4 lo = p[0], hi = p[1];
            x[0] = lo.x, x[1] = lo.y, x[2] = lo.z, x[3] = lo.w;
            x[4] = hi.x, x[5] = hi.y, x[6] = hi.z, x[7] = hi.w;
        }
    };
    auto load_q = [&]() {
        float most = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float x[8];
            read_q(ks, x);
#pragma unroll
            for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(x[e]));
            uint4 tm[kTerms];
            split8(x, tm);
            qop[ks][0] = tm[0];
            qop[ks][1] = tm[1];
            sm.q3[w][ks][lane] = tm[2];
        }
        if (unfit(most) && lane == 0) sm.plain_q = 1;
    };
    const int qpos = ql < P ? (a.causal ? wk.hist + ql : L - 1) : -1;
    const int wq0 = q_lo + w * WQ;
    const int wave_min_pos = (wq0 + WQ <= P) ? (a.causal ? wk.hist + wq0 : L - 1) : -1;

    f32x16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[dt][i] = 0.0f;
    float m = kNegBig;
    float lsum = 0.0f;   // this lane's keys only

    // ---- staging: 8 consecutive values per chunk, global -> registers ->
    // three planes in LDS ----------------------------------------------------
    int tbase = 0;
    const uint32_t row_bytes = (uint32_t)(a.Hkv * D * sizeof(float));
    const uint32_t page_bytes = row_bytes * kPage;
    const int64_t kv0 = (int64_t)kvh * D + (CG ? (int64_t)wk.kvo : 0);
    const char* kb_ = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.k) + kv0);
    const char* vb_ = reinterpret_cast<const char*>(reinterpret_cast<const float*>(a.v) + kv0);
    uint32_t off[CH_T];   // bytes inside the page (paged) / the row (contiguous)
    int slot[CH_T];       // page of the tile / key of the tile
    int kdst[CH_T], vdst[CH_T];   // halves inside a plane
    // Half-column hc of tile row `row` in the K / V planes (swizzled: the 16-byte
    // chunk index XORed with a permutation of the row's low bits).  K: the 16
    // lanes of a read phase hold rows 0 .. 15 of one chunk, lanes 0 .. 7 rows
    // 0 .. 3 and 8 .. 11.  V: a transposing read takes 2 chunks of 4 rows.
    auto kcol = [&](int row, int hc) {
        const int b0 = row & 1, b1 = (row >> 1) & 1, b2 = (row >> 2) & 1, b3 = (row >> 3) & 1;
        if constexpr (D == 64) return (((hc >> 3) ^ (b1 | (b3 << 1) | ((b0 ^ b2) << 2))) << 3) | (hc & 7);
        if constexpr (D == 128) return (((hc >> 3) ^ (b0 | (b1 << 1) | (b3 << 2) | (b2 << 3))) << 3) | (hc & 7);
        return hc;
    };
    auto vcol = [&](int row, int hc) {
        const int b0 = row & 1, b1 = (row >> 1) & 1, b2 = (row >> 2) & 1;
        if constexpr (D == 64) return (((hc >> 3) ^ ((b0 << 1) | (b1 << 2))) << 3) | (hc & 7);
        if constexpr (D == 128) return (((hc >> 3) ^ ((b2 << 1) | (b0 << 2) | (b1 << 3))) << 3) | (hc & 7);
        return hc;
    };
#pragma unroll
    for (int j = 0; j < CH_T; ++j) {
        const int ch = tid + 256 * j;
        const int key = ch / CPR, c = ch % CPR;
        slot[j] = CG ? key : key >> 4;
        off[j] = (CG ? 0u : (uint32_t)(key & 15) * row_bytes) + (uint32_t)c * 32u;
        kdst[j] = key * PAD + kcol(key, c * 8);
        vdst[j] = key * PAD + vcol(key, c * 8);
    }
    float kraw[CH_T][8], vraw[CH_T][8];
    auto load_tile = [&](const char* base, int t, float (&raw)[CH_T][8]) {
        const int* pg = sm.pages + (4 * t - tbase);
#pragma unroll
        for (int j = 0; j < CH_T; ++j) {
            uint64_t at;
            if constexpr (CG) at = (uint64_t)min(t * BN + slot[j], L - 1) * row_bytes;   // past the last: the last
            else at = (uint64_t)(uint32_t)max(pg[slot[j]], 0) * page_bytes;
            const f32x4* p = reinterpret_cast<const f32x4*>(base + at + off[j]);
            const f32x4 lo = p[0], hi = p[1];
#pragma unroll
            for (int e = 0; e < 4; ++e) raw[j][e] = lo[e], raw[j][4 + e] = hi[e];
        }
    };
    // Splits a staged tile into its planes; returns the lane's largest magnitude.
    auto split_tile = [&](const float (&raw)[CH_T][8], uint16_t (&planes)[kTerms][BN * PAD],
                          const int (&dst)[CH_T]) {
        float most = 0.0f;
#pragma unroll
        for (int j = 0; j < CH_T; ++j) {
            uint4 tm[kTerms];
#pragma unroll
            for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(raw[j][e]));
            split8(raw[j], tm);
#pragma unroll
            for (int p = 0; p < kTerms; ++p) *reinterpret_cast<uint4*>(&planes[p][dst[j]]) = tm[p];
        }
        return most;
    };
    // After a split that found tile t of K (kv 0) or V (kv 1) unfit: the whole
    // tile once more, plain.  Called by every wave (it ends with a barrier).
    auto restage_plain = [&](uint16_t (&planes)[kTerms][BN * PAD], const int (&dst)[CH_T], const char* base, int t) {
        float raw[CH_T][8];
        load_tile(base, t, raw);
#pragma unroll
        for (int j = 0; j < CH_T; ++j) {
            uint4 tm[2];
            plain8(raw[j], tm);
#pragma unroll
            for (int p = 0; p < 2; ++p) *reinterpret_cast<uint4*>(&planes[p][dst[j]]) = tm[p];
        }
        lds_barrier();
    };
    auto stage_pages = [&](int base) {
        if constexpr (CG) return;   // no page table
        tbase = base;
        for (int i = tid; i < kPageWindow; i += 256) sm.pages[i] = bt[min(base + i, last_page)];
        lds_barrier();
    };
    // A operand of S^T: row c32 of key tile kt holds key 32 kt + (c32 with bits
    // 2 and 3 exchanged), which makes the 8 scores of each 16-key step that a
    // lane receives (accumulator rows 8 (i / 4) + 4 h + i % 4) keys 8 h .. 8 h + 7.
    const int krow = (c32 & 0x13) | ((c32 & 4) << 1) | ((c32 & 8) >> 1);
    auto k_operand = [&](int kt, int ks, int p) {
        const int row = 32 * kt + krow;
        return *reinterpret_cast<const uint4*>(&sm.k[p][row * PAD + kcol(row, ks * 16 + h * 8)]);
    };
    // A operand of O^T: lane holds dim 32 dt + c32 of keys 16 j + 8 h .. + 7
    // (transposing reads, as in the 16-bit kernel).
    auto v_operand = [&](int dt, int j, int p) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        typedef unsigned u32x2v __attribute__((ext_vector_type(2)));
        const int r0 = 16 * j + 8 * h + ((lane & 15) >> 2), hc = dt * 32 + (lane & 16) + 4 * (lane & 3);
        const int a0 = r0 * PAD + vcol(r0, hc), a1 = (r0 + 4) * PAD + vcol(r0 + 4, hc);
        const u32x2v lo = __builtin_bit_cast(u32x2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(&sm.v[p][a0])));
        const u32x2v hi = __builtin_bit_cast(u32x2v, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(&sm.v[p][a1])));
        return make_uint4(lo.x, lo.y, hi.x, hi.y);
    };
    if (t_begin < t_end) {
        stage_pages(4 * t_begin);
        load_tile(kb_, t_begin, kraw);
        load_tile(vb_, t_begin, vraw);
        load_q();
        if (unfit(split_tile(kraw, sm.k, kdst)) && lane == 0) sm.plain[0][t_begin & 1] = t_begin;
    }
    lds_barrier();

    // A tile: QK^T (V of the tile split beside it, its buffer being free since
    // the last barrier), barrier, softmax and PV (K of the next tile split
    // beside them), barrier.  The raw values are loaded a phase ahead; the
    // barriers do not wait for them.
    for (int t = t_begin; t < t_end; ++t) {
        const bool next = t + 1 < t_end;   // uniform
        if (next) {
            if (4 * (t + 1) + 4 > tbase + kPageWindow) stage_pages(4 * t);   // (tile t: restage_plain)
            load_tile(kb_, t + 1, kraw);
        }
        // (the same for every wave: set before the last barrier)
        const bool k_plain = __builtin_amdgcn_readfirstlane(sm.plain_q) != 0 ||
                             __builtin_amdgcn_readfirstlane(sm.plain[0][t & 1]) == t;
        __builtin_amdgcn_sched_barrier(0);

        // ---- S^T = K Q^T; the lane's scores are keys 32 kt + 16 (i / 8) + 8 h + i % 8
        f32x16 s[2];
        float v_most, k_most;
        const float c = a.scale_log2;
        if (__builtin_expect(!k_plain, 1)) {
            SplitSeq<4 * CH_T> sq;
#pragma unroll
            for (int j = 0; j < CH_T; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) sq.x[8 * j + e] = vraw[j][e];
            typedef ScoreChain<KS> Ch;
            constexpr int kAhead = 2;
            uint4 ka[kAhead + 1][2];   // [group][key tile]
            uint4 q3;
            auto read_k = [&](int gr) {
#pragma unroll
                for (int kt = 0; kt < 2; ++kt)
                    ka[gr % (kAhead + 1)][kt] = k_operand(kt, Ch::group_step(gr), Ch::group_term(gr));
            };
#pragma unroll
            for (int gr = 0; gr < kAhead; ++gr) read_k(gr);
            constexpr int M = 2 * Ch::kLength, M0 = 4;   // MFMAs; those before V's split (its loads have time to land)
            static_for<M>([&](auto kc) {
                constexpr int k = kc, i = k / 2, kt = k & 1, ks = Ch::step(i), gr = Ch::group(i), qt = kProdB[Ch::prod(i)];
                if constexpr (kt == 0 && Ch::first(i) && gr + kAhead < Ch::kGroups) read_k(gr + kAhead);
                if constexpr (kt == 0 && i < 5 * KS && i % 5 == 0) q3 = sm.q3[w][ks][lane];
                s[kt] = Mfma<bf16_t>::mma32(ka[gr % (kAhead + 1)][kt], qt == 2 ? q3 : qop[ks][qt & 1],
                                            i == 0 ? f32x16{} : s[kt]);
                if constexpr (k >= M0) {
                    constexpr int s0 = (k - M0) * sq.kSteps / (M - M0), s1 = (k + 1 - M0) * sq.kSteps / (M - M0);
                    static_for<s1 - s0>([&](auto ec) {
                        constexpr int st = s0 + ec;
                        sq.template step<true>(st);
                        if constexpr ((st + 1) % sq.kStepsOf8 == 0) {
#pragma unroll
                            for (int p = 0; p < kTerms; ++p)
                                *reinterpret_cast<uint4*>(&sm.v[p][vdst[st / sq.kStepsOf8]]) = sq.term(p, st / sq.kStepsOf8);
                        }
                    });
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            v_most = sq.most;
        } else {
            restage_plain(sm.k, kdst, kb_, t);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) s[kt] = f32x16{};
            for (int ks = 0; ks < KS; ++ks) {
                float x[8];
                read_q(ks, x);
#pragma unroll
                for (int kt = 0; kt < 2; ++kt) {
                    const uint4 ka[2] = {k_operand(kt, ks, 0), k_operand(kt, ks, 1)};
#pragma unroll
                    for (int e = 0; e < 8; ++e)   // contracts dims 16 ks + 8 h + e
                        s[kt] = __builtin_amdgcn_mfma_f32_32x32x2f32(plain(ka, e), x[e], s[kt], 0, 0, 0);
                }
            }
            v_most = split_tile(vraw, sm.v, vdst);
        }
        if (unfit(v_most) && lane == 0) sm.plain[1][t & 1] = t;
        lds_barrier();   // V of the tile is in LDS; every wave is done with the K buffer
        const bool v_plain = __builtin_amdgcn_readfirstlane(sm.plain[1][t & 1]) == t;   // the same for every wave
        if (__builtin_expect(v_plain, 0)) restage_plain(sm.v, vdst, vb_, t);
        if (next) load_tile(vb_, t + 1, vraw);

        // ---- mask and online softmax (as the 16-bit kernel) ----------------
        const int key0 = t * BN;
        const bool unmasked = key0 + BN - 1 <= wave_min_pos && key0 + BN <= kend;
        if (!unmasked) {
            const int r = min(qpos, kend - 1) - key0 - 8 * h;
#pragma unroll
            for (int kt = 0; kt < 2; ++kt)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (32 * kt + 16 * (i >> 3) + (i & 7) > r) s[kt][i] = -INFINITY;
        }
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kt][i]);
        mx *= c;
        if (__builtin_amdgcn_ballot_w64(mx > m + 8.0f) != 0) {
            const float mnew = fmaxf(m, fmaxf(mx, __shfl_xor(mx, 32, 64)));
            const float corr = fast_exp2(m - mnew);
            m = mnew;
            lsum *= corr;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] *= corr;
        }

        // ---- P = 2^(S c - m), O^T += V^T P^T ------------------------------
        if (__builtin_expect(!v_plain, 1)) {
            // P's terms of 16-key step j + 1 are made beside the MFMAs of step j, the
            // next tile's K is split beside the last step's (after the last tile: into a
            // buffer nobody reads).
            uint4 pop[kTerms];
            float psum = 0.0f;
            {
                float p[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    p[e] = fast_exp2(fmaf(s[0][e], c, -m));
                    psum += p[e];
                }
                split8(p, pop);
            }
            SplitSeq<4 * CH_T> sq;
#pragma unroll
            for (int j = 0; j < CH_T; ++j)
#pragma unroll
                for (int e = 0; e < 8; ++e) sq.x[8 * j + e] = kraw[j][e];
            constexpr int kGroups = 4 * kTerms;
            uint4 va[2][DT];   // [group (a term of a step) mod 2]
            auto read_v = [&](int gr) {
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) va[gr & 1][dt] = v_operand(dt, gr / kTerms, 2 - gr % kTerms);
            };
            read_v(0);
            f32x16 od[DT];   // the tile's sums
            static_for<4>([&](auto jc) {
                constexpr int j = jc, M = kProducts * DT;
                SplitSeq<4> ps;
                static_for<M>([&](auto kc) {
                    constexpr int k = kc, dt = k % DT, pr = k / DT, gr = kTerms * j + 2 - kProdA[pr];
                    constexpr bool first = pr == 0 || kProdA[pr] != kProdA[pr - (pr > 0)];   // of its group
                    if constexpr (dt == 0 && first && gr + 1 < kGroups) read_v(gr + 1);
                    od[dt] = Mfma<bf16_t>::mma32(va[gr & 1][dt], pop[kProdB[pr]],
                                                 j == 0 && pr == 0 ? f32x16{} : od[dt]);
                    if constexpr (j < 3) {   // 8 exponentials, then their terms
                        constexpr int s0 = k * (8 + ps.kSteps) / M, s1 = (k + 1) * (8 + ps.kSteps) / M;
                        static_for<s1 - s0>([&](auto ec) {
                            constexpr int st = s0 + ec;
                            if constexpr (st < 8) {
                                constexpr int e = 8 * (j + 1) + st;
                                ps.x[st] = fast_exp2(fmaf(s[e >> 4][e & 15], c, -m));
                                psum += ps.x[st];
                            } else {
                                ps.template step<false>(st - 8);
                            }
                        });
                    } else {
                        constexpr int s0 = k * sq.kSteps / M, s1 = (k + 1) * sq.kSteps / M;
                        static_for<s1 - s0>([&](auto ec) {
                            constexpr int st = s0 + ec;
                            sq.template step<true>(st);
                            if constexpr ((st + 1) % sq.kStepsOf8 == 0) {
#pragma unroll
                                for (int p = 0; p < kTerms; ++p)
                                    *reinterpret_cast<uint4*>(&sm.k[p][kdst[st / sq.kStepsOf8]]) = sq.term(p, st / sq.kStepsOf8);
                            }
                        });
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
                if constexpr (j < 3) {
#pragma unroll
                    for (int p = 0; p < kTerms; ++p) pop[p] = ps.term(p, 0);
                }
            });
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) o[dt] += od[dt];
            lsum += psum;
            k_most = sq.most;
        } else {
            // (an opaque copy: the exponentials of the two branches must not be
            // merged and moved ahead of the branch)
            float mq = m;
            asm volatile("" : "+v"(mq));
            float psum = 0.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float p[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    p[e] = fast_exp2(fmaf(s[j >> 1][8 * (j & 1) + e], c, -mq));
                    psum += p[e];
                }
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) {
                    const uint4 va[2] = {v_operand(dt, j, 0), v_operand(dt, j, 1)};
#pragma unroll
                    for (int e = 0; e < 8; ++e)   // contracts keys 16 j + 8 h + e
                        o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(plain(va, e), p[e], o[dt], 0, 0, 0);
                }
            }
            lsum += psum;
            k_most = split_tile(kraw, sm.k, kdst);
        }
        if (unfit(k_most) && lane == 0) sm.plain[0][(t + 1) & 1] = t + 1;
        lds_barrier();   // K of the next tile is in LDS; every wave is done with the V buffer
    }

    lsum += __shfl_xor(lsum, 32, 64);
    if (ql >= P) return;
    const float inv = lsum > 0.f ? 1.0f / lsum : 0.f;
    const int64_t prow = ((int64_t)wk.part * a.Hq + hq) * BQ + w * WQ + c32;
    float* drow = wk.direct ? reinterpret_cast<float*>(a.out) + ((int64_t)(q0 + ql) * a.Hq + hq) * D
                            : a.part_o + prow * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)   // accumulator rows 8 i + 4 h .. + 3 of dim tile dt
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float4*>(drow + dt * 32 + 8 * i + 4 * h) =
                make_float4(o[dt][4 * i] * inv, o[dt][4 * i + 1] * inv, o[dt][4 * i + 2] * inv, o[dt][4 * i + 3] * inv);
    if (!wk.direct && h == 0) a.part_lse[prow] = lsum > 0.f ? m + fast_log2(lsum) : -INFINITY;
}

// Four consecutive output elements from fp32 values.
template <typename T>
__device__ inline void store4(T* p, float x, float y, float z, float w) {
    uint2 w2;
    w2.x = Mfma<T>::pack2(x, y);
    w2.y = Mfma<T>::pack2(z, w);
    *reinterpret_cast<uint2*>(p) = w2;
}
template <>
__device__ inline void store4<float>(float* p, float x, float y, float z, float w) {
    *reinterpret_cast<float4*>(p) = make_float4(x, y, z, w);
}

// Merge of a (sequence, query block, q head) unit's key chunks: grid
// (Hq, N x qblocks), 256 threads; thread (row, part) merges dims
// [part * D/TPR, (part + 1) * D/TPR) of one row over the chunks with an online
// log-sum-exp (each chunk's lse and row slice are loaded together).
template <typename T, int D>
__global__ __launch_bounds__(256) void prefill_merge_kernel(MfmaPrefillArgs a) {
    constexpr int TPR = 256 / BQ;     // threads per row
    constexpr int V4 = D / TPR / 4;   // float4 per thread
    const int hq = blockIdx.x, unit = blockIdx.y;
    // The unit's first partial slot and chunks, from the main kernel; loaded
    // together with the lengths below and checked before anything is written.
    const int2 cut = a.table[unit];
    const int n = unit / a.qblocks;
    const int qb = a.qblocks - 1 - (unit % a.qblocks);
    int q0, P, L, kvo, hist;
    seq_geom(a, n, q0, P, L, kvo, hist);
    const int nchunks = cut.y;
    if (nchunks <= 1) return;   // written directly (or no rows)
    const int q_lo = qb * BQ;
    const int row = threadIdx.x / TPR, part = threadIdx.x % TPR;
    if (q_lo + row >= P) return;
    const int64_t p0 = (int64_t)cut.x * a.Hq + hq;   // chunk c at p0 + c * Hq
    float M = -INFINITY, W = 0.0f;
    float4 acc[V4];
#pragma unroll
    for (int v = 0; v < V4; ++v) acc[v] = make_float4(0.f, 0.f, 0.f, 0.f);
    // CB chunks per memory round trip: every load of a batch is issued before
    // any of its values is used (chunks past nchunks load the last one and take
    // lse -inf), and the merge step has no branch, so the compiler cannot sink
    // the row loads behind the lse.  A chunk whose row saw no key has lse -inf
    // and a zero row: weight 0, no change.  Two chunks per batch: the plan cuts
    // most split units in two, and fp32 rows of four chunks held 128 registers
    // and loaded the last chunk three times (configuration 4 57.6 -> 56.9 us).
    constexpr int CB = 2;
    for (int c0 = 0; c0 < nchunks; c0 += CB) {
        float l[CB];
        float4 raw[CB][V4];
#pragma unroll
        for (int k = 0; k < CB; ++k) {
            const int c = min(c0 + k, nchunks - 1);
            const int64_t pc = (p0 + (int64_t)c * a.Hq) * BQ + row;
            const float lk = a.part_lse[pc];
            l[k] = c0 + k < nchunks ? lk : -INFINITY;
            const float4* src = reinterpret_cast<const float4*>(a.part_o + pc * D) + part * V4;
#pragma unroll
            for (int v = 0; v < V4; ++v) raw[k][v] = src[v];
        }
#pragma unroll
        for (int k = 0; k < CB; ++k) {
            const float4* o = raw[k];
            const float Mn = fmaxf(M, l[k]);
            const bool live = Mn != -INFINITY;   // some key seen by this row so far
            const float sc = live ? fast_exp2(M - Mn) : 1.0f;
            const float wt = live ? fast_exp2(l[k] - Mn) : 0.0f;
            W = fmaf(W, sc, wt);
#pragma unroll
            for (int v = 0; v < V4; ++v) {
                acc[v].x = fmaf(acc[v].x, sc, wt * o[v].x);
                acc[v].y = fmaf(acc[v].y, sc, wt * o[v].y);
                acc[v].z = fmaf(acc[v].z, sc, wt * o[v].z);
                acc[v].w = fmaf(acc[v].w, sc, wt * o[v].w);
            }
            M = live ? Mn : M;
        }
    }
    const float inv = W > 0.f ? 1.0f / W : 0.f;
    T* orow = reinterpret_cast<T*>(a.out) + ((int64_t)(q0 + q_lo + row) * a.Hq + hq) * D + part * V4 * 4;
#pragma unroll
    for (int v = 0; v < V4; ++v)
        store4(orow + 4 * v, acc[v].x * inv, acc[v].y * inv, acc[v].z * inv, acc[v].w * inv);
}

bool prefill_mfma_handles(int head_dim, int block_size, int dtype) {
    // head_dim 256: one work-group per CU (fp32: single-buffered tiles, 134 KB)
    return block_size == kPage && (head_dim == 64 || head_dim == 96 || head_dim == 128 || head_dim == 256);
}

// Key-range split (pick_item).  The host lets a launch cut units, which costs a
// merge kernel and the partials' traffic, when the units' heads alone would not
// fill the resident slots.  With more, cutting measured slower even where one
// unit is far longer than the others (32/8/128 bf16 chunks of 1 .. 1101 rows on
// prefixes up to 3000: 81 us, cut 86 .. 97).  Units are counted from the rows
// (at most total_q / BQ + N hold any), not as N x the longest sequence's blocks:
// 28/4/128 bf16 chunks of 64, 31, 700 and 5 rows 89 -> 38 us by that count.
// Kernels of one work-group per CU (fp32 at head_dim 96 / 128, head_dim 256) may cut
// up to twice their slots: no second work-group runs beside a long one there.
// A bound of the lengths that no unit can pass the rule of pick_item with (chunks
// of max_q_len rows on no prefixes) saves the merge kernel's launch, 2 .. 3 us
// (32/8/128 fp16 chunks of 1139, 226, 18, 2 and 10 rows 35.9 -> 32.9).
// The workspace is sized for kSizingSlots resident slots (256 CUs x 4
// work-groups, above what these kernels reach), so that it does not depend on
// the device.
constexpr int kSizingSlots = 1024;
constexpr int kSizingItems = 512;   // items per head that cuts may add, above a device's CUs

typedef void (*PrefillFn)(MfmaPrefillArgs);

template <typename T, bool CG>
PrefillFn kernel16(int head_dim) {
    switch (head_dim) {
        case 64: return prefill_mfma_kernel<T, 64, CG>;
        case 96: return prefill_mfma_kernel<T, 96, CG>;
        case 128: return prefill_mfma_kernel<T, 128, CG>;
        default: return prefill_mfma_kernel<T, 256, CG>;
    }
}

template <bool CG>
PrefillFn kernel32(int head_dim) {
    switch (head_dim) {
        case 64: return prefill_f32_split_kernel<64, CG>;
        case 96: return prefill_f32_split_kernel<96, CG>;
        case 128: return prefill_f32_split_kernel<128, CG>;
        default: return prefill_f32_kernel<256, CG>;
    }
}

template <bool CG>
PrefillFn prefill_kernel_cg(int dtype, int head_dim) {
    if (dtype == LLKV_DTYPE_F32) return kernel32<CG>(head_dim);
    if (dtype == LLKV_DTYPE_F16) return kernel16<_Float16, CG>(head_dim);
    return kernel16<bf16_t, CG>(head_dim);
}

PrefillFn prefill_kernel(int dtype, int head_dim, bool contig) {
    return contig ? prefill_kernel_cg<true>(dtype, head_dim) : prefill_kernel_cg<false>(dtype, head_dim);
}

template <typename T>
PrefillFn merge_for(int head_dim) {
    switch (head_dim) {
        case 64: return prefill_merge_kernel<T, 64>;
        case 96: return prefill_merge_kernel<T, 96>;
        case 128: return prefill_merge_kernel<T, 128>;
        default: return prefill_merge_kernel<T, 256>;
    }
}

PrefillFn merge_kernel(int dtype, int head_dim) {
    if (dtype == LLKV_DTYPE_F32) return merge_for<float>(head_dim);
    if (dtype == LLKV_DTYPE_F16) return merge_for<_Float16>(head_dim);
    return merge_for<bf16_t>(head_dim);
}

// Workspace: a 256-byte header (unused, part of the size that callers know), then
// max_parts partial slots (Hq x BQ rows each), then one slot for the merge kernel's
// table.
constexpr size_t kHeaderBytes = 256;

struct ChunkPlan {
    int qblocks, units;   // query blocks per sequence; bound of the units with rows
    int extra, parts;     // items beyond `units`; partial slots (0: nothing is cut)
};

ChunkPlan chunk_plan(int N, int Hq, int total_q, int max_q_len, int max_seq_len) {
    ChunkPlan c;
    const int qmax = (max_q_len > 0 && max_q_len < total_q) ? max_q_len : total_q;
    c.qblocks = (qmax + BQ - 1) / BQ;
    const int64_t all = (int64_t)N * c.qblocks;
    c.units = (int)std::min<int64_t>(all, (int64_t)total_q / BQ + N);   // sum of ceil(rows / BQ)
    const int max_tiles = (std::max(max_seq_len, 1) + BN - 1) / BN;
    c.extra = c.parts = 0;
    if (all <= kRankUnits && max_tiles >= 2 * kMinChunkTiles &&
        (int64_t)c.units * Hq < kSizingSlots) {
        const int64_t share = (kSizingItems + Hq - 1) / Hq;   // at least sum / limit (pick_item)
        c.extra = (int)share;
        c.parts = (int)std::max<int64_t>(2, std::min<int64_t>(2 * share, (int64_t)c.units * ((max_tiles - 1) / kMinChunkTiles + 2)));
    }
    return c;
}

// Key tiles of total_q rows in chunks of max_q_len on no prefixes.
int64_t causal_tiles(int total_q, int max_q_len) {
    const int64_t rows = (max_q_len > 0 && max_q_len < total_q) ? max_q_len : total_q;
    auto tiles = [](int64_t n) {   // 2, 4, .. of the whole query blocks, and the last
        const int64_t m = n / BQ;
        return m * (m + 1) + (n % BQ != 0 ? (n + BN - 1) / BN : 0);
    };
    return total_q / rows * tiles(rows) + tiles(total_q % rows);
}

// Tiles that cutting has to save (pick_item): a merge and the partials, whose bytes
// grow with head_dim, over a tile's time.  Of 475 random batches of every type and
// head_dim the slower of cut and uncut is taken by 1.1x at most so; by one margin of
// 4 tiles, 1.2x (16 bits at head_dim 128), of 16, 1.9x (fp32 at 256).
int cut_margin(int dtype, int head_dim) {
    return dtype == LLKV_DTYPE_F32 ? head_dim / 32 : 6 + head_dim / 64;
}

size_t part_bytes(int Hq, int head_dim) { return (size_t)Hq * BQ * (1 + head_dim) * sizeof(float); }

}  // namespace

size_t prefill_mfma_workspace(int N, int Hq, int head_dim, int block_size, int dtype, int total_q,
                              int max_q_len, int max_seq_len) {
    if (!prefill_mfma_handles(head_dim, block_size, dtype) || N <= 0 || total_q <= 0) return 0;
    const ChunkPlan c = chunk_plan(N, Hq, total_q, max_q_len, max_seq_len);
    return c.parts > 0 ? kHeaderBytes + (size_t)(c.parts + 1) * part_bytes(Hq, head_dim) : 0;
}

int launch_prefill_mfma(MfmaPrefillArgs a, int head_dim, int block_size, int dtype,
                        int total_q, int max_q_len, int max_seq_len, void* workspace,
                        size_t workspace_bytes, hipStream_t st) {
    if (!prefill_mfma_handles(head_dim, block_size, dtype)) return -1;
    if (((uintptr_t)a.q | (uintptr_t)a.out | (uintptr_t)a.k | (uintptr_t)a.v) & 15) return -1;
    const int slots = resident_workgroups(reinterpret_cast<const void*>(prefill_kernel(dtype, head_dim, false)), 256);
    a.n_cus = device_cus();
    a.resident = a.contig ? resident_workgroups(reinterpret_cast<const void*>(prefill_kernel(dtype, head_dim, true)), 256)
                          : slots;
    const ChunkPlan c = chunk_plan(a.N, a.Hq, total_q, max_q_len, max_seq_len);
    a.qblocks = c.qblocks;
    const size_t need = prefill_mfma_workspace(a.N, a.Hq, head_dim, block_size, dtype, total_q,
                                               max_q_len, max_seq_len);
    a.max_parts = 0;
    a.extra_items = 0;
    a.table = nullptr;
    a.part_lse = a.part_o = nullptr;
    a.cut_margin = cut_margin(dtype, head_dim);
    const int cut_below = a.resident < 2 * a.n_cus ? 2 * a.resident : a.resident;
    const int64_t max_tiles = (std::max(max_seq_len, 1) + BN - 1) / BN;
    const bool uneven = !a.causal || (max_tiles - a.cut_margin) * a.n_cus > causal_tiles(total_q, max_q_len) * a.Hq;
    if (need > 0 && uneven && (int64_t)c.units * a.Hq < cut_below && workspace != nullptr &&
        workspace_bytes >= need) {
        a.max_parts = c.parts;
        a.extra_items = c.extra;
        char* base = reinterpret_cast<char*>(workspace) + kHeaderBytes;
        const size_t rows = (size_t)c.parts * a.Hq * BQ;
        a.part_lse = reinterpret_cast<float*>(base);
        a.part_o = a.part_lse + rows;
        a.table = reinterpret_cast<int2*>(base + (size_t)c.parts * part_bytes(a.Hq, head_dim));
    }
    // every unit's own item (index order above kRankUnits units), and the cuts
    const int64_t all = (int64_t)a.N * a.qblocks;
    const int64_t groups = (all > kRankUnits ? all : c.units + a.extra_items) * a.Hkv;
    const int G = a.Hq / a.Hkv;
    a.groups = (int)groups;
    int64_t wgs = ((groups + kXcds - 1) / kXcds) * kXcds * G;
    if (a.resident >= 2 * a.n_cus && wgs > a.n_cus) wgs = std::max<int64_t>(wgs, 2 * a.n_cus);   // take_work
    dim3 grid((unsigned)wgs);
    prefill_kernel(dtype, head_dim, a.contig != 0)<<<grid, 256, 0, st>>>(a);
    if (a.max_parts > 0)
        merge_kernel(dtype, head_dim)<<<dim3(a.Hq, a.N * a.qblocks), 256, 0, st>>>(a);
    return check_launch(a.contig ? "llkv_first_prefill_batched" : "llkv_paged_prefill");
}

}  // namespace llkv
