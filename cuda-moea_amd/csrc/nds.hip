// Constrained non-dominated sorting on CDNA4.
//
// Replaces the reference's run_ndsort / run_ndsort_init
// (NS/selection/nsga3/kernels/non_dominated_sort.cu:1407-1574, 1333-1405):
// same dominance rule (constraint_dominatee_bitmask_kernel, :409-459), same
// stopping rule (fronts are peeled until at least stop_at individuals are
// assigned; the rest keep front -1; :824-840, 1182-1204), but with no pair
// buffer, no host round trip per front and no capacity limit.
//
// Pipeline (all on one stream, no host synchronisation):
//  1. nds_keys + radix sort: rows are ordered by the key
//       segment 0  feasible, no NaN objective    -> f0 (with -0 read as +0)
//       segment 1  feasible, some NaN objective  -> (input order)
//       segment 2  infeasible                    -> cv (NaN last)
//     In this order a later row can dominate an earlier row only when both
//     are in segment 0 with equal f0: a feasible row is never dominated by an
//     infeasible one, a NaN objective compares false both ways, infeasible
//     rows dominate by strictly smaller cv, and q <= p in every objective with
//     f0(q) > f0(p) is impossible.
//  2. nds_prep: objectives in sorted order; per 64-row block b, valid[b] (which
//     rows are in segment 0) and hi[b], the last block holding a row whose key
//     equals the key of block b's last row (b itself unless an f0 tie runs past
//     the block).  Dominators of a row of block b all lie in blocks <= hi[b].
//     Per chunk of 512 sorted rows and objective, a rank table (see RankTable).
//  3. nds_dominance: the dominator bitmask B in sorted order, words (p, w) for
//     w <= hi[p/64], from the rank tables: a search and a table row per
//     objective give a row's "q_k <= p_k" over a whole chunk.
//  4. nds_peel: front peeling of the feasible rows with per-row cursors on B,
//     by one workgroup up to 2048 rows (an ordinary launch) and by cooperating
//     ones above; the infeasible rows' fronts follow from their order alone;
//     fronts are written back in input order.
//
// Infeasible rows need no bitmask: every feasible row dominates them, among
// themselves they are ordered by cv alone, and a NaN cv neither dominates nor
// is dominated by another infeasible row.  So with F feasible fronts the rows
// with the j-th smallest distinct cv are front F + j and the NaN rows front F.
// Peeled one front a round they cost a grid barrier per distinct cv: 17.2 ms
// for 20001 rows of which a fifth are infeasible, against 0.2 ms this way.
//
// Data layout of B (u64 words, sorted row index p):
//   W  = ceil(n / 64) words per row (bit q%64 of word q/64 = "q dominates p"),
//   Wc = ceil(W / 8) chunks of 8 words per row,
//   word (p, w) lives at (((p/64) * Wc + w/8) * 64 + p%64) * 8 + w%8.
// A 64-row x 8-word chunk is 4 KiB contiguous: the dominance kernel writes it
// as one 64-byte segment per lane, the peel reads a row's words 8 at a time.
#include <algorithm>
#include <atomic>
#include <mutex>
#include <string>
#include <vector>

#include "batch_internal.hpp"
#include "common.hpp"
#include "moea_internal.hpp"

namespace moea {

namespace {

constexpr int kRowEndMinM = 4;           // fewest objectives for which the sort computes row ends
// Threads of a dominance workgroup, each wave a row block at a time: from six
// objectives one workgroup's tables fill a CU's LDS, so it brings all 16 waves.
constexpr int dom_threads(int m) { return m >= 6 ? 1024 : 512; }
constexpr int kChunk = 512;              // sorted rows q per rank table: the 8 words of a chunk of B
constexpr int kKeyBits = 34;             // segment (2 bits) above a 32-bit order key

__host__ __device__ __forceinline__ size_t bword_index(int p, int w, int Wc)
{
    return ((static_cast<size_t>(p >> 6) * Wc + (w >> 3)) * 64 + (p & 63)) * 8 + (w & 7);
}

__device__ __forceinline__ uint64_t nds_key_of(const float* __restrict__ f, int ldf, const float* __restrict__ cv,
                                      int s, int m)
{
    const float c = cv[s];
    bool nan = false;
    if (c == 0.0f)
        for (int k = 0; k < m; ++k) nan = nan || isnan(f[static_cast<size_t>(k) * ldf + s]);
    return nds_key_from(f[s], nan, c);
}

__global__ void nds_keys(const float* __restrict__ f, int ldf, const float* __restrict__ cv, int n,
                         int m, uint64_t* __restrict__ keys, int32_t* __restrict__ vals)
{
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    keys[s] = nds_key_of(f, ldf, cv, s, m);
    vals[s] = s;
}

// The infeasible rows of the sort order, found by one wave per 64-row block:
// gmask[b] has a bit for each row of block b that is the first of its cv (NaN
// cv left out); info[kInfoFeasible] is the number of feasible rows and
// info[kInfoOrdered] the end of the rows with a cv that is not NaN, each
// written by the wave whose row comes just before (row 0's wave for 0).
constexpr int kInfoFeasible = 0, kInfoOrdered = 1;

__device__ __forceinline__ int infeasible_class(uint64_t key)
{
    return ((key >> 32) & 3u) != 2 ? 0 : static_cast<uint32_t>(key) != 0xFFFFFFFFu ? 1 : 2;
}

__device__ __forceinline__ void infeasible_info(const uint64_t* __restrict__ keys, int n, int t,
                                                uint64_t* __restrict__ gmask, int32_t* __restrict__ info)
{
    const bool valid = t < n;
    const uint64_t key = valid ? keys[t] : 0;
    const uint64_t prev = (valid && t > 0) ? keys[t - 1] : 0;
    // 0 feasible, 1 infeasible with a number, 2 NaN cv, 3 past the end
    const int c = valid ? infeasible_class(key) : 3;
    const int c0 = t > 0 ? infeasible_class(prev) : 0;
    const uint64_t starts = ballot(c == 1 && (t == 0 || prev != key));
    if ((threadIdx.x & 63) == 0) gmask[t >> 6] = starts;
    if (valid && c0 == 0 && c != 0) info[kInfoFeasible] = t;
    if (valid && c0 <= 1 && c == 2) info[kInfoOrdered] = t;
    if (t == n - 1) {
        if (c == 0) info[kInfoFeasible] = n;
        if (c <= 1) info[kInfoOrdered] = n;
    }
}

// First position whose key is not below kl (kEqual: not below or equal) in
// keys[lo, hi), the same in every lane.
template <bool kEqual>
__device__ __forceinline__ int key_bound(const uint64_t* __restrict__ keys, uint64_t kl, int lo, int hi)
{
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        const uint64_t v = keys[mid];
        if (kEqual ? v <= kl : v < kl) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The run of equal keys [tie[0], tie[1]) of each row t of the wave's block
// (rows of segment 0; other rows' values are not read) and the block's hi.
// Runs are found in the block itself; one that crosses its border is searched.
__device__ __forceinline__ void tie_runs(const uint64_t* __restrict__ keys, int n, int b, int lane,
                                         int2* __restrict__ ties, int32_t* __restrict__ hi)
{
    const int first = b * 64, end = min(n, first + 64);
    const int t = first + lane;
    const uint64_t key = keys[min(t, n - 1)];
    const uint64_t prev = (t > 0 && t < n) ? keys[t - 1] : ~key;
    const uint64_t starts = ballot(t < end && prev != key);
    const uint64_t key_last = keys[end - 1];
    const bool seg0_first = ((keys[first] >> 32) & 3u) == 0, seg0_last = ((key_last >> 32) & 3u) == 0;
    int before = first, after = end;      // start of the block's first run, end of its last
    if (!(starts & 1ull) && seg0_first) before = key_bound<false>(keys, keys[first], 0, first);
    if (seg0_last && end < n && keys[end] == key_last) after = key_bound<true>(keys, key_last, end + 1, n);
    const uint64_t upto = starts & (lane == 63 ? ~0ull : (1ull << (lane + 1)) - 1);
    const uint64_t past = starts & ~(lane == 63 ? ~0ull : (1ull << (lane + 1)) - 1);
    if (t < n)
        ties[t] = make_int2(upto ? first + 63 - __builtin_clzll(upto) : before,
                            past ? first + __builtin_ctzll(past) : after);
    if (lane == 0) hi[b] = seg0_last ? (after - 1) >> 6 : b;
}

// Rank table of one objective over a chunk of kChunk sorted rows, in sub-chunks
// of S rows: the S values in ascending order, and for each r = 0 .. S the mask
// of the rows among the r smallest (S bits).  A row p whose objective has r
// values <= p_k among the S gets "q_k <= p_k" for all of them from mask r, so a
// (row, chunk, objective) costs a search and one 64-byte read instead of 512
// compares; "q_k == p_k" is mask r without the mask of the values < p_k.
//   bytes [0, 2048): float values, sub-chunk h at 4 S h;
//   then per sub-chunk S + 1 masks of S / 8 bytes in 16-byte pieces, pieces of
//   a mask swapped by bit 3 of r where a mask has two: reads at random r then
//   spread over all LDS banks instead of half of them.
// A small S makes the table smaller and the sort below shorter, a large one the
// searches fewer (9 steps per 256 rows against 8 per 128).  S = 256 holds up
// to 8 objectives' tables in LDS (7 x 18.5 KB; the first objective, the sort
// order itself, needs none), S = 128 up to 10 (9 x 10.3 KB).
constexpr int rank_sub(int m) { return m <= 8 ? 256 : 128; }
constexpr int kRankValueBytes = kChunk * 4;
constexpr int rank_mask_bytes(int S) { return (S + 1) * (S / 8); }         // one sub-chunk's masks
__host__ __device__ constexpr int rank_table_bytes(int S)
{
    return (kRankValueBytes + (kChunk / S) * ((S + 1) * (S / 8)) + 255) / 256 * 256;
}
// the largest of an objective count's tables per chunk, for buffers sized without it
constexpr int kRankChunkBytes = 9 * rank_table_bytes(128) > 7 * rank_table_bytes(256) ? 9 * rank_table_bytes(128)
                                                                                    : 7 * rank_table_bytes(256);
static_assert(kMaxM == 10, "kRankChunkBytes covers 8 and 10 objectives");

// Byte offset of 16-byte piece j of mask r.
template <int S>
__device__ __forceinline__ int rank_piece(int r, int j)
{
    if constexpr (S == 256) return (2 * r + (j ^ ((r >> 3) & 1))) * 16;
    else return r * 16;
}

// Number of the S ascending values v[0 .. S) that are <= x (kLess: < x).
template <int S, bool kLess>
__device__ __forceinline__ int rank_search(const float* v, float x)
{
    int pos = 0;
#pragma unroll
    for (int step = S / 2; step >= 1; step >>= 1) {
        const float u = v[pos + step - 1];
        pos += (kLess ? u < x : u <= x) ? step : 0;
    }
    const float u = v[pos];
    return pos + ((kLess ? u < x : u <= x) ? 1 : 0);
}

// What nds_prep writes besides the tables.
struct PrepOut {
    float* fs;               // (m, npad) sorted objectives, 0 in padding rows
    uint64_t* valid;         // (8 Wc) rows of segment 0 per block, 0 past the last block
    int32_t* hi;             // (W)
    int2* ties;              // (n) see tie_runs
    uint64_t* gmask;         // (W) see infeasible_info
    int32_t* info;           // (2)
    int32_t* rend;           // optional (n): row ends, cleared for the dominance kernel to raise
    unsigned char* tables;   // (Wc, m - 1) rank tables of the objectives after the first
};

// One workgroup of kChunk threads: chunk qc, objective k.
template <int S>
__device__ __forceinline__ void prep_chunk(const float* __restrict__ f, int ldf, int n, int m, int npad,
                                           const int32_t* __restrict__ perm, const uint64_t* __restrict__ keys,
                                           int qc, int k, const PrepOut& O)
{
    __shared__ __align__(16) float s_v[kChunk];     // values by position
    __shared__ float s_sort[kChunk];                // values of each 64-row block, ascending
    __shared__ uint16_t s_inv[kChunk];              // position (in its sub-chunk) of each rank
    const int tid = static_cast<int>(threadIdx.x);
    const int lane = lane_id();
    const int w = wave_uniform(tid >> 6);
    const int t = qc * kChunk + tid;
    const float v = t < n ? f[static_cast<size_t>(k) * ldf + perm[t]] : 0.0f;
    if (t < npad) O.fs[static_cast<size_t>(k) * npad + t] = v;
    if (k == 0) {
        // the wave's 64 rows are block 8 qc + w
        const int b = qc * 8 + w;
        const uint64_t seg0 = ballot(t < n && ((keys[min(t, n - 1)] >> 32) & 3u) == 0);
        if (lane == 0) O.valid[b] = seg0;
        if (b * 64 < n) {
            infeasible_info(keys, n, t, O.gmask, O.info);
            tie_runs(keys, n, b, lane, O.ties, O.hi);
            if (O.rend && t < n) O.rend[t] = 0;
        }
        return;
    }
    // rows without a number are never looked up (valid masks them): any order does
    const float x = (t < n && !isnan(v)) ? v : INFINITY;
    s_v[tid] = x;
    __builtin_amdgcn_wave_barrier();
    // rank among the wave's own 64 rows, ties by position
    int own = 0;
    {
        const float4* src = reinterpret_cast<const float4*>(s_v + w * 64);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const float4 u = src[j];
            own += (u.x < x || (u.x == x && 4 * j < lane)) ? 1 : 0;
            own += (u.y < x || (u.y == x && 4 * j + 1 < lane)) ? 1 : 0;
            own += (u.z < x || (u.z == x && 4 * j + 2 < lane)) ? 1 : 0;
            own += (u.w < x || (u.w == x && 4 * j + 3 < lane)) ? 1 : 0;
        }
    }
    s_sort[w * 64 + own] = x;
    __syncthreads();
    // and among the sub-chunk: its other blocks are searched, earlier ones for
    // the values <= x, later ones for those < x
    const int h = wave_uniform(tid / S);
    const int w0 = h * (S / 64);
    int rank = own;
#pragma unroll
    for (int o = 1; o < S / 64; ++o) {
        const int b = w0 + ((w - w0 + o) & (S / 64 - 1));
        rank += (b < w) ? rank_search<64, false>(s_sort + b * 64, x) : rank_search<64, true>(s_sort + b * 64, x);
    }
    s_inv[h * S + rank] = static_cast<uint16_t>(tid & (S - 1));
    unsigned char* tab = O.tables + (static_cast<size_t>(qc) * (m - 1) + k - 1) * rank_table_bytes(S);
    reinterpret_cast<float*>(tab)[h * S + rank] = x;
    __syncthreads();
    // wave w: its 64 rows' word of every mask of their sub-chunk.  Mask r + 1
    // is mask r and the bit of the row of rank r: a prefix OR over the ranks,
    // 64 a step.
    unsigned char* masks = tab + kRankValueBytes + h * rank_mask_bytes(S);
    const int jj = w - w0;
    uint64_t before = 0;
#pragma unroll
    for (int r0 = 0; r0 < S; r0 += 64) {
        const int e = s_inv[h * S + r0 + lane];
        uint64_t acc = (e >> 6) == jj ? 1ull << (e & 63) : 0ull;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t lo = static_cast<uint32_t>(__shfl_up(static_cast<int>(acc), o));
            const uint32_t hi = static_cast<uint32_t>(__shfl_up(static_cast<int>(acc >> 32), o));
            if (lane >= o) acc |= (static_cast<uint64_t>(hi) << 32) | lo;
        }
        acc |= before;
        const int r = r0 + lane;
        *reinterpret_cast<uint64_t*>(masks + rank_piece<S>(r + 1, jj >> 1) + (jj & 1) * 8) = acc;
        before = (static_cast<uint64_t>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(acc >> 32), 63))) << 32) |
                 static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(acc), 63));
    }
    if (lane == 0) *reinterpret_cast<uint64_t*>(masks + rank_piece<S>(0, jj >> 1) + (jj & 1) * 8) = 0ull;
}

// Grid (Wc, m).  zero (optional, `words` of them): cleared on the way, for a
// later launch; mf_init: set to -1, the value the peel replaces with its result.
template <int S>
__global__ __launch_bounds__(kChunk) void nds_prep(const float* __restrict__ f, int ldf, int n, int m, int npad,
                                                   const int32_t* __restrict__ perm,
                                                   const uint64_t* __restrict__ keys, PrepOut O,
                                                   uint32_t* __restrict__ zero, int words,
                                                   int32_t* __restrict__ mf_init)
{
    if (blockIdx.x == 0 && blockIdx.y == 0) {
        for (int j = static_cast<int>(threadIdx.x); j < words; j += kChunk) zero[j] = 0u;
        if (threadIdx.x == 0) mf_init[0] = -1;
    }
    prep_chunk<S>(f, ldf, n, m, npad, perm, keys, static_cast<int>(blockIdx.x), static_cast<int>(blockIdx.y), O);
}

// Mask r of sub-chunk h of a table.
template <int S>
__device__ __forceinline__ void rank_mask(const unsigned char* tab, int h, int r, uint64_t (&out)[S / 64])
{
    const unsigned char* masks = tab + kRankValueBytes + h * rank_mask_bytes(S);
#pragma unroll
    for (int j = 0; j < S / 128; ++j) {
        const ulonglong2 u = *reinterpret_cast<const ulonglong2*>(masks + rank_piece<S>(r, j));
        out[2 * j] = u.x;
        out[2 * j + 1] = u.y;
    }
}

// The first r of the 64 rows of a word (r clamped to 0 .. 64).
__device__ __forceinline__ uint64_t first_rows(int r)
{
    return r <= 0 ? 0ull : r >= 64 ? ~0ull : (1ull << r) - 1;
}

// A chunk whose f0 ties with row block pb, or that holds pb itself (or rows
// after it): every objective's <=, without the rows equal in all of them.  f0
// is the sort order: rows before `tie`'s end are <=, those in it equal.
template <int M, int S>
__device__ __forceinline__ void tied_bits(const unsigned char* s_tab, const float (&pv)[M], int2 tie, int q0,
                                          uint64_t (&bits)[8])
{
#pragma unroll
    for (int h = 0; h < kChunk / S; ++h) {
        uint64_t eq[S / 64], le[S / 64], lt[S / 64];
#pragma unroll
        for (int j = 0; j < S / 64; ++j) {
            const int b = h * (S / 64) + j;
            const uint64_t le0 = first_rows(tie.y - q0 - b * 64);
            bits[b] &= le0;
            eq[j] = le0 & ~first_rows(tie.x - q0 - b * 64);
        }
#pragma unroll 1
        for (int k = 1; k < M; ++k) {
            const unsigned char* tab = s_tab + (k - 1) * rank_table_bytes(S);
            float x = pv[M > 1 ? 1 : 0];
#pragma unroll
            for (int c = 2; c < M; ++c) x = (k == c) ? pv[c] : x;
            const float* v = reinterpret_cast<const float*>(tab) + h * S;
            rank_mask<S>(tab, h, rank_search<S, false>(v, x), le);
            rank_mask<S>(tab, h, rank_search<S, true>(v, x), lt);
#pragma unroll
            for (int j = 0; j < S / 64; ++j) {
                bits[h * (S / 64) + j] &= le[j];
                eq[j] &= le[j] & ~lt[j];
            }
        }
#pragma unroll
        for (int j = 0; j < S / 64; ++j) bits[h * (S / 64) + j] &= ~eq[j];
    }
}

// Four lanes of a quad with four 16-byte pieces each (words 4j .. 4j + 3):
// afterwards lane q holds piece q of the quad's lanes 0 .. 3, by two rounds of
// exchange.
template <int kCtrl>
__device__ __forceinline__ void quad_trade(uint32_t& a, uint32_t& b, bool high)
{
    const uint32_t got = static_cast<uint32_t>(
        __builtin_amdgcn_mov_dpp(static_cast<int>(high ? a : b), kCtrl, 0xf, 0xf, true));
    a = high ? got : a;
    b = high ? b : got;
}

__device__ __forceinline__ void quad_transpose(uint32_t (&w)[16], int lane)
{
    constexpr int kXor1 = 0xB1, kXor2 = 0x4E;   // quad_perm [1,0,3,2] and [2,3,0,1]
    const bool odd = lane & 1, top = lane & 2;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        quad_trade<kXor1>(w[i], w[4 + i], odd);
        quad_trade<kXor1>(w[8 + i], w[12 + i], odd);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        quad_trade<kXor2>(w[i], w[8 + i], top);
        quad_trade<kXor2>(w[4 + i], w[12 + i], top);
    }
}

// One workgroup: chunk qc against the row blocks [pb0, pb1), a row block per
// wave at a time.  s_tab: LDS for the tables of objectives 1 .. M - 1.  A chunk
// that ends before block pb with no f0 tie has f0 strictly below pb's, so its
// words need objectives 1 .. M - 1 only.  rend (optional): each row's end, one
// past its last non-zero word, raised with atomicMax.
//
// Bound: the bitmask's write (n^2 / 16 bytes).  Rows of one wave hit unrelated
// ranks, so searches and mask reads go to LDS, where a random 16-byte read of a
// wave costs about 12 cycles.
template <int M>
__device__ __forceinline__ void dom_chunk(const float* __restrict__ fs, int npad, int n, int W, int Wc,
                                          const uint64_t* __restrict__ valid, const int32_t* __restrict__ hi,
                                          const int2* __restrict__ ties, const unsigned char* __restrict__ tables,
                                          uint64_t* __restrict__ B, int32_t* __restrict__ rend, int qc, int pb0, int pb1, unsigned char* s_tab)
{
    constexpr int S = rank_sub(M);
    constexpr int kTab = rank_table_bytes(S);
    constexpr int kThreads = dom_threads(M);
    if (hi[pb1 - 1] < 8 * qc) return;            // hi ascends: no row block here reaches the chunk
    if constexpr (M > 1) {
        const uint4* src = reinterpret_cast<const uint4*>(tables + static_cast<size_t>(qc) * (M - 1) * kTab);
        uint4* dst = reinterpret_cast<uint4*>(s_tab);
#pragma unroll 4
        for (int j = static_cast<int>(threadIdx.x); j < (M - 1) * kTab / 16; j += kThreads) dst[j] = src[j];
        __syncthreads();
    }
    const int lane = lane_id();
    uint64_t vq[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) vq[j] = ld_uniform(valid, static_cast<size_t>(qc) * 8 + j);
    const int tie_to = ld_uniform(hi, min(8 * qc + 7, W - 1));   // last block that ties with the chunk
    for (int pb = pb0 + wave_uniform(static_cast<int>(threadIdx.x >> 6)); pb < pb1; pb += kThreads / 64) {
        if (ld_uniform(hi, pb) < 8 * qc) continue;
        const uint64_t vp = ld_uniform(valid, pb);
        // rows outside segment 0: feasible ones with a NaN objective have no
        // dominators, infeasible ones no words that are read
        const int p = pb * 64 + lane;
        float pv[M];
#pragma unroll
        for (int k = 0; k < M; ++k) pv[k] = fs[static_cast<size_t>(k) * npad + p];
        const bool in0 = (vp >> lane) & 1ull;
        uint64_t bits[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) bits[j] = in0 ? vq[j] : 0ull;
        if (8 * qc + 7 < pb && tie_to < pb) {
#pragma unroll
            for (int k = 1; k < M; ++k) {
                const unsigned char* tab = s_tab + (k - 1) * kTab;
                int r[kChunk / S];
#pragma unroll
                for (int h = 0; h < kChunk / S; ++h)
                    r[h] = rank_search<S, false>(reinterpret_cast<const float*>(tab) + h * S, pv[k]);
#pragma unroll
                for (int h = 0; h < kChunk / S; ++h) {
                    uint64_t le[S / 64];
                    rank_mask<S>(tab, h, r[h], le);
#pragma unroll
                    for (int j = 0; j < S / 64; ++j) bits[h * (S / 64) + j] &= le[j];
                }
            }
        } else {
            tied_bits<M, S>(s_tab, pv, ties[min(p, n - 1)], qc * kChunk, bits);
        }
        // a lane quad trades pieces so that it writes whole 64-byte rows, one a
        // store, instead of 16 bytes of four rows: a quarter of the L2 requests
        uint32_t w[16];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            w[2 * j] = static_cast<uint32_t>(bits[j]);
            w[2 * j + 1] = static_cast<uint32_t>(bits[j] >> 32);
        }
        quad_transpose(w, lane);
        uint4* dst = reinterpret_cast<uint4*>(B + ((static_cast<size_t>(pb) * Wc + qc) * 64 + (lane & ~3)) * 8) + (lane & 3);
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[j * 4] = make_uint4(w[4 * j], w[4 * j + 1], w[4 * j + 2], w[4 * j + 3]);
        if (rend && p < n) {
            int top = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (bits[j]) top = j + 1;
            if (top) atomicMax(&rend[p], qc * 8 + top);
        }
    }
}

// LDS of the dominance kernel: the tables of objectives 1 .. m - 1.
constexpr size_t dom_lds_bytes(int m) { return static_cast<size_t>(m > 1 ? m - 1 : 0) * rank_table_bytes(rank_sub(m)); }

// Grid (ceil(W / seg), Wc).
template <int M>
__global__ __launch_bounds__(dom_threads(M)) void nds_dominance(const float* __restrict__ fs, int npad, int n, int W,
                                                            int Wc, const uint64_t* __restrict__ valid,
                                                            const int32_t* __restrict__ hi,
                                                            const int2* __restrict__ ties,
                                                            const unsigned char* __restrict__ tables,
                                                            uint64_t* __restrict__ B, int32_t* __restrict__ rend,
                                                            int seg)
{
    extern __shared__ __align__(16) unsigned char s_tab[];
    const int pb0 = static_cast<int>(blockIdx.x) * seg;
    dom_chunk<M>(fs, npad, n, W, Wc, valid, hi, ties, tables, B, rend, static_cast<int>(blockIdx.y), pb0,
                 min(pb0 + seg, W), s_tab);
}

// Row blocks per dominance workgroup: enough workgroups to fill the chip, and
// enough row blocks in each to pay for loading its tables.  1024 workgroups
// against 512 and 2048, in us: 33.4 / 34.3 / 29.8 at 32768 rows, M = 3, 160 / 150 /
// 160 at M = 10; 521 / 522 / 540 at 65536, M = 10; within 1 % below 32768 rows.  At
// most 64 row blocks against 32 and 128: 101 / 96 / 99 at 65536, M = 3, 521 / 541 / 522
// at M = 10; at 131072 rows 32 is faster (362 / 287 / 342, 2079 / 1631 / 1999).
int dom_segment(int W, int Wc, int m)
{
    const int waves = dom_threads(m) / 64;
    const long long units = static_cast<long long>(W) * Wc / 2;
    const long long per = units / 1024 / waves * waves;
    return static_cast<int>(std::max<long long>(waves, std::min<long long>(64, per)));
}

// Peel state (device), u32 words: [0, kBarWords) group barrier,
// [kPeelTotal] total assigned, [kPeelTotal + 1] last round, [kPeelTotal + 2]
// spare output word, [kPeelTotal + 4 + (k & 1)] the total as of the barrier
// ending round k (snapshot read by every block).  A0 / A1: assigned-set
// bitsets in sorted order (W words each), double-buffered across rounds.
//
// Workgroup g owns row blocks g, g + G, g + 2G, ... (G workgroups, spread over
// the whole sort order).  A row's dominator words are scanned from its last
// one (its own block, or its row end) down to word 0.  Each owned row keeps,
// in LDS for the whole launch, its blocking word c (the highest word of its
// dominator row that held an unassigned dominator when last looked at) and
// rem, the dominators of word c that were still unassigned then.  Round k:
//   A  rem &= ~A[c] against the set assigned before round k, a lane per row,
//      in LDS alone.  A row with rem left stays blocked; the others go to the
//      workgroup's queue in LDS as (row, c).
//   B  the workgroup's 16 waves scan the queued rows downwards from c in sweeps
//      of one round trip per row, each until it meets its next blocking word
//      (the row keeps (c, rem)) or runs out of words (front k).  The first
//      sweep reads kFirstLanes chunks a row, which ends most scans; the later
//      ones as many as the queue leaves lanes for (a wave, 512 words, for 16
//      rows or fewer), as a row that got past the first mostly runs out.
// Why downwards: the dominators next to a row in the sort order (f0 just
// below its own) are on average much deeper than those with a small f0, so the
// blocker found first stays unassigned for most of the rounds before the row's
// own front.  On the merged objectives of the N = 32768, M = 3, D = 1024 run
// (generation 25, 24 fronts) the rows are scanned 176 thousand times over the
// launch instead of 1.23 million from word 0 up, and read 121 MB of words
// instead of 225 MB.
// A scan ends at the first word with an unassigned feasible row: all below it are
// assigned.  That word is looked for in the sorts of many fronts alone (every 8th
// round from the 64th on, and not by a group of one), whose assigned set grows in
// sort order: with every scan down to word 0 a row's last scan reads its whole
// width, one front after another.  One objective, a front a row: 65536 rows 397
// -> 282 ms, 2112 rows 8.9 -> 7.6 ms; sorts of few fronts as before.
// Rows, cursors, fronts and tasks never leave their workgroup (the fronts go
// out once, when the peel stops); only the assigned set and the total cross
// workgroups, at the one grid barrier per round.
//
// Everything the workgroups exchange inside the launch (barrier words,
// totals, the assigned sets) is accessed with device-scope atomics, which the
// hardware keeps coherent across the XCDs' L2 caches; nothing else written in
// the launch is read in it.  The barrier therefore orders only those
// accesses (coherent_barrier) and does not write back or invalidate the L2.
struct PeelArgs {
    const uint64_t* B;
    const int32_t* hi;       // (W,) last word block of each row block
    const int32_t* perm;     // (n,) sorted position -> input index
    int n, W, Wc, stop_at;
    int blocks_per_group;    // ceil(W / group size)
    int32_t* fronts;         // (n,) out, input order
    uint64_t* A0;
    uint64_t* A1;
    uint32_t* state;
    int32_t* out_max_front;  // (1,) out: last front, kPeelFailed when a bounded wait gave up
    const int32_t* rend;     // (n,) optional: one past each row's last non-zero word (sorted order)
    uint32_t spin_limit;     // polls before a barrier wait gives up
    uint32_t* error;         // optional sticky flag: set to 1 when a bounded wait gave up
    const uint64_t* gmask;   // (W,) first rows of each distinct infeasible cv (infeasible_info)
    const int32_t* info;     // feasible rows, end of the infeasible rows whose cv is a number
};

constexpr int32_t kPeelFailed = -2;
constexpr int kPeelTotal = kBarWords;
constexpr int kPeelStateWords = kBarWords + 16;
static_assert(kPeelStateWords <= kBatchPeelStateWords, "batched peel state too small");
constexpr int kPeelThreads = 1024;
constexpr int kPeelWaves = kPeelThreads / 64;
constexpr int kFirstLanes = 4;      // lanes (chunks) per row of the first sweep
constexpr int kMinLanes = 8;        // and of the later ones, at least
constexpr int kLowFrom = 64;        // round from which words assigned throughout are looked for,
constexpr int kLowEvery = 8;        // once in so many rounds

// LDS layout of the peel (dynamic): s_A (W u64), s_next (bpg u64), s_rem
// (64 bpg u64), s_task (2 x 64 bpg rows and cursors), s_cur and s_front (64 bpg
// int each).
__host__ __device__ __forceinline__ size_t peel_lds_bytes(int W, int bpg)
{
    const size_t rows = static_cast<size_t>(bpg) * 64;
    return (static_cast<size_t>(W) + 7) / 8 * 64 + static_cast<size_t>(bpg) * 8 + rows * 32;
}

// One trip: groups of L lanes (a power of two) of a wave, one queued row each.
// Lane sl of a row's group reads chunk (c - 1) / 8 - sl of the row, a 64-byte
// segment; words from c on count as clear.  Returns true when the row meets a
// word holding an unassigned dominator (its index in c, its unassigned bits in
// rem, the same in every lane of the group); otherwise c moves below the words
// read (to 0 when they run out).  Every lane of the wave calls it; lanes of a
// group without a row pass has = false.  c >= 1 for a row.
__device__ __forceinline__ bool peel_trip(const uint64_t* __restrict__ B, int Wc, int p, int& c,
                                          const uint64_t* s_A, int lane, int L, bool has, uint64_t& rem)
{
    const int sl = lane & (L - 1);
    const int shift = lane - sl;
    const int ch0 = (c - 1) >> 3;
    const int ch = ch0 - sl;
    const bool in = has && ch >= 0;
    ulonglong2 v[4];
    if (in) {
        const ulonglong2* src = reinterpret_cast<const ulonglong2*>(B + bword_index(p, ch * 8, Wc));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = src[i];
    }
    // the assigned-set words, read while the row's words are in flight
    const int w0 = in ? ch * 8 : 0;
    uint64_t am[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) am[i] = s_A[w0 + i];
    int fw = -1;
    uint64_t hit = 0;
    if (in) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint64_t x = ((i & 1) ? v[i >> 1].y : v[i >> 1].x) & ~am[i];
            if (w0 + i < c && x != 0) { fw = w0 + i; hit = x; }
        }
    }
    // the row's highest blocking word: from its lowest lane that has one
    const uint64_t gmask = (L == 64) ? ~0ull : ((1ull << L) - 1);
    const uint64_t gm = (ballot(fw >= 0) >> shift) & gmask;
    const int src = shift + (gm ? __builtin_ctzll(gm) : 0);
    const int bw = __shfl(fw, src);
    const uint32_t lo = static_cast<uint32_t>(__shfl(static_cast<int>(hit), src));
    const uint32_t hi = static_cast<uint32_t>(__shfl(static_cast<int>(hit >> 32), src));
    if (gm) {
        c = bw;
        rem = (static_cast<uint64_t>(hi) << 32) | lo;
        return true;
    }
    c = max((ch0 + 1 - L) * 8, 0);
    return false;
}

// Records a failed bounded wait: the run's front count becomes kPeelFailed
// and the optional sticky flag is set.
__device__ __forceinline__ void peel_fail(const PeelArgs& P)
{
    if (threadIdx.x != 0) return;
    __hip_atomic_exchange(P.out_max_front, kPeelFailed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (P.error) __hip_atomic_fetch_or(P.error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The end of the peel, once the feasible rows' fronts (0 .. F - 1) are known or
// the stop rule has ended them: with `tail`, the infeasible rows get front
// F + (index of their distinct cv) as long as fewer than stop_at rows are
// assigned before (at least one front when no row is feasible), rows with a
// NaN cv front F.  Every owned row's front goes out in input order; block 0
// of the group leaves the last front.  s_A (free by now) takes the prefix
// counts of the first rows.
__device__ __forceinline__ void peel_finish(const PeelArgs& P, int g, int G, int nf, int ne, int last_front,
                                            bool tail, const int* s_front, uint64_t* s_A)
{
    const int lane = lane_id();
    const int lw = wave_uniform(static_cast<int>(threadIdx.x >> 6));
    int cut = nf;                 // first infeasible row that is not assigned
    int* s_start = reinterpret_cast<int*>(s_A);   // (W) first rows before each block
    __shared__ int s_cut, s_base[kPeelWaves], s_run;
    if (tail) {
        // the first group that begins at or after `from` finds enough rows assigned
        const int from = max(nf + 1, P.stop_at - (P.n - ne));
        if (threadIdx.x == 0) { s_cut = ne; s_run = 0; }
        __syncthreads();
        for (int w0 = 0; w0 < P.W; w0 += kPeelThreads) {
            const int w = w0 + static_cast<int>(threadIdx.x);
            const uint64_t m = w < P.W ? P.gmask[w] : 0ull;
            uint64_t late = m;
            if (w * 64 < from) late = (from - w * 64 >= 64) ? 0ull : m & (~0ull << (from - w * 64));
            if (late) atomicMin(&s_cut, w * 64 + __builtin_ctzll(late));
            // prefix of the counts over the block's words
            const int cnt = __builtin_popcountll(m);
            int incl = cnt;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int u = __shfl_up(incl, o);
                if (lane >= o) incl += u;
            }
            if (lane == 63) s_base[lw] = incl;
            __syncthreads();
            int before = s_run;
            for (int v = 0; v < lw; ++v) before += s_base[v];
            if (w < P.W) s_start[w] = before + incl - cnt;
            __syncthreads();
            if (threadIdx.x == 0) {
                int all = s_run;
                for (int v = 0; v < kPeelWaves; ++v) all += s_base[v];
                s_run = all;
            }
            __syncthreads();
        }
        cut = s_cut;
    }
    const auto groups_to = [&](int t) {           // first rows at sorted positions <= t
        const uint64_t m = P.gmask[t >> 6];
        const int b = t & 63;
        return s_start[t >> 6] + __builtin_popcountll(m & (b == 63 ? ~0ull : (1ull << (b + 1)) - 1));
    };
    if (g == 0 && threadIdx.x == 0) {
        int last = last_front;
        if (tail && ne > nf) last += groups_to(cut - 1);
        else if (tail && P.n > ne) last += 1;
        // the launch before the peel set the output to -1; a block that gave
        // up in this last barrier may already have marked the run failed, and
        // that mark stays
        int32_t expected = -1;
        __hip_atomic_compare_exchange_strong(P.out_max_front, &expected, last, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
    }
    for (int j = lw; j < P.blocks_per_group; j += kPeelWaves) {
        const int p = (g + j * G) * 64 + lane;
        if (p >= P.n) continue;
        int fr = s_front[j * 64 + lane];
        if (tail && p >= nf) fr = p >= ne ? last_front + 1 : p < cut ? last_front + groups_to(p) : -1;
        P.fronts[P.perm[p]] = fr;
    }
}

// One peel over the G blocks of a group; g is this block's rank.  Returns
// false when a barrier gave up (the launch is broken; the block exits after
// recording the failure).
__device__ __forceinline__ bool peel_body(const PeelArgs& P, int g, int G, uint64_t* s_dyn)
{
    const int nblk = P.W;
    const int bpg = P.blocks_per_group;
    uint64_t* s_A = s_dyn;                                          // (W) assigned before this round, whole chunks
    uint64_t* s_next = s_A + (nblk + 7) / 8 * 8;                    // (bpg) rows of own blocks assigned this round
    const int rows = bpg * 64;
    uint64_t* s_rem = s_next + bpg;                                 // (64 bpg) unassigned bits of the blocking word
    int2* s_task = reinterpret_cast<int2*>(s_rem + rows);           // (2 x 64 bpg) queued (row, cursor)
    int* s_cur = reinterpret_cast<int*>(s_task + 2 * static_cast<size_t>(rows));   // (64 bpg) blocking word
    int* s_front = s_cur + rows;                                    // (64 bpg) front of each owned row
    __shared__ int s_nq[3];         // queue lengths, rotating over the sweeps of phase B
    __shared__ int s_count;
    __shared__ int s_low;           // first word with an unassigned feasible row
    const int lane = lane_id();
    const int lw = wave_uniform(static_cast<int>(threadIdx.x >> 6));
    uint32_t phase = 0;
    const int nf = P.info[kInfoFeasible], ne = P.info[kInfoOrdered];

    for (int j = lw; j < bpg; j += kPeelWaves) {
        const int rb = g + j * G;
        s_cur[j * 64 + lane] = 0;               // words 0 .. cur - 1 may hold unassigned dominators
        s_rem[j * 64 + lane] = 0ull;
        s_front[j * 64 + lane] = -1;
        if (lane == 0) s_next[j] = 0ull;
        if (rb >= nblk) continue;
        const int p = rb * 64 + lane;
        s_cur[j * 64 + lane] = (P.rend && p < P.n) ? P.rend[p] : P.hi[rb] + 1;
        if (G > 1 && lane == 0) { st_relaxed_u64(&P.A0[rb], 0ull); st_relaxed_u64(&P.A1[rb], 0ull); }
    }
    // a group of one keeps the assigned set and the total to itself, in LDS
    if (G == 1) {
        for (int w = threadIdx.x; w < nblk; w += kPeelThreads) s_A[w] = 0ull;
        __syncthreads();
    } else if (!coherent_barrier(P.state, g, G, phase, P.spin_limit)) {
        peel_fail(P);
        return false;
    }
    if (nf == 0) {
        peel_finish(P, g, G, nf, ne, -1, true, s_front, s_A);
        return true;
    }

    int total_prev = 0, low = 0;    // words below low hold no unassigned feasible row
    for (int k = 0;; ++k) {
        const uint64_t* Acur = (k & 1) ? P.A1 : P.A0;
        uint64_t* Anext = (k & 1) ? P.A0 : P.A1;
        if (G > 1)
            for (int w = threadIdx.x; w < nblk; w += kPeelThreads) s_A[w] = ld_relaxed_u64(&Acur[w]);
        const int turn = (G > 1 && k >= kLowFrom) ? k & (kLowEvery - 1) : 0;
        if (turn == kLowEvery - 1) {
            for (int w = threadIdx.x; w < nblk; w += kPeelThreads) {
                const uint64_t open = ballot((first_rows(nf - w * 64) & ~s_A[w]) != 0);
                if (open && lane == __builtin_ctzll(open)) atomicMin(&s_low, w);
            }
        }
        if (threadIdx.x == 0) {
            s_count = 0; s_nq[0] = 0; s_nq[1] = 0;
            if (turn == kLowEvery - 2) s_low = nblk;
        }
        __syncthreads();
        if (turn == kLowEvery - 1) low = s_low;

        // ---- phase A: lane per row, in LDS
        int my_new = 0;
        for (int j = lw; j < bpg; j += kPeelWaves) {
            const int rb = g + j * G;
            if (rb >= nblk) break;
            const uint64_t amask = s_A[rb];
            const int p = rb * 64 + lane;
            const int slot = j * 64 + lane;
            const bool live = (p < nf) && !((amask >> lane) & 1ull);
            bool ready = false, queued = false;
            int cur = 0;
            if (live) {
                cur = s_cur[slot];
                // still blocked while dominators of its blocking word are
                // unassigned (before its first scan rem is 0 and cur may be W)
                const uint64_t rem = s_rem[slot] & ~s_A[min(cur, nblk - 1)];
                s_rem[slot] = rem;
                ready = (rem == 0) && cur <= low;
                queued = (rem == 0) && !ready;
            }
            if (ready) s_front[slot] = k;
            const uint64_t ready_m = ballot(ready);
            const uint64_t task_m = ballot(queued);
            if (task_m) {
                int base = 0;
                if (lane == 0) base = atomicAdd(&s_nq[0], __builtin_popcountll(task_m));
                base = __builtin_amdgcn_readfirstlane(base);
                if (queued) {
                    const int below = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
                        static_cast<uint32_t>(task_m >> 32),
                        __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(task_m), 0u)));
                    s_task[base + below] = make_int2(slot, cur);
                }
            }
            if (lane == 0) {
                s_next[j] = ready_m;
                my_new += __builtin_popcountll(ready_m);
            }
        }

        // ---- phase B: sweep s takes queue s % 2 (length s_nq[s % 3]) and
        // queues the rows still clear in the other
        for (int sw = 0;; ++sw) {
            __syncthreads();
            const int nq = s_nq[sw % 3];
            if (nq == 0) break;
            if (threadIdx.x == 0) s_nq[(sw + 2) % 3] = 0;
            int L = kFirstLanes;
            if (sw > 0) {
                L = 64;
                while (L > kMinLanes && nq > kPeelWaves * (64 / L)) L >>= 1;
            }
            const int gpw = 64 / L;
            const int2* q_in = s_task + (sw & 1) * static_cast<size_t>(rows);
            int2* q_out = s_task + ((sw + 1) & 1) * static_cast<size_t>(rows);
            for (int t0 = lw * gpw; t0 < nq; t0 += kPeelWaves * gpw) {
                const int t = t0 + lane / L;
                const bool has = t < nq;
                const int2 rec = has ? q_in[t] : make_int2(0, 1);
                const int slot = rec.x;
                int c = rec.y;
                const int p = (g + (slot >> 6) * G) * 64 + (slot & 63);
                uint64_t rem = 0;
                const bool blocked = peel_trip(P.B, P.Wc, p, c, s_A, lane, L, has, rem);
                if (has && (lane & (L - 1)) == 0) {
                    if (blocked) {
                        s_cur[slot] = c;
                        s_rem[slot] = rem;
                    } else if (c <= low) {
                        s_front[slot] = k;
                        atomicOr(reinterpret_cast<unsigned long long*>(&s_next[slot >> 6]),
                                 static_cast<unsigned long long>(1ull << (slot & 63)));
                        ++my_new;
                    } else {
                        q_out[atomicAdd(&s_nq[(sw + 1) % 3], 1)] = make_int2(slot, c);
                    }
                }
            }
        }
        if (my_new) atomicAdd(&s_count, my_new);
        __syncthreads();
        for (int j = threadIdx.x; j < bpg; j += kPeelThreads) {
            const int rb = g + j * G;
            if (rb < nblk) {
                const uint64_t now = s_A[rb] | s_next[j];
                if (G == 1) s_A[rb] = now;
                else st_relaxed_u64(&Anext[rb], now);
            }
            s_next[j] = 0ull;
        }
        if (G > 1 && threadIdx.x == 0 && s_count)
            __hip_atomic_fetch_add(&P.state[kPeelTotal], static_cast<uint32_t>(s_count), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
        // the running total is read from the snapshot block 0 takes inside
        // the barrier: a block that reads late must not see counts that
        // faster blocks already add for the next round, or the blocks could
        // disagree about stopping and strand each other at the next barrier
        const int snap = kPeelTotal + 4 + (k & 1);
        int total = total_prev + s_count;
        if (G == 1) {
            __syncthreads();
        } else {
            if (!coherent_barrier(P.state, g, G, phase, P.spin_limit, kPeelTotal, snap)) {
                peel_fail(P);
                return false;
            }
            total = static_cast<int>(ld_relaxed_u32(&P.state[snap]));
        }
        if (total >= P.stop_at || total == total_prev || total >= nf) {
            // the infeasible rows follow once every feasible one is assigned
            peel_finish(P, g, G, nf, ne, (total == total_prev) ? k - 1 : k, total >= nf && total < P.stop_at, s_front,
                        s_A);
            return true;
        }
        total_prev = total;
    }
}

__global__ __launch_bounds__(kPeelThreads) void nds_peel(PeelArgs P)
{
    extern __shared__ uint64_t s_dyn[];
    const int G = static_cast<int>(gridDim.x);
    __builtin_assume(G > 1);           // one workgroup goes to nds_peel_one
    peel_body(P, static_cast<int>(blockIdx.x), G, s_dyn);
}

// The same with one workgroup, which needs no grid barrier and so no
// cooperative launch (that leaves the device idle for about 10 us on each
// side).  Up to kOneGroupBlocks row blocks its 16 waves hold two blocks each,
// and the rounds cost less than the barriers of more workgroups.  Peel stage in us,
// one workgroup / cooperating ones (shell of many fronts, then one front): 184
// rows 7 / 28; 2048 rows M = 2 78 / 132, 19 / 32, M = 10 11 / 29, 9 / 28; 3072 rows M = 3
// 63 / 63, 35 / 33, M = 10 14 / 30, 10 / 28; 4096 rows M = 3 88 / 71, 52 / 33, M = 10 18 / 30,
// 12 / 29: above 2048 rows it depends on the fronts.
constexpr int kOneGroupBlocks = 32;

__global__ __launch_bounds__(kPeelThreads) void nds_peel_one(PeelArgs P)
{
    extern __shared__ uint64_t s_dyn[];
    peel_body(P, 0, 1, s_dyn);
}

// ---------------------------------------------------------------- batched --
// The NDS of every instance of a batch: mode 0 ranks the n parents (slot cur)
// into fronts[fcur], mode 1 the 2n merged rows into fronts_mix and meta[0].  Keys carry the instance index above the 34 NDS bits, so one
// stable sort orders every instance's rows exactly as its own sort would.
struct BRows {
    const float* f;
    const float* cv;
    int rows;
    long long key_off;
    int32_t* fronts;
};

__device__ __forceinline__ BRows brows(const BInst& I, int mode)
{
    BRows r;
    if (mode == 0) {
        r.f = I.f[I.cur]; r.cv = I.cv[I.cur]; r.rows = I.n; r.key_off = I.key_off_n; r.fronts = I.fronts[I.fcur];
    } else {
        r.f = I.fm; r.cv = I.cvm; r.rows = I.nm; r.key_off = I.key_off; r.fronts = I.fronts_mix;
    }
    return r;
}

__global__ void b_nds_keys(const BInst* __restrict__ insts, BMap mp, int mode, uint64_t* __restrict__ keys,
                           int32_t* __restrict__ vals)
{
    int local;
    const int i = bmap_find(mp, static_cast<int>(blockIdx.x), local);
    const BInst& I = insts[i];
    const BRows R = brows(I, mode);
    const int s = local * 256 + static_cast<int>(threadIdx.x);
    if (s >= R.rows) return;
    keys[R.key_off + s] = nds_key_of(R.f, R.rows, R.cv, s, I.m) | (static_cast<uint64_t>(i) << kKeyBits);
    vals[R.key_off + s] = s;
}

// nds_prep of every instance: Wc x m workgroups each.
__global__ __launch_bounds__(kChunk) void b_nds_prep(const BInst* __restrict__ insts, BMap mp, int mode,
                                                     const uint64_t* __restrict__ keys_sorted,
                                                     const int32_t* __restrict__ vals_sorted)
{
    int local;
    const int i = bmap_find(mp, static_cast<int>(blockIdx.x), local);
    const BInst& I = insts[i];
    const BRows R = brows(I, mode);
    const int W = (R.rows + 63) / 64;
    const int qc = local / I.m, k = local % I.m;
    const int t = qc * kChunk + static_cast<int>(threadIdx.x);
    const int32_t* perm = vals_sorted + R.key_off;
    if (k == 0 && t < R.rows) I.perm[t] = perm[t];
    const PrepOut O{I.fs, I.valid, I.hi, I.ties, I.gmask, I.ninfo, I.m >= kRowEndMinM ? I.rend : nullptr, I.tables};
    if (rank_sub(I.m) == 256) prep_chunk<256>(R.f, R.rows, R.rows, I.m, W * 64, perm, keys_sorted + R.key_off, qc, k, O);
    else prep_chunk<128>(R.f, R.rows, R.rows, I.m, W * 64, perm, keys_sorted + R.key_off, qc, k, O);
}

// nds_dominance of the instances with M objectives: Wc x ceil(W / kBatchDomSeg)
// workgroups each.
template <int M>
__global__ __launch_bounds__(dom_threads(M)) void b_nds_dominance(const BInst* __restrict__ insts, BMap mp, int mode)
{
    extern __shared__ __align__(16) unsigned char s_tab[];
    int local;
    const int i = bmap_find(mp, static_cast<int>(blockIdx.x), local);
    const BInst& I = insts[i];
    const BRows R = brows(I, mode);
    const int W = (R.rows + 63) / 64, Wc = (W + 7) / 8;
    const int qc = local % Wc, pb0 = local / Wc * kBatchDomSeg;
    dom_chunk<M>(I.fs, W * 64, R.rows, W, Wc, I.valid, I.hi, I.ties, I.tables, I.B,
                 M >= kRowEndMinM ? I.rend : nullptr, qc, pb0, min(pb0 + kBatchDomSeg, W), s_tab);
}

// Where a batched peel leaves the index of its last front: the selection's
// meta word for the merged rows, a spare peel-state word for the parents.
__device__ __forceinline__ int32_t* peel_max_front(const BInst& I, int mode)
{
    return mode == 1 ? I.meta : reinterpret_cast<int32_t*>(I.pstate + kPeelTotal + 2);
}

// Front peeling of every instance of a batch in one cooperative launch.  The
// blocks form groups; each group peels its instances one after another
// (peel_body, with the group barrier on the instance's own state words), so
// a large instance gets many blocks and small ones share single blocks.
// Jobs of block w: jobs[first[w] .. first[w + 1]) as (instance, rank, group size).
__global__ __launch_bounds__(kPeelThreads) void b_nds_peel_groups(const BInst* __restrict__ insts, int mode,
                                                                 const int* __restrict__ first,
                                                                 const int* __restrict__ jobs, uint32_t spin_limit,
                                                                 uint32_t* error)
{
    extern __shared__ uint64_t s_dyn[];
    const int w = static_cast<int>(blockIdx.x);
    const int j1 = first[w + 1];
    for (int j = first[w]; j < j1; ++j) {
        const int i = jobs[3 * j], g = jobs[3 * j + 1], G = jobs[3 * j + 2];
        const BInst& I = insts[i];
        const BRows R = brows(I, mode);
        const int W = (R.rows + 63) / 64, Wc = (W + 7) / 8;
        PeelArgs P{I.B, I.hi, I.perm, R.rows, W, Wc, mode == 1 ? I.n : R.rows, (W + G - 1) / G, R.fronts,
                   I.A, I.A + W, I.pstate, peel_max_front(I, mode), I.m >= kRowEndMinM ? I.rend : nullptr,
                   spin_limit, error, I.gmask, I.ninfo};
        __syncthreads();
        if (!peel_body(P, g, G, s_dyn)) return;
    }
}

// Clears the peel state words of the instances in `state` (barrier flags and
// totals start at zero) and sets their front-count outputs to -1.
__global__ void b_peel_reset(const BInst* __restrict__ insts, int mode, int state)
{
    const BInst& I = insts[blockIdx.x];
    if (I.state != state) return;
    for (int t = threadIdx.x; t < kPeelStateWords; t += blockDim.x) I.pstate[t] = 0u;
    __syncthreads();
    if (threadIdx.x == 0) peel_max_front(I, mode)[0] = -1;
}


constexpr int kMaxWords = 4096;   // n <= 262144: the assigned set fits in 32 KiB of LDS

// Polls before a peel barrier gives up (kSpinLimit unless a test lowers it
// with moea_debug_set_spin_limit to make the bounded wait give up on purpose).
std::atomic<uint32_t> g_spin_limit{kSpinLimit};

uint32_t peel_spin_limit() { return g_spin_limit.load(std::memory_order_relaxed); }

struct NdsLayout {
    uint64_t* B;
    uint64_t* keys_in;
    uint64_t* keys_out;
    int32_t* vals_in;
    int32_t* perm;
    void* sort_temp;
    size_t sort_bytes;
    float* fs;
    unsigned char* tables;
    int32_t* hi;
    int2* ties;
    uint64_t* valid;
    uint64_t* A0;
    uint64_t* A1;
    uint32_t* state;
    int32_t* rend;
    uint64_t* gmask;
    int32_t* info;
};

size_t carve_nds(void* ws, int n, NdsLayout& L)
{
    const int W = ceil_div(n, 64);
    const int Wc = ceil_div(W, 8);
    const int npad = W * 64;
    Carve c(ws, ~size_t{0});
    L.B = c.take<uint64_t>(static_cast<size_t>(W) * Wc * 8 * 64);
    L.keys_in = c.take<uint64_t>(n);
    L.keys_out = c.take<uint64_t>(n);
    L.vals_in = c.take<int32_t>(n);
    L.perm = c.take<int32_t>(n);
    L.sort_bytes = sort_pairs_temp_bytes(n, kKeyBits);
    L.sort_temp = c.take_bytes(L.sort_bytes);
    L.fs = c.take<float>(static_cast<size_t>(kMaxM) * npad);
    L.tables = c.take<unsigned char>(static_cast<size_t>(Wc) * kRankChunkBytes);
    L.hi = c.take<int32_t>(W);
    L.ties = c.take<int2>(n);
    L.valid = c.take<uint64_t>(static_cast<size_t>(Wc) * 8);
    L.A0 = c.take<uint64_t>(W);
    L.A1 = c.take<uint64_t>(W);
    L.state = c.take<uint32_t>(kPeelStateWords);
    L.rend = c.take<int32_t>(npad);
    L.gmask = c.take<uint64_t>(W);
    L.info = c.take<int32_t>(2);
    return c.used;
}

// Cooperative grid of the peel: at most one 1024-thread workgroup per CU and
// about 4 row blocks per workgroup; 0 if the kernel cannot be resident.
int peel_grid_size(int nblk)
{
    static int cus = 0;
    if (cus == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    }
    int grid = ceil_div(nblk, 4);
    if (grid > cus) grid = cus;
    if (grid > kBarMaxBlocks) grid = kBarMaxBlocks;
    if (grid < 1) grid = 1;
    const int bpg = ceil_div(nblk, grid);
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(nds_peel),
                                                    kPeelThreads, peel_lds_bytes(nblk, bpg)) != hipSuccess ||
        per_cu < 1)
        return 0;
    return grid;
}

}  // namespace

// Rank-table bytes of one instance with nm rows and m objectives.
size_t nds_table_bytes(int nm, int m)
{
    return static_cast<size_t>(ceil_div(nm, kChunk)) * (m - 1) * rank_table_bytes(rank_sub(m));
}

size_t nds_workspace_bytes(int n)
{
    NdsLayout L;
    return carve_nds(nullptr, n, L);
}

int nds_max_n() { return kMaxWords * 64; }

void nds_key_buffers(void* ws, int n, uint64_t** keys, int32_t** vals)
{
    NdsLayout L;
    carve_nds(ws, n, L);
    *keys = L.keys_in;
    *vals = L.vals_in;
}

int nds_run(const float* f, int ldf, const float* cv, int n, int m, int stop_at, int32_t* fronts,
            int32_t* max_front, void* ws, size_t ws_bytes, hipStream_t stream, uint32_t* error, bool keys_ready)
{
    if (n <= 0 || m <= 0 || m > kMaxM || !f || !cv || !fronts || !max_front || ldf < n)
        return fail(kInvalidArgument, "nds: invalid arguments");
    if (n > nds_max_n()) return fail(kUnsupported, "nds: population larger than supported");
    if (!ws || ws_bytes < nds_workspace_bytes(n)) return fail(kWorkspaceTooSmall, "nds: workspace too small");
    const int W = ceil_div(n, 64);
    const int Wc = ceil_div(W, 8);
    const int npad = W * 64;
    NdsLayout L;
    carve_nds(ws, n, L);

    stage_begin(kStNdsSort, stream);
    const int tb = 256;
    if (!keys_ready) {
        hipLaunchKernelGGL(nds_keys, dim3(ceil_div(n, tb)), dim3(tb), 0, stream, f, ldf, cv, n, m,
                           L.keys_in, L.vals_in);
        MOEA_HIP(hipGetLastError());
    }
    MOEA_CHECK(sort_pairs(L.sort_temp, L.sort_bytes, L.keys_in, L.keys_out, L.vals_in, L.perm, n,
                          stream, kKeyBits));
    // row ends pay for their atomics when many rows have no dominator near
    // their own block, which is the case for many objectives
    int32_t* rend = m >= kRowEndMinM ? L.rend : nullptr;
    const PrepOut O{L.fs, L.valid, L.hi, L.ties, L.gmask, L.info, rend, L.tables};
    const dim3 pgrid(Wc, m), pblock(kChunk);
    // also clears the peel's barrier state (not read before the peel)
    if (rank_sub(m) == 256)
        hipLaunchKernelGGL(nds_prep<256>, pgrid, pblock, 0, stream, f, ldf, n, m, npad, L.perm, L.keys_out, O, L.state,
                           kPeelStateWords, max_front);
    else
        hipLaunchKernelGGL(nds_prep<128>, pgrid, pblock, 0, stream, f, ldf, n, m, npad, L.perm, L.keys_out, O, L.state,
                           kPeelStateWords, max_front);
    MOEA_HIP(hipGetLastError());
    stage_end(kStNdsSort, stream);

    stage_begin(kStDominance, stream);
    const int seg = dom_segment(W, Wc, m);
    const dim3 dgrid(ceil_div(W, seg), Wc), dblock(dom_threads(m));
    MOEA_LAUNCH_M(m, nds_dominance, dgrid, dblock, dom_lds_bytes(m), stream, L.fs, npad, n, W, Wc, L.valid, L.hi,
                  L.ties, L.tables, L.B, rend, seg);
    MOEA_HIP(hipGetLastError());
    stage_end(kStDominance, stream);

    const int grid = W <= kOneGroupBlocks ? 1 : peel_grid_size(W);
    if (grid <= 0) return fail(kUnsupported, "nds: peel kernel cannot be resident on this device");
    const int bpg = ceil_div(W, grid);
    const size_t lds = peel_lds_bytes(W, bpg);
    PeelArgs args{L.B, L.hi, L.perm, n, W, Wc, stop_at, bpg, fronts, L.A0, L.A1, L.state, max_front, rend,
                  peel_spin_limit(), error, L.gmask, L.info};
    void* kargs[] = {&args};
    stage_begin(kStPeel, stream);
    if (grid == 1)
        hipLaunchKernelGGL(nds_peel_one, dim3(1), dim3(kPeelThreads), static_cast<unsigned>(lds), stream, args);
    else
        MOEA_HIP(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(nds_peel), dim3(grid),
                                        dim3(kPeelThreads), kargs, static_cast<unsigned>(lds), stream));
    MOEA_HIP(hipGetLastError());
    stage_end(kStPeel, stream);
    return kOk;
}

// ------------------------------------------------------ allocation-free --
// moea_nds_rank_static: the same sort with its workspace in this file-scope
// device array instead of a caller's buffer, for callers that cannot allocate
// (graph capture, serving loops).  Every GPU holds its own copy until the
// process ends; host code reaches it only through the address that
// hipGetSymbolAddress reports for the current device (the array's name is a
// host-side stand-in, not a device address).  Nothing in it needs clearing
// between calls: nds_prep zeroes the peel state and the peel
// initializes cursors, fronts and the assigned sets.  Calls that overlap on
// one GPU share the array and race.
constexpr size_t kStaticScratchBytes = size_t{16} << 20;
constexpr int kStaticMaxN = 8192;
constexpr int kStaticMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
std::mutex g_scratch_mu;
void* g_scratch_ptr[kStaticMaxDevices] = {};
}  // namespace

int nds_run_static(const float* f, int ldf, const float* cv, int n, int m, int stop_at, int32_t* fronts,
                   int32_t* max_front, hipStream_t stream)
{
    if (n > kStaticMaxN)
        return fail(kInvalidArgument, "moea_nds_rank_static: n = " + std::to_string(n) + " exceeds the " +
                                          std::to_string(kStaticMaxN) + " rows its static workspace holds");
    if (n > 0 && nds_workspace_bytes(n) > kStaticScratchBytes)
        return fail(kInvalidArgument, "moea_nds_rank_static: workspace for n = " + std::to_string(n) +
                                          " exceeds the static scratch array");
    int dev = 0;
    MOEA_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kStaticMaxDevices) return fail(kUnsupported, "moea_nds_rank_static: device index too large");
    void* ptr = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mu);
        if (!g_scratch_ptr[dev]) {
            void* p = nullptr;
            const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
            if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
            if (!p) return fail(kHipError, "hipGetSymbolAddress(scratch) returned a null address");
            g_scratch_ptr[dev] = p;
        }
        ptr = g_scratch_ptr[dev];
    }
    return nds_run(f, ldf, cv, n, m, stop_at, fronts, max_front, ptr, kStaticScratchBytes, stream);
}

int nds_static_max_n() { return kStaticMaxN; }

void set_peel_spin_limit(uint32_t limit) { g_spin_limit.store(limit == 0 ? kSpinLimit : limit); }

int batch_peel_capacity()
{
    int dev = 0, cus = 0, per_cu = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(b_nds_peel_groups),
                                                    kPeelThreads, kBatchPeelMaxLds) != hipSuccess)
        return 0;
    const int cap = cus * per_cu;
    return cap < kBarMaxBlocks ? cap : kBarMaxBlocks;
}

// Groups for the batched peel.  An instance of W row blocks wants one block
// per `rows_per_block` row blocks (16: one row block per wave; 32: two) and
// needs at least one per 32 (the per-block task queue is sized for 32).  When
// the wanted blocks exceed the capacity, the largest instances still get
// groups of their own (scaled down) and the rest join the least-loaded group
// large enough for them; a group's blocks run its instances in the same
// order, so no two groups wait on each other.  The plan decides only which
// workgroup peels which rows: the fronts do not depend on it.
int batch_peel_plan(const std::vector<int>& inst, const std::vector<int>& W, int capacity, int rows_per_block,
                    std::vector<int>& first, std::vector<int>& jobs, size_t& lds)
{
    const int count = static_cast<int>(inst.size());
    first.assign(1, 0);
    jobs.clear();
    lds = 0;
    if (count == 0) return 0;
    if (capacity < 1) return fail(kUnsupported, "batched peel cannot be resident on this device");
    if (rows_per_block < 1 || rows_per_block > 32) return fail(kInvalidArgument, "batched peel: rows per block out of range");
    std::vector<int> want(count), need(count), order(count);
    long long demand = 0;
    for (int i = 0; i < count; ++i) {
        want[i] = std::max(1, std::min(ceil_div(W[i], rows_per_block), capacity));
        need[i] = std::max(1, ceil_div(W[i], 32));
        if (need[i] > capacity) return fail(kUnsupported, "batched peel: population too large for one device");
        demand += want[i];
        order[i] = i;
    }
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return W[a] > W[b]; });
    struct Group { int size; double load; std::vector<int> members; };
    std::vector<Group> groups;
    int used = 0;
    for (int oi = 0; oi < count; ++oi) {
        const int i = order[oi];
        int size = want[i];
        if (demand > capacity)
            size = std::max(need[i], static_cast<int>(static_cast<double>(want[i]) * capacity / demand));
        const double cost = static_cast<double>(W[i]) * W[i];
        if (used + size <= capacity) {
            groups.push_back({size, cost / size, {i}});
            used += size;
            continue;
        }
        int best = -1;
        for (int gi = 0; gi < static_cast<int>(groups.size()); ++gi)
            if (groups[gi].size >= need[i] && (best < 0 || groups[gi].load < groups[best].load)) best = gi;
        if (best < 0) return fail(kUnsupported, "batched peel: no group can hold an instance");
        groups[best].members.push_back(i);
        groups[best].load += cost / groups[best].size;
    }
    for (const Group& gr : groups) {
        for (int r = 0; r < gr.size; ++r) {
            for (int i : gr.members) {
                jobs.push_back(inst[i]);
                jobs.push_back(r);
                jobs.push_back(gr.size);
            }
            first.push_back(static_cast<int>(jobs.size() / 3));
        }
        for (int i : gr.members) lds = std::max(lds, peel_lds_bytes(W[i], ceil_div(W[i], gr.size)));
    }
    if (lds > static_cast<size_t>(kBatchPeelMaxLds)) return fail(kUnsupported, "batched peel: LDS bound exceeded");
    return kOk;
}

size_t batch_nds_sort_bytes(long long total_rows, int inst_bits)
{
    return sort_pairs_temp_bytes(static_cast<int>(total_rows), kKeyBits + inst_bits);
}

int batch_nds(const BatchLaunch& L, const BNdsGrids& G, const BNdsScratch& S, int mode, int state)
{
    hipStream_t st = L.stream;
    if (G.rows256.blocks <= 0) return kOk;
    stage_begin(kStNdsSort, st);
    hipLaunchKernelGGL(b_nds_keys, dim3(G.rows256.blocks), dim3(256), 0, st, L.insts, G.rows256.map, mode,
                       S.keys_in, S.vals_in);
    MOEA_HIP(hipGetLastError());
    MOEA_CHECK(sort_pairs(S.sort_temp, S.sort_bytes, S.keys_in, S.keys_out, S.vals_in, S.vals_out,
                          static_cast<int>(G.total_rows), st, kKeyBits + S.inst_bits));
    hipLaunchKernelGGL(b_nds_prep, dim3(G.prep.blocks), dim3(kChunk), 0, st, L.insts, G.prep.map, mode, S.keys_out,
                       S.vals_out);
    MOEA_HIP(hipGetLastError());
    stage_end(kStNdsSort, st);
    stage_begin(kStDominance, st);
    for (int m = 1; m <= kMaxM; ++m) {
        if (G.dom[m].blocks <= 0) continue;
        const dim3 grid(G.dom[m].blocks), block(dom_threads(m));
        MOEA_LAUNCH_M(m, b_nds_dominance, grid, block, dom_lds_bytes(m), st, L.insts, G.dom[m].map, mode);
        MOEA_HIP(hipGetLastError());
    }
    stage_end(kStDominance, st);
    stage_begin(kStPeel, st);
    hipLaunchKernelGGL(b_peel_reset, dim3(L.count), dim3(256), 0, st, L.insts, mode, state);
    MOEA_HIP(hipGetLastError());
    int mode_arg = mode;
    const BInst* insts_arg = L.insts;
    const int* first_arg = G.peel_first;
    const int* jobs_arg = G.peel_jobs;
    uint32_t spin_arg = peel_spin_limit();
    uint32_t* error_arg = S.error;
    void* kargs[] = {&insts_arg, &mode_arg, &first_arg, &jobs_arg, &spin_arg, &error_arg};
    MOEA_HIP(hipLaunchCooperativeKernel(reinterpret_cast<const void*>(b_nds_peel_groups), dim3(G.peel_wgs),
                                        dim3(kPeelThreads), kargs, static_cast<unsigned>(G.peel_lds), st));
    MOEA_HIP(hipGetLastError());
    stage_end(kStPeel, st);
    return kOk;
}

}  // namespace moea
