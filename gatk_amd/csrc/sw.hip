// sw.hip -- gfx950 Smith-Waterman (read -> haplotype and haplotype -> reference realignment).
//
// Model: SmithWatermanJavaAligner.calculateMatrix / calculateCigar
// (src/main/java/org/broadinstitute/hellbender/utils/smithwaterman/SmithWatermanJavaAligner.java:
// 104-377), the algorithm behind GKL's SWAlignerNativeBinding.  Integer scores; rows are reference
// positions i, columns alternate positions j; affine gaps in the reference's "best gap" form:
//   V(i,j) = sw(i-1,j) + open  if that beats V(i-1,j) + extend  (then its length is 1, else +1)
//   H(i,j) = sw(i,j-1) + open  if that beats H(i,j-1) + extend
//   sw(i,j) = max(-1e8, diag if diag >= V and diag >= H, else H if H >= V, else V)
// with the backtrack code 0 (diagonal), -len(H) or +len(V) per cell (:160-229).
//
// Mapping: one pair per wave.  A lane owns K consecutive alternate columns (K = ceil(A / 64) up to 4:
// a read of up to 256 bases is one sweep; longer ones take stripes of 256 columns) and at step t
// computes row i = t - lane + 1 of all K (anti-diagonal sweep down the reference).  It keeps its
// columns' previous scores and vertical gaps in registers; the row's score and horizontal gap to the
// left come from the lane before by DPP wave_shr:1, once per K cells, and that score one step
// earlier is the diagonal.  Lane 0 takes column 0's edge, or from the second stripe on an 8-byte LDS
// record per row: every lane stores its last column's record at its own row, so no step has a
// one-lane branch and lane 63, which writes a row last, leaves the stripe's last column there.
//
// What is kept of a cell is four bits: whether its vertical and its horizontal gap were opened
// there, whether the cell is not a diagonal one, and whether it then took the vertical gap.  The
// reference's backtrack value is a gap's length; walking the open bits back from the cell gives the
// same length (a gap at row 1 or column 1 has length 1 whatever its bit), so the sweep carries no
// lengths: 19 VALU instructions a cell and one store of 4..16 bytes per lane every 8 steps.  The
// wave then picks the end point by reductions and walks the bits as calculateCigar does, 64 diagonal
// cells or 64 gap cells per fetch, writing the CIGAR elements in the reference's list order (the
// host reverses them into text).
//
// Bound by VALU issue: 19 K + 10 instructions a step.  20,000 reads of 100-250 bases against
// haplotypes of 150-600: 1.30 ms (980 GCUPS), where one column per lane, gap lengths carried as
// values, a 2-byte store and LDS round trips every step took 4.23 ms; one region's 81 reads, a wave
// each: 126 us against 773 (few pairs: sw_split_kernel).
#include "pairhmm_device.hpp"
#include "pairhmm_kernels.hpp"

namespace gatk_pairhmm {
namespace {

using namespace dev;

// A row's boundary record between stripes: score and horizontal gap of the stripe's last column.
struct alignas(8) SwScore {
    int32_t sw, bgh;
};

constexpr int kSwBlock = 8;        // steps per unrolled block
constexpr int kSwMaxCols = 4;      // columns per lane of the widest sweep
constexpr int kSwLow = 64;         // LDS slots before row 0 (rows of lanes that have not started)
constexpr int kSwHigh = kWave + kSwBlock;  // and after the last row
constexpr int32_t kLowInit = INT32_MIN / 2;          // :125
constexpr int32_t kMinCutoff = -100000000;           // (int) -1.0e8, :123
enum : uint32_t { kOpM = 0, kOpI = 1, kOpD = 2, kOpS = 3 };
// Bits of a cell, in the order they are appended (first = highest).
constexpr uint32_t kBitVOpen = 8, kBitHOpen = 4, kBitGap = 2, kBitVertical = 1;

__host__ __device__ constexpr int sw_cols_per_lane(int A) {
    return A > kSwMaxCols * kWave ? kSwMaxCols : (A + kWave - 1) / kWave;
}
// Steps whose K nibbles share a 32-bit word, and words per lane and 8-step block.
__host__ __device__ constexpr int sw_steps_per_word(int K) { return K == 1 ? 8 : K == 2 ? 4 : 2; }
__host__ __device__ constexpr int sw_words(int K) { return kSwBlock / sw_steps_per_word(K); }
__host__ __device__ constexpr int sw_stripes(int A) { return (A + kSwMaxCols * kWave - 1) / (kSwMaxCols * kWave); }
__host__ __device__ constexpr int sw_blocks(int R) { return (R + kWave - 1 + kSwBlock - 1) / kSwBlock; }

__device__ __forceinline__ int32_t shr1_keep_i(int32_t old, int32_t src) {
    return __builtin_amdgcn_update_dpp(old, src, kDppWaveShr1, 0xF, 0xF, false);
}

// Score of row 0 / column 0 at position p >= 1 (INDEL and LEADING_INDEL start with gap penalties,
// :133-149), 0 otherwise.
__device__ __forceinline__ int32_t edge_score(int p, bool gap_edges, int32_t open, int32_t extend) {
    return (gap_edges && p >= 1) ? open + (p - 1) * extend : 0;
}

// The end-point search's candidates.  col_*: the last column's best score and the last step that
// reached it, on the lane that owns column A.  bot_*: this lane's best bottom-row cell: highest
// score, then least distance from the main diagonal, then lowest column.
struct SwEnds {
    int32_t col_best = INT32_MIN, col_step = 0;
    int32_t bot_best = INT32_MIN, bot_dist = INT32_MAX, bot_col = INT32_MAX;
};

__device__ __forceinline__ bool better_end(int32_t s, int32_t d, int32_t j, int32_t s0, int32_t d0, int32_t j0) {
    return s > s0 || (s == s0 && (d < d0 || (d == d0 && j < j0)));
}

// One lane's columns of a stripe.
template <int K>
struct SwLane {
    int32_t up[K], bgv[K];  // previous row's scores and vertical gaps
    uint32_t alt[K];
    int32_t left, bgh;      // left neighbour's score and horizontal gap of the current row
    int32_t s_last, h_last; // own last column, what the next lane takes
};

// Appends the bit a > b to w: a compare and an add with carry (the compiler makes a select and a shift-or
// of it, and puts the appends of a whole block off, which keeps every score of the block live).
__device__ __forceinline__ void append_gt(uint32_t &w, int32_t a, int32_t b) {
    asm("v_cmp_gt_i32 vcc, %1, %2\n\tv_addc_co_u32 %0, vcc, %0, %0, vcc" : "+v"(w) : "v"(a), "v"(b) : "vcc");
}

// Eight steps from t0.  kGuard: some lane's row lies outside 1..R; such a lane keeps its state (row 0
// before it starts, row R after it ends).  kA: the owner lane's index of column A.
template <int K, bool kRec, bool kGuard>
__device__ __forceinline__ void sw_block(SwLane<K> &st, SwEnds &ends, const SwBatch &b, const uint8_t *lref,
                                         const SwScore *rec_in, SwScore *rec_out, uint32_t *out, int lane, int t0, int R,
                                         int kA, bool gap_edges) {
    using lds_u8 = const volatile __attribute__((address_space(3))) uint8_t;
    lds_u8 *rp = (lds_u8 *)(lref + kSwLow - lane);  // address-space cast: C-style only
    uint32_t base[kSwBlock];
    SwScore in[kSwBlock];
#pragma unroll
    for (int u = 0; u < kSwBlock; ++u) base[u] = rp[t0 + u];
    if constexpr (kRec) {
#pragma unroll
        for (int u = 0; u < kSwBlock; ++u) in[u] = rec_in[kSwLow + t0 + u + 1];
        __builtin_amdgcn_wave_barrier();
    }
    uint32_t words[sw_words(K)];
    uint32_t w = 0;
#pragma unroll
    for (int u = 0; u < kSwBlock; ++u) {
        const int t = t0 + u;
        const int i = t - lane + 1;
        int32_t diag = st.left;
        st.left = shr1_keep_i(kRec ? in[u].sw : edge_score(t + 1, gap_edges, b.open, b.extend), st.s_last);
        st.bgh = shr1_keep_i(kRec ? in[u].bgh : kLowInit, st.h_last);
        const bool active = !kGuard || (i >= 1 && i <= R);
        int32_t left = st.left, bgh = st.bgh, at_a = 0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int32_t sd = diag + (base[u] == st.alt[k] ? b.match : b.mismatch);
            const int32_t vo = st.up[k] + b.open, ve = st.bgv[k] + b.extend;
            append_gt(w, vo, ve);
            const int32_t v = vo > ve ? vo : ve;
            const int32_t ho = left + b.open, he = bgh + b.extend;
            append_gt(w, ho, he);
            bgh = ho > he ? ho : he;
            const int32_t gap = bgh > v ? bgh : v;
            int32_t s = gap > sd ? gap : sd;
            append_gt(w, gap, sd);
            append_gt(w, v, bgh);
            s = s > kMinCutoff ? s : kMinCutoff;
            diag = st.up[k];
            if (k == 0 || k == kA) at_a = s;
            st.up[k] = active ? s : st.up[k];
            st.bgv[k] = active ? v : st.bgv[k];
            left = s;
        }
        st.s_last = active ? left : st.s_last;
        st.h_last = bgh;
        const bool better = active && at_a >= ends.col_best;
        ends.col_best = better ? at_a : ends.col_best;
        ends.col_step = better ? t : ends.col_step;
        if constexpr (kRec) {
            // Rows outside 1..R land in the low and high slots, or on rows that a later lane rewrites.
            SwScore *r = rec_out + kSwLow + i;
            r->sw = left;
            r->bgh = bgh;
            asm volatile("" ::: "memory");  // the steps' stores stay in order: lane 63's to a row comes last
        }
        constexpr int kSpw = sw_steps_per_word(K);
        if (u % kSpw == kSpw - 1) {
            words[u / kSpw] = w;
            w = 0;
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    __builtin_memcpy(__builtin_assume_aligned(out, sw_words(K) * 4), words, sizeof(words));
}

// A stripe's lanes before its first step.
template <int K>
__device__ __forceinline__ SwLane<K> sw_lane_start(const SwBatch &b, const uint8_t *alt, int j0, int A, bool gap_edges) {
    SwLane<K> st;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        st.up[k] = edge_score(j0 + k + 1, gap_edges, b.open, b.extend);
        st.bgv[k] = kLowInit;
        st.alt[k] = j0 + k < A ? alt[j0 + k] : 0xFFFFu;
    }
    st.left = edge_score(j0, gap_edges, b.open, b.extend);
    st.bgh = kLowInit;
    st.s_last = st.up[K - 1];
    st.h_last = kLowInit;
    return st;
}

// Bottom-row candidates of a stripe's lane (columns j0 + 1 .. j0 + K).
template <int K>
__device__ __forceinline__ void sw_bottom(SwEnds &ends, const SwLane<K> &st, int j0, int R, int A) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int j = j0 + k + 1;
        const int d = R - j < 0 ? j - R : R - j;
        if (j <= A && better_end(st.up[k], d, j, ends.bot_best, ends.bot_dist, ends.bot_col)) {
            ends.bot_best = st.up[k];
            ends.bot_dist = d;
            ends.bot_col = j;
        }
    }
}

// All stripes of a pair: cell bits into bt, the end-point candidates into `ends`.
template <int K, bool kRec>
__device__ __forceinline__ void sw_matrix(const SwBatch &b, const uint8_t *lref, SwScore *recs, uint32_t *bt, const uint8_t *alt,
                          int lane, int R, int A, bool gap_edges, SwEnds &ends) {
    constexpr int kCols = K * kWave;
    const int n_stripes = kRec ? sw_stripes(A) : 1;
    const int n_blocks = sw_blocks(R);
    for (int s = 0; s < n_stripes; ++s) {
        const int j0 = s * kCols + lane * K;  // this lane's columns are j0 + 1 .. j0 + K
        SwLane<K> st = sw_lane_start<K>(b, alt, j0, A, gap_edges);
        const bool last = s == n_stripes - 1;
        const int kA = last ? (A - 1) % K : 0;
        SwEnds col;
        uint32_t *out = bt + (static_cast<size_t>(s) * n_blocks * kWave + lane) * sw_words(K);
        for (int tb = 0; tb < n_blocks; ++tb) {
            const int t0 = tb * kSwBlock;
            if (t0 < kWave - 1 || t0 + kSwBlock > R)
                sw_block<K, kRec, true>(st, col, b, lref, recs, recs, out, lane, t0, R, kA, gap_edges);
            else
                sw_block<K, kRec, false>(st, col, b, lref, recs, recs, out, lane, t0, R, kA, gap_edges);
            out += kWave * sw_words(K);
        }
        if (last) {
            ends.col_best = col.col_best;
            ends.col_step = col.col_step;
        }
        sw_bottom<K>(ends, st, j0, R, A);
        __builtin_amdgcn_wave_barrier();
    }
}

// Bits of cell (i, j), both >= 1.
template <int K>
__device__ __forceinline__ uint32_t sw_cell(const uint32_t *bt, int n_blocks, int i, int j) {
    constexpr int kCols = K * kWave, kSpw = sw_steps_per_word(K);
    const int s = (j - 1) / kCols, c = (j - 1) % kCols, l = c / K, k = c % K;
    const int t = i - 1 + l, u = t % kSwBlock;
    const uint32_t w = bt[((static_cast<size_t>(s) * n_blocks + t / kSwBlock) * kWave + l) * sw_words(K) + u / kSpw];
    return (w >> (4 * ((kSpw - 1 - u % kSpw) * K + (K - 1 - k)))) & 15u;
}

// calculateCigar (:256-377), run by the whole wave on wave-uniform state; lane 0 stores.
template <int K>
__device__ __forceinline__ void sw_traceback(const SwBatch &b, const uint32_t *bt, uint32_t p, int lane, int R, int A, SwEnds ends) {
    const int n_blocks = sw_blocks(R);
    int p1 = R, p2 = A, segment = 0;
    if (b.strategy != 1) {
        // The last column: its highest score, the last row on ties (kept by the owner lane).
        const int owner = ((A - 1) % (K * kWave)) / K;
        const int32_t best = __builtin_amdgcn_readlane(ends.col_best, owner);
        p1 = __builtin_amdgcn_readlane(ends.col_step, owner) - owner + 1;
        if (b.strategy != 2) {
            // The bottom row, left to right: a cell replaces the end point if it scores higher, or as
            // high and nearer to the main diagonal; so the best of it decides.
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const int32_t s = __shfl_xor(ends.bot_best, off, kWave), d = __shfl_xor(ends.bot_dist, off, kWave);
                const int32_t j = __shfl_xor(ends.bot_col, off, kWave);
                if (better_end(s, d, j, ends.bot_best, ends.bot_dist, ends.bot_col)) {
                    ends.bot_best = s;
                    ends.bot_dist = d;
                    ends.bot_col = j;
                }
            }
            const int32_t s = __builtin_amdgcn_readfirstlane(ends.bot_best);
            const int32_t d = __builtin_amdgcn_readfirstlane(ends.bot_dist);
            const int d_col = p1 - p2 < 0 ? p2 - p1 : p1 - p2;
            if (s > best || (s == best && d < d_col)) {
                p1 = R;
                p2 = __builtin_amdgcn_readfirstlane(ends.bot_col);
                segment = A - p2;
            }
        }
    }
    uint32_t *elems = b.elems + b.elem_off[p];
    uint32_t *elems_short = b.elems_short + static_cast<size_t>(p) * kSwShortElems;
    int n = 0;
    auto put = [&](uint32_t op, int32_t len) {
        const uint32_t e = (static_cast<uint32_t>(len) << 2) | op;
        if (lane == 0) {
            elems[n] = e;
            if (n < kSwShortElems) elems_short[n] = e;
        }
        ++n;
    };
    if (segment > 0 && b.strategy == 0) {
        put(kOpS, segment);
        segment = 0;
    }
    uint32_t state = kOpM;
    do {
        // The next 64 cells down the diagonal from (p1, p2): a run of diagonal cells is a run of
        // single MATCH steps, taken at once; the first other cell is one gap step.
        const int ci = p1 - lane, cj = p2 - lane;
        uint32_t bits = kBitGap;  // outside the matrix: stop
        if (ci >= 1 && cj >= 1) bits = sw_cell<K>(bt, n_blocks, ci, cj);
        const uint64_t stop = __ballot((bits & kBitGap) != 0);
        const int f = stop ? __builtin_ctzll(stop) : kWave;
        if (f > 0) {
            if (state == kOpM) {
                segment += f;
            } else {
                if (segment > 0) put(state, segment);
                segment = f;
                state = kOpM;
            }
            p1 -= f;
            p2 -= f;
        }
        if (f < kWave && p1 > 0 && p2 > 0) {
            const bool vertical = (__builtin_amdgcn_readlane(static_cast<int>(bits), f) & kBitVertical) != 0;
            // The gap's length: cells back along it to the first one that opened it.
            int step = 0;
            for (;;) {
                const int gi = vertical ? p1 - step - lane : p1, gj = vertical ? p2 : p2 - step - lane;
                bool open = true;  // row 1 and column 1 end a gap
                if ((vertical ? gi : gj) > 1)
                    open = (sw_cell<K>(bt, n_blocks, gi, gj) & (vertical ? kBitVOpen : kBitHOpen)) != 0;
                const uint64_t m = __ballot(open);
                if (m != 0) {
                    step += __builtin_ctzll(m) + 1;
                    break;
                }
                step += kWave;
            }
            const uint32_t ns = vertical ? kOpD : kOpI;
            if (vertical)
                p1 -= step;
            else
                p2 -= step;
            if (ns == state) {
                segment += step;
            } else {
                if (segment > 0) put(state, segment);
                segment = step;
                state = ns;
            }
        }
    } while (p1 > 0 && p2 > 0);
    int offset;
    if (b.strategy == 0) {
        put(state, segment);
        if (p2 > 0) put(kOpS, p2);
        offset = p1;
    } else if (b.strategy == 3) {
        put(state, segment + p2);
        offset = p1 - p2;
    } else {
        put(state, segment);
        if (p1 > 0)
            put(kOpD, p1);
        else if (p2 > 0)
            put(kOpI, p2);
        offset = 0;
    }
    if (lane == 0) {
        b.n_elems[p] = n;
        b.offset[p] = offset;
    }
}

template <int K, bool kRec>
__device__ __forceinline__ void sw_pair(const SwBatch &b, const uint8_t *lref, SwScore *recs, uint32_t *bt, uint32_t p,
                                        int lane, int R, int A) {
    const bool gap_edges = b.strategy == 1 || b.strategy == 2;
    SwEnds ends;
    sw_matrix<K, kRec>(b, lref, recs, bt, b.alt_bases + b.alt_off[p], lane, R, A, gap_edges, ends);
    // Lanes read what other lanes stored to global memory: wait for the stores, and drop the vector
    // L1 lines an earlier pair's traceback may hold for this scratch.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    sw_traceback<K>(b, bt, p, lane, R, A, ends);
}

// kLong: some alternate of the batch is longer than one sweep's columns.
template <bool kLong>
__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(kLong ? 3 : 5))) void sw_kernel(SwBatch b, uint32_t n_pairs) {
    extern __shared__ SwScore lds_sw[];
    const int lane = static_cast<int>(threadIdx.x);
    SwScore *recs = lds_sw;
    uint8_t *lref = reinterpret_cast<uint8_t *>(lds_sw + (kLong ? kSwLow + b.max_ref_len + kSwHigh : 0));
    uint32_t *bt = reinterpret_cast<uint32_t *>(b.scratch + static_cast<size_t>(blockIdx.x) * b.scratch_per_wave);
    // The first pair is the one of the wave's own number, the next ones come from the queue head (an atomic
    // on one address, about 14 ns each).
    for (uint32_t p = blockIdx.x; p < n_pairs;) {
        const int R = __builtin_amdgcn_readfirstlane(b.ref_len[p]), A = __builtin_amdgcn_readfirstlane(b.alt_len[p]);
        const uint8_t *ref = b.ref_bases + b.ref_off[p];
        __builtin_amdgcn_wave_barrier();
        for (int i = lane; i < R; i += kWave) lref[kSwLow + i] = ref[i];  // rows outside 1..R read leftovers
        if (kLong && A > kSwMaxCols * kWave) {
            const bool gap_edges = b.strategy == 1 || b.strategy == 2;
            for (int i = lane; i <= R; i += kWave)
                recs[kSwLow + i] = SwScore{edge_score(i, gap_edges, b.open, b.extend), kLowInit};
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (kLong && A > kSwMaxCols * kWave)
            sw_pair<4, kLong>(b, lref, recs, bt, p, lane, R, A);
        else if (A > 3 * kWave)
            sw_pair<4, false>(b, lref, recs, bt, p, lane, R, A);
        else if (A > 2 * kWave)
            sw_pair<3, false>(b, lref, recs, bt, p, lane, R, A);
        else if (A > kWave)
            sw_pair<2, false>(b, lref, recs, bt, p, lane, R, A);
        else
            sw_pair<1, false>(b, lref, recs, bt, p, lane, R, A);
        __builtin_amdgcn_wave_barrier();
        if (n_pairs <= gridDim.x) break;
        // All lanes issue the atomic (lane 0 adds 1): the fetch has no lane-divergent branch.
        p = gridDim.x + __builtin_amdgcn_readfirstlane(atomicAdd(b.queue_head, lane == 0 ? 1u : 0u));
    }
}

// Few pairs: a workgroup of kSplitWaves waves per pair, one stripe of 64 K columns per wave, K the least
// of 1, 2, 4 that covers the alternate.  Wave w runs kSplitLag blocks behind wave w - 1, whose lane 63 has then
// stored the records of the rows that the block reads; a barrier a block keeps the distance.  The record
// arrays are a ring: the last wave's records, which nobody reads, land on rows that wave 0 read long before.
// The cell bits lie as the one-wave kernel lays out stripes of K columns a lane, and wave 0 walks them.
//
// A lone wave is bound by its own issue, 19 K + 10 instructions a step; here four SIMDs share a pair, and waits
// bound it: 29 % of the waves' cycles issue a VALU instruction, 56 % wait.  Cycle stamps in a pair (which cost some
// themselves): 1,400 to 1,500 a block of 8 steps (1,800 to 1,900 where lanes lie outside the rows), of which
// about 900 are issue and the rest LDS reads and the chain; about 160 more at the barrier; and after 120,000 to
// 170,000 of sweep 14,000 to 69,000 of traceback, whose reads depend on each other.  One region's 81 reads of
// 100-250 by haplotypes of 150-460: 126 us with a wave per pair, 94 us with this; 81 haplotypes of up to 612 by
// references of up to 696, whole call: 448 us and 222 us.
constexpr int kSplitWaves = 4;
constexpr int kSplitLag = (kWave + 2 * kSwBlock - 2) / kSwBlock;  // row t + 8 is complete 70 steps after step t

struct SwSplitLds {
    SwScore *recs;      // kSplitWaves arrays of `stride` records
    int stride;
    SwEnds *ends;       // kSplitWaves x 64
    uint8_t *ref;
};

// LDS is all that the waves exchange inside the sweep: the barrier waits for LDS alone, stores of cell bits
// stay in flight.
__device__ __forceinline__ void sw_split_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int K>
__device__ __forceinline__ void sw_split_pair(const SwBatch &b, const SwSplitLds &L, uint32_t *bt, uint32_t p, int lane,
                                              int wave, int R, int A) {
    const bool gap_edges = b.strategy == 1 || b.strategy == 2;
    const int n_stripes = (A + K * kWave - 1) / (K * kWave), n_blocks = sw_blocks(R);
    const int j0 = wave * K * kWave + lane * K;
    SwLane<K> st = sw_lane_start<K>(b, b.alt_bases + b.alt_off[p], j0, A, gap_edges);
    const int kA = wave == n_stripes - 1 ? (A - 1) % K : 0;
    const SwScore *rec_in = L.recs + wave * L.stride;
    SwScore *rec_out = L.recs + (wave + 1) % kSplitWaves * L.stride;
    SwEnds ends;
    uint32_t *out = bt + (static_cast<size_t>(wave) * n_blocks * kWave + lane) * sw_words(K);
    const int rounds = n_blocks + kSplitLag * (n_stripes - 1);
    for (int g = 0; g < rounds; ++g) {
        sw_split_barrier();  // the first one also ends the staging of the reference and the edges
        const int tb = g - kSplitLag * wave;
        if (wave >= n_stripes || tb < 0 || tb >= n_blocks) continue;
        const int t0 = tb * kSwBlock;
        if (t0 < kWave - 1 || t0 + kSwBlock > R)
            sw_block<K, true, true>(st, ends, b, L.ref, rec_in, rec_out, out, lane, t0, R, kA, gap_edges);
        else
            sw_block<K, true, false>(st, ends, b, L.ref, rec_in, rec_out, out, lane, t0, R, kA, gap_edges);
        out += kWave * sw_words(K);
    }
    if (wave < n_stripes) sw_bottom<K>(ends, st, j0, R, A);
    L.ends[wave * kWave + lane] = ends;
    // The cell bits too have to be out before wave 0 reads them, past lines that its L1 may hold.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    if (wave != 0) return;
    for (int w = 1; w < n_stripes; ++w) {
        const SwEnds e = L.ends[w * kWave + lane];
        if (better_end(e.bot_best, e.bot_dist, e.bot_col, ends.bot_best, ends.bot_dist, ends.bot_col)) {
            ends.bot_best = e.bot_best;
            ends.bot_dist = e.bot_dist;
            ends.bot_col = e.bot_col;
        }
    }
    const SwEnds last = L.ends[(n_stripes - 1) * kWave + lane];
    ends.col_best = last.col_best;
    ends.col_step = last.col_step;
    sw_traceback<K>(b, bt, p, lane, R, A, ends);
}

__global__ __launch_bounds__(kSplitWaves *kWave) void sw_split_kernel(SwBatch b) {
    extern __shared__ SwScore lds_sw[];
    const int lane = static_cast<int>(threadIdx.x) % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
    SwSplitLds L;
    L.recs = lds_sw;
    L.stride = kSwLow + b.max_ref_len + kSwHigh;
    L.ends = reinterpret_cast<SwEnds *>(lds_sw + kSplitWaves * L.stride);
    L.ref = reinterpret_cast<uint8_t *>(L.ends + kSplitWaves * kWave);
    const uint32_t p = blockIdx.x;
    uint32_t *bt = reinterpret_cast<uint32_t *>(b.scratch + static_cast<size_t>(p) * b.scratch_per_wave);
    const int R = __builtin_amdgcn_readfirstlane(b.ref_len[p]), A = __builtin_amdgcn_readfirstlane(b.alt_len[p]);
    const uint8_t *ref = b.ref_bases + b.ref_off[p];
    const bool gap_edges = b.strategy == 1 || b.strategy == 2;
    for (int i = static_cast<int>(threadIdx.x); i <= R; i += kSplitWaves * kWave) {
        if (i < R) L.ref[kSwLow + i] = ref[i];  // rows outside 1..R read leftovers
        L.recs[kSwLow + i] = SwScore{edge_score(i, gap_edges, b.open, b.extend), kLowInit};
    }
    if (A > 2 * kSplitWaves * kWave)
        sw_split_pair<4>(b, L, bt, p, lane, wave, R, A);
    else if (A > kSplitWaves * kWave)
        sw_split_pair<2>(b, L, bt, p, lane, wave, R, A);
    else
        sw_split_pair<1>(b, L, bt, p, lane, wave, R, A);
}

size_t sw_split_lds_bytes(int max_ref_len) {
    const size_t rows = static_cast<size_t>(kSwLow + max_ref_len + kSwHigh);
    return rows * (kSplitWaves * sizeof(SwScore) + 1) + kSplitWaves * kWave * sizeof(SwEnds);
}

}  // namespace

int sw_max_ref_len() {
    // What the entry points take: a twelfth of the LDS, in rows.  The sweep needs less (sw_lds_bytes: 9 bytes a row and
    // 1,224 in all, or 1 a row), the split kernel, which needs 33, is left out where they don't fit (sw_splits).
    return static_cast<int>(max_lds_per_block() / 12) - 66;
}

size_t sw_lds_bytes(int max_ref_len, int max_alt_len) {
    const size_t rows = static_cast<size_t>(kSwLow + max_ref_len + kSwHigh);
    return rows * (max_alt_len > kSwMaxCols * kWave ? sizeof(SwScore) + 1 : 1);
}

size_t sw_scratch_bytes_per_wave(int max_ref_len, int max_alt_len) {
    const size_t words = static_cast<size_t>(sw_words(sw_cols_per_lane(max_alt_len)));
    return static_cast<size_t>(sw_stripes(max_alt_len)) * static_cast<size_t>(sw_blocks(max_ref_len)) * kWave * words *
           sizeof(uint32_t);
}

// Whether a batch takes the split kernel: its alternates fit (1,024 bases), its LDS allows two workgroups
// a CU, and its pairs are few.  Whole calls with a wave per pair and split, alternates of up to 250: 256
// pairs 162 / 131 us, 512 pairs 173 / 149, 640 pairs 178 / 177, 1,024 pairs 190 / 209.  Alternates of more than
// one sweep (up to 612), where a lone wave runs its stripes one after another: 1,024 pairs 499 / 417 us,
// 2,048 pairs 811 / 733.
bool sw_splits(uint32_t n_pairs, int max_ref_len, int max_alt_len, int num_cus) {
    const uint32_t per_cu = max_alt_len > kSwMaxCols * kWave ? 8u : 2u;
    return n_pairs <= per_cu * static_cast<uint32_t>(num_cus) && max_alt_len <= kSplitWaves * kSwMaxCols * kWave &&
           sw_split_lds_bytes(max_ref_len) <= max_lds_per_block() / 2;
}

hipError_t launch_sw(const SwBatch &batch, uint32_t n_pairs, int grid_blocks, hipStream_t stream) {
    if (n_pairs == 0) return hipSuccess;
    if (batch.max_ref_len > sw_max_ref_len() || grid_blocks < 1) return hipErrorInvalidValue;
    const size_t lds = sw_lds_bytes(batch.max_ref_len, batch.max_alt_len);
    if (lds > max_lds_per_block()) return hipErrorInvalidValue;
    if (batch.split) {
        // A workgroup per pair, each with a wave's scratch.
        const size_t bytes = sw_split_lds_bytes(batch.max_ref_len);
        if (bytes > max_lds_per_block() || batch.max_alt_len > kSplitWaves * kSwMaxCols * kWave ||
            static_cast<uint32_t>(grid_blocks) < n_pairs)
            return hipErrorInvalidValue;
        if (bytes > 65536)
            (void)hipFuncSetAttribute(reinterpret_cast<const void *>(sw_split_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
        hipLaunchKernelGGL(sw_split_kernel, dim3(n_pairs), dim3(kSplitWaves * kWave), bytes, stream, batch);
        return hipGetLastError();
    }
    auto launch = [&](auto kernel) {
        if (lds > 65536)
            (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(lds));
        hipLaunchKernelGGL(kernel, dim3(grid_blocks), dim3(kWave), lds, stream, batch, n_pairs);
        return hipGetLastError();
    };
    return batch.max_alt_len > kSwMaxCols * kWave ? launch(sw_kernel<true>) : launch(sw_kernel<false>);
}

}  // namespace gatk_pairhmm
