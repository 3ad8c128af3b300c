// pdhmm.hip -- gfx950 FP64 kernel of the partially determined PairHMM.
//
// Model: LoglessPDPairHMM.subComputeReadLikelihoodGivenHaplotypeLog10
// (src/main/java/org/broadinstitute/hellbender/utils/pairhmm/LoglessPDPairHMM.java:34-150).  Next to
// M, I, D each row carries branch values bM, bI, bD (:15-17): the main values just before an
// optional deletion span, held across the span and merged back with max() after it.  A per-row
// state machine (NORMAL / INSIDE_DEL / AFTER_DEL, :22-31, 63, 129-136) picks the branch update; SNP
// columns accept a set of alternative bases (isBasePDMatching, :175-194).
//
// Restated for a lane-per-row sweep.  Let E(r,c) be the value a cell hands to its right and lower
// neighbours: E = max(b, X) for X in {M, I, D} when haplotype column c carries DEL_END, else E = X.
// A column is in state AFTER_DEL exactly when the column before it carries DEL_END, and the branch
// and the I rule read column c's own DEL_END bit, so the reference's three cases collapse to
//   M(r,c) = prior (E_M(r-1,c-1) MM + E_I(r-1,c-1) GM + E_D(r-1,c-1) GM)
//   I(r,c) = E_M(r-1,c) MI + E_I(r-1,c) II
//   D(r,c) = E_M(r,c-1) MD + E_D(r,c-1) DD
//   b(r,c) = INSIDE_DEL(r,c) ? b(r,c-1) : E(r,c-1)
// (in NORMAL and INSIDE_DEL the column before carries no DEL_END, so E = X there).  Only
// INSIDE_DEL depends on the row: the state variable is declared outside the row loop (:63), so row 1
// starts NORMAL and every later row starts in the state the previous row ended in, which is the
// same for all rows >= 2.  pd_codes_kernel folds this into each column's code.
//
// Mapping: one pair per wave.  A lane owns kRows = 2 consecutive rows (a stripe of 128; 1 row for a last
// part of up to 64) and at step t computes column c = t - lane + 1 of all of them.  Each row forms, from its new E values and the transitions of the
// row below, the two sums that row needs:
//   A(r+1, c+1) = E_M(r,c) MM' + (E_I(r,c) + E_D(r,c)) GM'    (so M(r+1,c+1) = prior' A)
//   B(r+1, c)   = E_M(r,c) MI' + E_I(r,c) II'                 (so I(r+1,c) = B)
// Along a lane the row below takes B at once and A at the next step; the next lane's first row takes A
// two steps later and B one step later by DPP wave_shr:1, so two doubles cross lanes per step for
// kRows cells.  Lane 0 takes them from a 16-byte LDS record per column, (B(c), A(c+1)): every lane
// stores its last row's record at its own column (no one-lane branch in the step; lane 63 writes a
// column last), and lane 0 reads a block's records at its start, before any lane of the stripe
// stores to them (A of the block's first column was read with the block before).  Stripe 0 starts
// from row 0: M = I = 0, D = 2^1020 / H, so A(1,c) = D GM_1 and B(1,c) = 0.  A wave holds 20 bytes of LDS
// per column with the column's 4-byte code.
//
// Steps run in blocks of 4; a block in which no lane is on a special column (kPdSpecial: a
// deletion end, a column inside a span, or the column before a span) skips the branch update and
// hands on E = X, which is exact because a row's branch values are only read on special columns and
// the column before each span sets them from E.
//
// The result is the sum of M + I (not E) of row R over columns 1..H: rows past R pass the row above
// down (M = D = 0, I = B with MI' = II' = 1), and from row R on B is formed from the plain M and I, so the
// records end holding it.
//
// The prior of the fast path (as in the FP64 forward kernel): the match prior is folded into the
// transitions that form A, a mismatch multiplies by px / pm in the lanes that have one, and M carries
// the factor its next row in the lane would multiply it with.  A column's code holds one bit per class
// of read base that it accepts, a row the bit of its base, so the match test is one AND.  Haplotype
// bytes outside ACGTacgtN and qualities whose match prior or MM is near 0 take selected priors.
//
// Bound by VALU issue: 21 instructions per step of two cells, 47 in a block with a special column, at up
// to 4 waves per SIMD (20 bytes of LDS per column hold longer haplotypes to less), where one row per
// lane took 16 to 18 and 39 per cell.  One region of 81 reads (100-250 bases) and 65 haplotypes of 377,
// kernel under the profiler: 306 us, against 437.  Four rows per lane take 255 VGPRs (two waves per
// SIMD) and were slower: a region's pairs are few, and their tail weighs.
#include "pairhmm_device.hpp"
#include "pairhmm_kernels.hpp"

namespace gatk_pairhmm {
namespace {

using namespace dev;

// One column of a wave's LDS records: B of this column and A of the next one for the stripe's first
// row (the row below lane 63's last row of the stripe before).  The column codes are a separate uint32
// array after the records.
struct alignas(16) PdRecord {
    double b, a;
};
static_assert(sizeof(PdRecord) == 16, "PdRecord is one 16-byte LDS word");

constexpr int kPdPadColumns = 68;  // records past H that lane 0 reads (c <= H + 66 with 4-step blocks)
constexpr int kPdLowPad = 64;      // records below column 0, where stores of columns < 0 land
constexpr int kPdU = 4;            // wave-steps per unrolled block

// Read-base class bit (placed like the column code's alternative mask) of isBasePDMatching
// (:179-195): A/a, C/c, G/g, T/t, and 0x80 for any other base, which only an 'N' haplotype
// base's full mask matches.
__device__ __forceinline__ uint32_t read_base_bit(uint32_t x) {
    switch (x) {
    case 'A': case 'a': return kPdAltA << 8;
    case 'C': case 'c': return kPdAltC << 8;
    case 'G': case 'g': return kPdAltG << 8;
    case 'T': case 't': return kPdAltT << 8;
    default: return 0x80u << 8;
    }
}

// The bit of a read base among the classes a column accepts (kPdAccept*).
__device__ __forceinline__ uint32_t accept_bit(uint32_t x) {
    switch (x) {
    case 'A': return kPdAcceptA;
    case 'C': return kPdAcceptA << 1;
    case 'G': return kPdAcceptA << 2;
    case 'T': return kPdAcceptA << 3;
    case 'a': return kPdAcceptA << 4;
    case 'c': return kPdAcceptA << 5;
    case 'g': return kPdAcceptA << 6;
    case 't': return kPdAcceptA << 7;
    default: return kPdAcceptOther;
    }
}

// Row parameters of read position p (row p + 1); rows past the read are the pass-through row.
struct PdRow {
    double MM, GM, MI, II, MD, DD, pm, px;
    uint32_t x;
};

__device__ __forceinline__ PdRow pd_row(const PdBatch &b, const DeviceTables &tab, int64_t ro, int R, int p) {
    PdRow w{0, 0, 1, 1, 0, 0, 0, 0, 0u};
    if (p >= R) return w;
    w.x = b.rd_bases[ro + p];
    const int q = b.rd_quals[ro + p], qi = b.rd_ins[ro + p], qd = b.rd_del[ro + p], qc = b.rd_gcp[ro + p];
    const int mn = qi < qd ? qi : qd, mx = qi < qd ? qd : qi;
    w.MM = tab.mm_prob[((mx * (mx + 1)) >> 1) + mn];
    w.MI = tab.qual_err[qi];
    w.MD = tab.qual_err[qd];
    w.II = tab.qual_err[qc];
    w.DD = w.II;
    w.GM = 1.0 - w.II;
    const double eq = tab.qual_err[q];
    w.pm = 1.0 - eq;
    w.px = b.tristate ? eq / 3.0 : eq;
    if (w.x == 'N') w.px = w.pm;
    return w;
}

// Rows per lane of the stripe that starts with `left` rows to go.
__device__ __forceinline__ int pd_stripe_rows(int left) { return left > kWave ? 2 : 1; }

// The factor folded into the sums that reach the row at read position p, the first of its lane in a
// stripe of `rows` rows per lane (wave-uniform arguments; fast path).
__device__ __forceinline__ double pd_first_fold(const PdBatch &b, const DeviceTables &tab, int64_t ro, int R, int p,
                                                int rows) {
    double f = 1.0;
    for (int j = 0; j < rows && p + j < R; ++j) {
        const PdRow w = pd_row(b, tab, ro, R, p + j);
        f *= j == 0 ? w.pm : w.pm * w.MM;
    }
    return f;
}

// A lane's rows: own MD, DD and priors, the transitions of the row below each (n), and the state: E and
// branch values at the column before, the row-below sums.  The D values (ED, bD) are carried divided by
// the row's MD: D(c) = E_D(c-1) DD + E_M(c-1) MD becomes D/MD = (E_D/MD) DD + E_M, one FMA, and max()
// commutes with the positive scale (rows past R have MD = DD = 0 and stay 0).  M's factor g scales EM, bM,
// ED and bD alike.
template <int kRows>
struct PdLane {
    double MD[kRows], DD[kRows], pm[kRows], px[kRows], MMn, GMn[kRows], MIn[kRows], IIn[kRows];
    double MMr[kRows];             // generic path: every row's own factor of E_M in A
    uint32_t bit[kRows], x[kRows]; // fast: accepted-class bit; generic: alternative bit and base
    uint32_t inside0;              // the inside bit of the lane's first row
    uint64_t inner[kRows];         // lanes whose row comes before row R
    double EM[kRows], EI[kRows], ED[kRows], bM[kRows], bI[kRows], bD[kRows];
    double an1[kRows], an2, bn1;
};

// Per row, in the lanes whose column does not accept the row's base (m == 0): a *= ratio.  EXEC is all
// ones before and after (a workgroup is one whole wave in uniform control flow); the s_nop completes the
// five wait states a DPP needs after a VALU write of EXEC, which the compiler does not track across
// inline assembly.
__device__ __forceinline__ void scale_unaccepted(double (&a)[1], const double (&ratio)[1], const uint32_t (&m)[1]) {
    asm("v_cmpx_eq_u32_e32 vcc, 0, %2\n\t"
        "v_mul_f64 %0, %0, %1\n\t"
        "s_mov_b64 exec, -1\n\t"
        "s_nop 2"
        : "+&v"(a[0])
        : "v"(ratio[0]), "v"(m[0])
        : "vcc");
}
__device__ __forceinline__ void scale_unaccepted(double (&a)[2], const double (&ratio)[2], const uint32_t (&m)[2]) {
    asm("v_cmpx_eq_u32_e32 vcc, 0, %4\n\t"
        "v_mul_f64 %0, %0, %2\n\t"
        "s_mov_b64 exec, -1\n\t"
        "v_cmpx_eq_u32_e32 vcc, 0, %5\n\t"
        "v_mul_f64 %1, %1, %3\n\t"
        "s_mov_b64 exec, -1\n\t"
        "s_nop 2"
        : "+&v"(a[0]), "+&v"(a[1])
        : "v"(ratio[0]), "v"(ratio[1]), "v"(m[0]), "v"(m[1])
        : "vcc");
}
// The branch update's two masked parts (EXEC as above; SALU writes of it need no wait states).  Outside
// a span the branch values follow the E values of the column before:
__device__ __forceinline__ void pd_hold(double &bM, double &bI, double &bD, double EM, double EI, double ED,
                                        uint64_t outside) {
    asm("s_mov_b64 exec, %6\n\t"
        "v_mov_b64_e32 %0, %3\n\t"
        "v_mov_b64_e32 %1, %4\n\t"
        "v_mov_b64_e32 %2, %5\n\t"
        "s_mov_b64 exec, -1"
        : "+&v"(bM), "+&v"(bI), "+&v"(bD)
        : "v"(EM), "v"(EI), "v"(ED), "s"(outside));
}
// At a deletion's end E is max(b, X), and B of the row below is formed from it except from row R on.
__device__ __forceinline__ void pd_merge(double &EM, double &EI, double &ED, double &bn, double bM, double bI, double bD,
                                         double MIn, double IIn, uint64_t ends, uint64_t ends_inner) {
    asm("s_mov_b64 exec, %9\n\t"
        "v_max_f64 %0, %0, %4\n\t"
        "v_max_f64 %1, %1, %5\n\t"
        "v_max_f64 %2, %2, %6\n\t"
        "s_mov_b64 exec, %10\n\t"
        "v_mul_f64 %3, %0, %7\n\t"
        "v_fma_f64 %3, %1, %8, %3\n\t"
        "s_mov_b64 exec, -1"
        : "+&v"(EM), "+&v"(EI), "+&v"(ED), "+&v"(bn)
        : "v"(bM), "v"(bI), "v"(bD), "v"(MIn), "v"(IIn), "s"(ends), "s"(ends_inner));
}

// One step of a lane at its column.  kBranch: the full branch update; without it E = X and the branch
// values are left alone, which is exact on a block where no lane's column is special: a row's branch
// values are only read at its special columns, and a deletion start (special) sets them from E.
template <int kRows, bool kBranch, bool kGeneric>
__device__ __forceinline__ PdRecord pd_step(PdLane<kRows> &st, double a0, double b0, uint32_t code) {
    double a[kRows];
    double I = wave_shr1(b0, st.bn1);  // lane 0 keeps its record's values
    a[0] = wave_shr1(a0, st.an2);
#pragma unroll
    for (int j = 1; j < kRows; ++j) a[j] = st.an1[j - 1];
    st.an2 = st.an1[kRows - 1];
    if constexpr (!kGeneric) {
        uint32_t accepted[kRows];
#pragma unroll
        for (int j = 0; j < kRows; ++j) accepted[j] = code & st.bit[j];
        scale_unaccepted(a, st.px, accepted);
    }
    uint64_t ends = 0;
    if constexpr (kBranch) ends = __ballot((code & kPdDelEnd) != 0u);
    PdRecord r{0, 0};
#pragma unroll
    for (int j = 0; j < kRows; ++j) {
        if constexpr (kGeneric)
            a[j] *= ((code & 0xFFu) == st.x[j] || (code & st.bit[j]) != 0u) ? st.pm[j] : st.px[j];
        if constexpr (kBranch)
            pd_hold(st.bM[j], st.bI[j], st.bD[j], st.EM[j], st.EI[j], st.ED[j],
                    __ballot((code & (j == 0 ? st.inside0 : kPdInsideLater)) == 0u));
        st.ED[j] = fma(st.ED[j], st.DD[j], st.EM[j]);  // D / MD
        st.EM[j] = a[j];
        st.EI[j] = I;
        r.b = fma(I, st.IIn[j], a[j] * st.MIn[j]);
        if constexpr (kBranch)
            pd_merge(st.EM[j], st.EI[j], st.ED[j], r.b, st.bM[j], st.bI[j], st.bD[j], st.MIn[j], st.IIn[j], ends,
                     ends & st.inner[j]);
        const double s = fma(st.ED[j], st.MD[j], st.EI[j]);
        r.a = fma(s, st.GMn[j], kGeneric ? st.EM[j] * st.MMr[j] : j + 1 == kRows ? st.EM[j] * st.MMn : st.EM[j]);
        st.an1[j] = r.a;
        I = r.b;
    }
    st.bn1 = r.b;
    return r;
}

// A record as two 8-byte stores.  The barrier between them also keeps the steps' stores in order: the lanes
// store to one column a step apart, and the last lane's has to come last.  One 16-byte store takes ten more
// registers to scratch and the same time (374 and 375 us for 81 reads by 65 haplotypes of 377).
__device__ __forceinline__ void pd_store(PdRecord *r, const PdRecord &v) {
    r->b = v.b;
    asm volatile("" ::: "memory");
    r->a = v.a;
}

// One stripe: rows of read positions p0 + kRows lane .. + kRows - 1.
template <int kRows, bool kGeneric>
__device__ __forceinline__ void pd_stripe(const PdBatch &b, const DeviceTables &tab, PdRecord *rec, const uint32_t *cds,
                                          int lane, int H, int64_t ro, int R, int p0) {
    PdLane<kRows> st;
    {
        PdRow w[kRows];
        bool real[kRows];
        double g[kRows];
        const int p = p0 + kRows * lane;
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            w[j] = pd_row(b, tab, ro, R, p + j);
            real[j] = p + j < R;
        }
        g[kRows - 1] = 1.0;
#pragma unroll
        for (int j = kRows - 2; j >= 0; --j) g[j] = real[j + 1] ? w[j + 1].pm * w[j + 1].MM * g[j + 1] : 1.0;
        const int p_next = p0 + kRows * kWave;
        double fold = 1.0;
        if constexpr (!kGeneric) {
            fold = pd_first_fold(b, tab, ro, R, p_next, pd_stripe_rows(R - p_next));
            fold = wave_shl1(fold, real[0] ? w[0].pm * g[0] : 1.0);
        }
        const PdRow below = pd_row(b, tab, ro, R, p + kRows);
        st.inside0 = p == 0 ? kPdInsideRow1 : kPdInsideLater;
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            const PdRow wn = j + 1 < kRows ? w[j + 1 < kRows ? j + 1 : 0] : below;
            const double f = kGeneric ? 1.0 : j + 1 < kRows ? wn.pm * g[j + 1 < kRows ? j + 1 : 0] : fold;
            const double inv_g = kGeneric || j + 1 == kRows ? 1.0 : 1.0 / g[j];
            st.MMr[j] = wn.MM * f;
            if (j + 1 == kRows) st.MMn = wn.MM * f;
            st.GMn[j] = wn.GM * f;
            st.MIn[j] = wn.MI * inv_g;
            st.IIn[j] = wn.II;
            st.MD[j] = w[j].MD * inv_g;
            st.DD[j] = w[j].DD;
            st.pm[j] = w[j].pm;
            st.px[j] = kGeneric ? w[j].px : real[j] ? w[j].px / w[j].pm : 0.0;
            // A pass-through row accepts nothing: M = 0.
            st.bit[j] = !real[j] ? 0u : kGeneric ? read_base_bit(w[j].x) : accept_bit(w[j].x);
            st.x[j] = real[j] ? w[j].x : 0x1FFu;
            st.inner[j] = __ballot(p + j < R - 1);
            st.EM[j] = st.EI[j] = st.ED[j] = st.bM[j] = st.bI[j] = st.bD[j] = st.an1[j] = 0.0;
        }
        st.an2 = st.bn1 = 0.0;
    }
    const int steps = round_up(H + kWave - 1, kPdU);
    const uint32_t *cp = cds + 1 - lane;  // column t - lane + 1 at step t
    PdRecord *wr = rec + 1 - lane;
    double a_first = rec[0].a;  // A of the block's first column
    for (int t0 = 0; t0 < steps; t0 += kPdU) {
        PdRecord cur[kPdU];
        uint32_t cc[kPdU];
        uint32_t any = 0;
#pragma unroll
        for (int u = 0; u < kPdU; ++u) {
            cur[u] = rec[t0 + u + 1];
            cc[u] = cp[t0 + u];
            any |= cc[u];
        }
        __builtin_amdgcn_wave_barrier();
        if (__builtin_amdgcn_ballot_w64((any & kPdSpecial) != 0u) != 0) {
#pragma unroll
            for (int u = 0; u < kPdU; ++u)
                pd_store(wr + t0 + u, pd_step<kRows, true, kGeneric>(st, u == 0 ? a_first : cur[u - 1].a, cur[u].b, cc[u]));
        } else {
#pragma unroll
            for (int u = 0; u < kPdU; ++u)
                pd_store(wr + t0 + u, pd_step<kRows, false, kGeneric>(st, u == 0 ? a_first : cur[u - 1].a, cur[u].b, cc[u]));
        }
        a_first = cur[kPdU - 1].a;
        __builtin_amdgcn_wave_barrier();
    }
}

__device__ __forceinline__ void pd_wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Every stripe of a pair; the records end holding M(R,c) + I(R,c) in b.
template <bool kGeneric>
__device__ __forceinline__ void pd_pair(const PdBatch &b, const DeviceTables &tab, PdRecord *rec, const uint32_t *cds,
                                        int lane, int H, int64_t ro, int R) {
    for (int p0 = 0; p0 < R;) {
        const int rows = pd_stripe_rows(R - p0);
        if (rows == 2)
            pd_stripe<2, kGeneric>(b, tab, rec, cds, lane, H, ro, R, p0);
        else
            pd_stripe<1, kGeneric>(b, tab, rec, cds, lane, H, ro, R, p0);
        p0 += rows * kWave;
        pd_wave_sync();
    }
}

// Column codes of one haplotype per workgroup (layout in pairhmm_kernels.hpp).  A column is processed inside
// a deletion when the last column before it that starts or ends one starts one (and does not also end
// it), LoglessPDPairHMM.java:63-136; row 1 begins outside, every later row in the state the row before
// ended in (the state variable lives outside the row loop, :63), which is the same for all rows >= 2.  Bound by
// latency (a few chunks of loads and ballots per haplotype); the same loop on the host was a fifth of the
// call (81 reads of 100-250 by 65 haplotypes of 377: 467 us with it, 383 us with this kernel).
__global__ __launch_bounds__(kWave) void pd_codes_kernel(const uint8_t *__restrict__ bases, const uint8_t *__restrict__ pd,
                                                         const int64_t *__restrict__ hap_off,
                                                         const int32_t *__restrict__ hap_len, uint32_t *code,
                                                         uint32_t *odd_bases) {
    const int lane = static_cast<int>(threadIdx.x);
    const int64_t o = hap_off[blockIdx.x];
    const int H = hap_len[blockIdx.x];
    // Columns that start a deletion (and do not end one) and columns that start or end one, of a chunk.
    auto events = [&](int j0, uint64_t &starts, uint64_t &any) {
        const int j = j0 + lane;
        const uint32_t v = j < H ? pd[o + j] : 0u;
        starts = __ballot((v & (kPdByteDelStart | kPdByteDelEnd)) == kPdByteDelStart);
        any = __ballot((v & (kPdByteDelStart | kPdByteDelEnd)) != 0u);
        return v;
    };
    // Whether the last of the events `any` starts a deletion; `before` where there is none.
    auto inside_after = [](uint64_t starts, uint64_t any, bool before) {
        return any ? ((starts >> (kWave - 1 - __builtin_clzll(any))) & 1u) != 0u : before;
    };
    bool row1_end = false;
    for (int j0 = 0; j0 < H; j0 += kWave) {
        uint64_t starts, any;
        events(j0, starts, any);
        row1_end = inside_after(starts, any, row1_end);
    }
    bool row1 = false, later = row1_end;
    bool odd = false;
    const uint64_t below = lane == 0 ? 0ull : ~0ull >> (kWave - lane), upto = ~0ull >> (kWave - 1 - lane);
    for (int j0 = 0; j0 < H; j0 += kWave) {
        uint64_t starts, any;
        const uint32_t v = events(j0, starts, any);
        const int j = j0 + lane;
        if (j < H) {
            const uint32_t y = bases[o + j], alt = (v & kPdByteSnp) ? (v & kPdByteAlts) : 0u;
            uint32_t c = y | (alt << 8) | ((alt >> 3) * 0x11u * kPdAcceptA);  // an alternative accepts both cases
            if (y == 'N')  // an 'N' haplotype base matches every read base (:163)
                c |= (0xF8u << 8) | (0xFFu * kPdAcceptA) | kPdAcceptOther;
            else if (accept_bit(y) != kPdAcceptOther)
                c |= accept_bit(y);
            else
                odd = true;
            if (v & kPdByteDelEnd) c |= kPdDelEnd | kPdSpecial;
            if (inside_after(starts & below, any & below, row1)) c |= kPdInsideRow1 | kPdSpecial;
            if (inside_after(starts & below, any & below, later)) c |= kPdInsideLater | kPdSpecial;
            // The column before one inside a span.
            if (j + 1 < H && (inside_after(starts & upto, any & upto, row1) || inside_after(starts & upto, any & upto, later)))
                c |= kPdSpecial;
            code[o + j] = c;
        }
        row1 = inside_after(starts, any, row1);
        later = inside_after(starts, any, later);
    }
    if (__any(odd)) *odd_bases = 1u;
}

__global__ __launch_bounds__(kWave) __attribute__((amdgpu_waves_per_eu(4))) void pd_forward_kernel(
    PdBatch b, DeviceTables tab, uint32_t n_pairs, int rec_columns) {
    extern __shared__ PdRecord lds_rec[];
    PdRecord *const rec = lds_rec + kPdLowPad;
    uint32_t *const cds = reinterpret_cast<uint32_t *>(rec + rec_columns) + kPdLowPad;
    const int lane = static_cast<int>(threadIdx.x);
    for (int c = lane - kPdLowPad; c < 0; c += kWave) cds[c] = 0u;  // columns below 1 carry no code
    const double log10_init = log10(ldexp(1.0, Scale<double>::kExp));
    for (uint32_t k = blockIdx.x; k < n_pairs; k += gridDim.x) {
        const uint32_t pair = b.order ? b.order[k] : k;
        const int r = static_cast<int>(pair / static_cast<uint32_t>(b.n_haps));
        const int h = static_cast<int>(pair % static_cast<uint32_t>(b.n_haps));
        const int R = b.rd_len[r], H = b.hap_len[h];
        if (R == 0) {  // no rows: the final sum over row 0's M and I is 0
            b.out[pair] = -__builtin_inf();
            continue;
        }
        const uint32_t *codes = b.hap_code + b.hap_off[h];
        const int64_t ro = b.rd_off[r];
        const double d0 = ldexp(1.0, Scale<double>::kExp) / static_cast<double>(H);
        // Base quality 0 (pm = 0) and gap-open qualities under 4 (from there on MM >= 0.2) leave the fast
        // path, which divides by both.
        int low = 0;
        for (int p = lane; p < R; p += kWave)
            low |= b.rd_quals[ro + p] == 0 || b.rd_ins[ro + p] < 4 || b.rd_del[ro + p] < 4;
        const bool generic = *b.odd_bases != 0u || __any(low);
        // Row 1's sums over row 0 (M = I = 0, D = d0 on columns 0..H): A(c) = d0 GM_1 for 1 <= c <= H + 1.
        const double gm1 = pd_row(b, tab, ro, R, 0).GM * (generic ? 1.0 : pd_first_fold(b, tab, ro, R, 0, pd_stripe_rows(R)));
        __builtin_amdgcn_wave_barrier();
        for (int c = lane; c < H + kPdPadColumns && c < rec_columns; c += kWave) {
            pd_store(rec + c, PdRecord{0.0, c <= H ? d0 * gm1 : 0.0});
            cds[c] = (c >= 1 && c <= H) ? codes[c - 1] : 0u;
        }
        pd_wave_sync();
        if (generic)
            pd_pair<true>(b, tab, rec, cds, lane, H, ro, R);
        else
            pd_pair<false>(b, tab, rec, cds, lane, H, ro, R);
        double acc = 0.0;
        for (int c = 1 + lane; c <= H; c += kWave) acc += rec[c].b;
        // Every lane holds the same sum and stores the same value.
        b.out[pair] = log10(wave_sum(acc)) - log10_init;
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace

int pd_record_columns(int max_hap_len) { return max_hap_len + kPdPadColumns; }

size_t pd_lds_bytes(int max_hap_len) {
    return static_cast<size_t>(kPdLowPad + pd_record_columns(max_hap_len)) * (sizeof(PdRecord) + sizeof(uint32_t));
}

hipError_t launch_pd_codes(const uint8_t *bases, const uint8_t *pd, const int64_t *hap_off, const int32_t *hap_len,
                           int32_t n_haps, uint32_t *code, uint32_t *odd_bases, hipStream_t stream) {
    if (n_haps <= 0) return hipSuccess;
    hipLaunchKernelGGL(pd_codes_kernel, dim3(n_haps), dim3(kWave), 0, stream, bases, pd, hap_off, hap_len, code, odd_bases);
    return hipGetLastError();
}

hipError_t launch_pd_forward(const PdBatch &batch, const DeviceTables &tables, uint32_t n_pairs, int max_hap_len,
                             int grid_blocks, hipStream_t stream) {
    if (n_pairs == 0) return hipSuccess;
    const size_t lds = pd_lds_bytes(max_hap_len);
    if (lds > max_lds_per_block()) return hipErrorInvalidValue;
    if (grid_blocks < 1) grid_blocks = 1;
    if (lds > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(pd_forward_kernel),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    hipLaunchKernelGGL(pd_forward_kernel, dim3(grid_blocks), dim3(kWave), lds, stream, batch, tables, n_pairs,
                       pd_record_columns(max_hap_len));
    return hipGetLastError();
}

}  // namespace gatk_pairhmm
