// pairhmm_fwd.hip -- gfx950 PairHMM forward kernels (FP32 bulk pass and FP64 pass).
//
// Model: LoglessPairHMM.subComputeReadLikelihoodGivenHaplotypeLog10
// (src/main/java/org/broadinstitute/hellbender/utils/pairhmm/LoglessPairHMM.java:20-68):
//   M(r,c) = prior(r,c) * (M(r-1,c-1) MM_r + I(r-1,c-1) GM_r + D(r-1,c-1) GM_r)
//   I(r,c) = M(r-1,c) MI_r + I(r-1,c) II_r
//   D(r,c) = M(r,c-1) MD_r + D(r,c-1) DD_r
// with M(0,.) = I(0,.) = 0, D(0,.) = 2^S / H, column 0 zero, and
// log10 L = log10(sum_c M(R,c) + I(R,c)) - S log10 2.  Row r uses the qualities of read base r-1
// (PairHMMModel.java:169-171); priors follow LoglessPairHMM.java:84-92 with tristate correction.
//
// Mapping onto a CDNA wavefront (one read/haplotype pair per wave):
//   * Rows are processed in stripes of 64, one row per lane: lane k owns row 64 s + k + 1 of stripe
//     s and keeps its row's six transition probabilities and two priors in registers.
//   * At step t lane k computes column c = t - k (an anti-diagonal sweep).  Its upper neighbours
//     (row above, columns c and c-1) are lane k-1's values from the last two steps; they arrive as
//     DPP wave_shr:1 source operands of v_mul / v_fmac, so the exchange costs no instructions of
//     its own.
//   * Lane 0's row above is the last row of the previous stripe, which lane 63 wrote into LDS
//     boundary planes as it went.  Lane 0 does not read that row cell by cell: it takes two
//     ready-made sums per column, A(c) (its diagonal term) and B(c) (its vertical term), 8 columns
//     per LDS read ahead of use, and the DPP products leave lane 0's preloaded value in place
//     (wave_shr:1 without bound_ctrl), so no step waits on LDS.  FP32 forms A and B in a side pass
//     over the planes lane 63 left; FP64, whose planes are twice as large, has every row form the
//     sums of the row below it, and gives a lane up to four rows.
//   * Rows past R on the last stripe pass the last row down (M = D = 0, I = M + I of the row
//     above), so the last stripe's planes end up holding M(R,c) + I(R,c).
//   * Cells with c <= 0 or c > H are computed too (they are exact zeros, resp. never read by a real
//     cell), which keeps the inner loop free of masks.
//   * The last-row sum, the unscaling and log10 are done in FP64.  FP32 launches use S = 120 and
//     flag pairs whose scaled sum is below the underflow threshold for an FP64 recompute (S = 1020).
//   * Launches are per LDS column class (kColClasses): a wave's LDS slice holds the haplotype and
//     the planes for the class's longest haplotype, so short haplotypes get more waves per CU.
#include <algorithm>

#include "pairhmm_device.hpp"
#include "pairhmm_kernels.hpp"

namespace gatk_pairhmm {
namespace {

using namespace dev;

constexpr int kUnroll = 8;  // wave-steps per unrolled loop body

// Every lane stores its cell at its own column, so a column is stored by all lanes, a step apart, and the last
// store, lane 63's, has to come last.  The compiler sees one lane, whose stores are to different addresses,
// and its schedulers reorder them unless the steps are held apart.  FP32 steps are held apart in pairs:
// two steps' stores go out as one ds_write2, lower column first (single stores: 44.8 against 39.7 ms on 300
// regions, LDS-bound).  check_isa.py checks the order in the assembly.
__device__ __forceinline__ void store_order() { asm volatile("" ::: "memory"); }

template <typename T>
struct WaveLds {
    uint8_t *hap;      // [cols]: haplotype byte of column c (1-based) at kLdsPad + c - 1
    T *bm, *bi;        // [cols]: boundary planes, column c at kLdsPad + c
    T *ring;           // FP64: LDS ring of the rows' (B, A) sums for the next row (kRing64 slots)
};

template <int kCols>
constexpr int plane_stride() { return lds_plane_stride(kCols); }

// Plane slots lane 0 reads over a stripe of `steps` wave-steps (8-column blocks from slot kLdsPad),
// rounded up to whole 64-slot chunks of the side pass; never more than kCols.
template <int kCols>
__device__ __forceinline__ int plane_span(int steps) {
    const int j = round_up(kLdsPad + steps, kWave);
    return j < kCols ? j : kCols;
}

// Two boundary planes per wave: lane 63's row (FP32: M and I in LDS, turned into lane 0's sums A
// and B by the side pass; FP64: A and B formed by lane 63 itself, in global memory).
constexpr int kPlanes = 2;
// FP64 step loop: every lane stores the sums it forms for the row below, (B(c), A(c+1)), at its
// own column into an LDS ring of 128 slots (plus 8 for a block that runs past slot 127), from which
// each 8-step block copies lane 63's finished columns out as lane 0's sums of the next stripe.
constexpr int kRing64 = 136;
constexpr size_t kRing64Bytes = kRing64 * 2 * sizeof(double);

template <typename T, int kCols>
constexpr size_t lds_per_wave() {
    return static_cast<size_t>(kCols) + (sizeof(T) == sizeof(float)
                                             ? kPlanes * static_cast<size_t>(plane_stride<kCols>()) * sizeof(T)
                                             : kRing64Bytes);
}

// Transition probabilities and priors of the row that read position p feeds (PairHMMModel.java:
// 158-172, LoglessPairHMM.java:84-92); positions past the read give the pass-through row
// (MI = II = 1, everything else 0).
template <typename T>
struct RowTrans {
    T MM, GM, MI, II, MD, DD, pm, px;
    uint32_t base;
};

template <typename T>
__device__ __forceinline__ RowTrans<T> row_trans(int p, int R, const uint8_t *__restrict__ rb,
                                                 const uint8_t *__restrict__ rq, const uint8_t *__restrict__ ri,
                                                 const uint8_t *__restrict__ rd, const uint8_t *__restrict__ rg,
                                                 const DeviceTables &tab) {
    RowTrans<T> w{0, 0, 0, 0, 0, 0, 0, 0, 0u};
    if (p < R) {
        w.base = rb[p];
        const int q = rq[p], qi = ri[p], qd = rd[p], qc = rg[p];
        const double eq = tab.qual_err[q], ei = tab.qual_err[qi], ed = tab.qual_err[qd], ec = tab.qual_err[qc];
        const int mn = qi < qd ? qi : qd, mx = qi < qd ? qd : qi;
        w.MM = static_cast<T>(tab.mm_prob[((mx * (mx + 1)) >> 1) + mn]);
        w.MI = static_cast<T>(ei);
        w.MD = static_cast<T>(ed);
        w.GM = static_cast<T>(1.0 - ec);
        w.II = static_cast<T>(ec);
        w.DD = w.II;
        w.pm = static_cast<T>(1.0 - eq);
        w.px = static_cast<T>(tab.qual_err[256 + q]);  // eq / 3.0
        if (w.base == 'N') w.px = w.pm;
    } else {
        // Rows past R pass the last row down unchanged: M = D = 0 and I(r,c) = M(r-1,c) + I(r-1,c).
        w.MI = 1;
        w.II = 1;
    }
    return w;
}

// A wave's haplotype bytes (LDS) and boundary planes: LDS for FP32, the wave's slice of the global
// FP64 planes otherwise.
template <typename T, int kCols>
__device__ __forceinline__ WaveLds<T> carve(uint8_t *base, const DeviceBatch &b, size_t gwave) {
    WaveLds<T> w;
    w.hap = base;
    if constexpr (sizeof(T) == sizeof(float)) {
        w.bm = reinterpret_cast<T *>(base + kCols);
        w.ring = nullptr;
    } else {
        w.bm = b.f64_planes + gwave * kPlanes * static_cast<size_t>(plane_stride<kCols>());
        w.ring = reinterpret_cast<T *>(base + kCols);
    }
    w.bi = w.bm + plane_stride<kCols>();
    return w;
}


// Side pass before stripe s > 0.  Lane 63 left the previous stripe's last row r in the two planes
// (M in P0, I in P1).  The pass rebuilds D of that row from its own recurrence,
//   D(c) = M(c-1) MD' + D(c-1) DD'   (MD', DD' of row r),
// and turns the row into lane 0's sums in place, in ascending column order:
//   A(c) = M(c-1) MM0 + (I(c-1) + D(c-1)) GM0 over M,   B(c) = M(c) MI0 + I(c) II0 over I.
// Per 64-column chunk D is a linear scan (linear_scan64) plus the carry D(j0-1) DD'^(l+1); column
// j0-1's M, I and D come from the previous chunk's lane 63 (the chunk itself is already overwritten).
// The pass covers plane slots [0, jmax) (jmax a multiple of 64, at most kCols): the slots lane 0 of
// the next stripe reads.  cd0 is D left of slot 0 (0 for every row but a constant one).  Lane 63
// wrote slots [1, wend) in the previous stripe (column t - 63 at step t); slot 0 and slots from wend
// on still hold what earlier passes left there and are read as M = I = 0.  Leftovers past a
// shorter stripe's end, turned over again by every later pass, can grow to inf, and a summing row
// that meets inf beyond its haplotype (times its prior 0) turns NaN.
//
// SidePass holds what goes from chunk to chunk, so a wave that works on a row while another still
// computes it (forward_kernel_split) can take the chunks one at a time.
struct SidePass {
    float MM0, GM0, MI0, II0, MDr;
    float a1, a2, a4, a8, p_row, p_in, p_31;
    float cm = 0.f, ci = 0.f, cd;  // M, I, D of column j0 - 1

    __device__ __forceinline__ SidePass(int lane, float MM0, float GM0, float MI0, float II0, float MDr, float DDr,
                                        float cd0)
        : MM0(MM0), GM0(GM0), MI0(MI0), II0(II0), MDr(MDr), cd(cd0) {
        a1 = DDr;
        a2 = a1 * a1;
        a4 = a2 * a2;
        a8 = a4 * a4;
        const float a16 = a8 * a8, a32 = a16 * a16;
        // DD'^((l mod 16) + 1) by the bits of l mod 16, then the row's 16-lane steps on top:
        // p_in = DD'^(l+1), p_31 = DD'^(l-31) for l >= 32 (1 below).
        p_row = a1;
        p_row = (lane & 1) ? p_row * a1 : p_row;
        p_row = (lane & 2) ? p_row * a2 : p_row;
        p_row = (lane & 4) ? p_row * a4 : p_row;
        p_row = (lane & 8) ? p_row * a8 : p_row;
        const float p_16 = (lane & 16) ? p_row * a16 : p_row;
        p_in = (lane & 32) ? p_16 * a32 : p_16;
        p_31 = (lane & 32) ? p_16 : 1.f;
    }

    // Chunk of slots j0 .. j0 + 63.
    __device__ __forceinline__ void chunk(float *P0, float *P1, int lane, int j0, int wend) {
        const int j = j0 + lane;
        const bool written = j >= kLdsPad - (kWave - 1) && j < wend;
        const float mj = written ? P0[j] : 0.f, ij = written ? P1[j] : 0.f;
        const float mprev = wave_shr1(cm, mj), iprev = wave_shr1(ci, ij);
        const float dj = fmaf(cd, p_in, linear_scan64(mprev * MDr, a1, a2, a4, a8, p_row, p_31));
        const float dprev = wave_shr1(cd, dj);
        __builtin_amdgcn_wave_barrier();
        P0[j] = fmaf(iprev + dprev, GM0, mprev * MM0);
        P1[j] = fmaf(ij, II0, mj * MI0);
        cm = lane63(mj);
        ci = lane63(ij);
        cd = lane63(dj);
        __builtin_amdgcn_wave_barrier();
    }
};

template <int kCols>
__device__ __forceinline__ void side_pass_f32(float *P0, float *P1, int lane, float MM0, float GM0, float MI0,
                                              float II0, float MDr, float DDr, int jmax, float cd0 = 0.f,
                                              int wend = kCols) {
    SidePass side(lane, MM0, GM0, MI0, II0, MDr, DDr, cd0);
    __builtin_amdgcn_wave_barrier();
    for (int j0 = 0; j0 < jmax; j0 += kWave) side.chunk(P0, P1, lane, j0, wend);
}

// One pass over a pair, stripe by stripe.  Returns the scaled last-row sum (FP64, every lane).
//
// Stripe s covers rows 64 s + 1 .. 64 s + 64, one per lane.  Per step each lane keeps its own M, I,
// D from the previous step and M, S = I + D from two steps back:
//   M(r,c) = prior * (M(r-1,c-1) MM + S(r-1,c-1) GM)     [lane k-1, two steps back]
//   I(r,c) = M(r-1,c) MI + I(r-1,c) II                    [lane k-1, one step back]
//   D(r,c) = M(r,c-1) MD + D(r,c-1) DD                    [own lane, one step back]
// Lane 0's row above is the last row of the previous stripe, which lane 63 left in the LDS
// boundary planes (M and I; D is rebuilt by the side pass).  Before the stripe the side pass turns
// those planes into lane 0's two sums,
//   A(c) = M(r-1,c-1) MM + S(r-1,c-1) GM   and   B(c) = M(r-1,c) MI + I(r-1,c) II,
// in place (A over M, B over I).  Lane 0 reads them ahead with wave-uniform loads and brings them
// into the DPP products, which leave lane 0 unwritten, so no step waits on LDS.
template <typename T, int kCols, bool kHapHasN>
__device__ double forward_pair_f32(const WaveLds<T> &L, int lane, int H, int R, const uint8_t *__restrict__ rb,
                               const uint8_t *__restrict__ rq, const uint8_t *__restrict__ ri,
                               const uint8_t *__restrict__ rd, const uint8_t *__restrict__ rg,
                               const DeviceTables &tab) {
    constexpr int kStripe = kWave;
    const int n_stripes = (R + kStripe - 1) / kStripe;
    const int steps = round_up(H + kWave, kUnroll);
    const int jmax = plane_span<kCols>(steps);
    for (int s = 0; s < n_stripes; ++s) {
        const RowTrans<T> w = row_trans<T>(s * kStripe + lane, R, rb, rq, ri, rd, rg, tab);
        const T MM = w.MM, GM = w.GM, MI = w.MI, II = w.II, MD = w.MD, DD = w.DD, pm = w.pm, px = w.px;
        const uint32_t base = w.base;
        if (s > 0) {
            // Row 64 s (read position 64 s - 1) is the previous stripe's last row; wave-uniform.
            const RowTrans<T> up = row_trans<T>(s * kStripe - 1, R, rb, rq, ri, rd, rg, tab);
            side_pass_f32<kCols>(L.bm, L.bi, lane, rfl(MM), rfl(GM), rfl(MI), rfl(II), up.MD, up.DD, jmax);
        }
    T m1 = 0, i1 = 0, d1 = 0, s1 = 0;  // own cell one step back (column c-1)
        T m2 = 0, s2 = 0;                  // own cell two steps back (column c-2)
        // Byte loads of the haplotype, eight per block.  volatile keeps them from being merged into
        // unaligned 8-byte loads; the explicit LDS address space keeps them ds_read_u8.
        using lds_u8 = const volatile __attribute__((address_space(3))) uint8_t;
        lds_u8 *hp = (lds_u8 *)(L.hap + kLdsPad - 1 - lane);  // address-space cast: C-style only
        // Every lane stores its M and I at its own column c = t - lane at step t (no one-lane exec
        // mask in the step).  Lane 63 writes column c last, at step c + 63, so the planes end with
        // its row; lane 0 reads A, B of column c by step c, before any lane overwrites it.
        using lds_t = __attribute__((address_space(3))) T;
        int lane_w = lane;
        asm volatile("" : "+v"(lane_w));
        lds_t *wm = (lds_t *)(L.bm + kLdsPad) - lane_w, *wi = (lds_t *)(L.bi + kLdsPad) - lane_w;
        for (int t0 = 0; t0 < steps; t0 += kUnroll) {
            lds_t *wmb = wm + t0, *wib = wi + t0;
            T av[kUnroll], bv[kUnroll];
            __builtin_memcpy(av, __builtin_assume_aligned(L.bm + kLdsPad + t0, 16), sizeof(av));
            __builtin_memcpy(bv, __builtin_assume_aligned(L.bi + kLdsPad + t0, 16), sizeof(bv));
            uint32_t hbs[kUnroll];
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) hbs[u] = hp[t0 + u];
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int u = 0; u < kUnroll; ++u) {
                const uint32_t hb = hbs[u];
                const bool match = (hb == base) || (kHapHasN && hb == 'N');
                const T prior = match ? pm : px;
                T a = av[u], i = bv[u];
                dpp_upper2(a, m2, MM, s2, GM, i, m1, MI, i1, II);
                const T m = a * prior;
                // The lane carries D' = D / MD: D'(c) = M(c-1) + D'(c-1) DD and S = I + MD D', one FMA
                // each instead of a multiply, an FMA and an add.  D' <= sum_c M(r,c), so it keeps
                // FP32's range even where DD is close to 1.
                const T d = fma(d1, DD, m1);
                const T sx = fma(MD, d, i);
                wmb[u] = m;
                wib[u] = i;
                if (u % 2 == 1) store_order();
                m2 = m1;
                s2 = s1;
                m1 = m;
                i1 = i;
                d1 = d;
                s1 = sx;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    double acc = 0.0;
    for (int c = 1 + lane; c <= H; c += kWave)
        acc += static_cast<double>(L.bm[kLdsPad + c]) + static_cast<double>(L.bi[kLdsPad + c]);
    return wave_sum(acc);
}

// FP64 pass.  A lane owns kRows consecutive rows and computes the same column of all of them at a
// step: 4 rows (a stripe of 256) while more than 192 are left, then 2, then 1 for a last part of up to
// 64, so a read is padded to 64 rows as with one row per lane.
// Each row forms the sums the row below it needs from its own new M, S and I, with the transitions
// of the row below:
//   A(c+1) = M(c) MM' + S(c) GM'   and   B(c) = M(c) MI' + I(c) II'.
// Within a lane the row below takes B at once and A at the next step; the next lane's first row takes
// them one lane over: B at the next step (same column), A two steps later (the next column).  So two
// doubles cross lanes per step (four 32-bit DPP moves) for kRows cells.  The last row's
// sums of lane 63 are lane 0's A and B of the next stripe; after the last stripe the next row is the
// pass-through row (MM = GM = 0, MI = II = 1), so the B plane ends up holding M(R,c) + I(R,c).  Lane 0
// takes A and B as the old values of the DPP moves (wave_shr:1 without bound_ctrl leaves lane 0
// unwritten).
//
// The prior: a row's match prior pm is folded into the transitions that form its A, so that a match
// leaves M = A and only a mismatch multiplies, by px / pm, in the lanes that have one (an EXEC mask
// around one product: two VALU instructions where a compare, two selects and a product were four).
// An 'N' in the haplotype and qualities whose pm or MM is near 0 take the selects (kGeneric).
//
// Bound by VALU issue: 33 instructions per step of four cells and about 2 of block overhead, where one
// row per lane and selected priors took 15 a cell.  Precision stress (40 regions, 1.07e11 cells, all
// launches): 67.1 ms then, 49.2 with two rows per lane at 4 waves per SIMD, 45.2 with four at 3
// (168 VGPRs), 43.2 with M's factor folded.
//
// Every lane stores its (B(c), A(c+1)) at its own column c = t - lane into an LDS ring at step t (no
// one-lane exec mask in the step); lane 63 writes column c last, at step c + 63.  After each block
// of 8 steps the whole wave copies lane 63's 8 columns finished in it out to the plane, one 16-byte
// store per column, with every lane storing (lanes 8-63 repeat lanes 0-7).  A lane's ring slots for
// block t0 start at (t0 - lane) mod 128, so a block never wraps and two live columns (less than 128
// apart) never share a slot.
//
// A and B live in the wave's slice of global memory rather than LDS (an FP64 plane is 8 bytes a
// column; in LDS the long-haplotype classes held a CU to 5-7 waves); the slice stays in L2.  They
// are interleaved, P[2 j] = A and P[2 j + 1] = B at j = kLdsPad + c, so a block's 8 columns are 16
// contiguous doubles.  Lane 0's values are read through a VGPR address (an opaque zero offset keeps
// the compiler from turning the uniform load into a scalar one, whose cache does not see vector
// stores) and rolled in half a block ahead of use: after step 3 a block's first half of the buffer
// is reloaded with the next block's first four columns, after step 7 the second half.  A wait for
// the wave's stores at each stripe start orders the previous stripe's stores before these loads;
// all accesses come from one wave on one CU, so its L1 holds no stale copy.

// Per row, in the lanes whose haplotype byte differs from the row's base: a *= ratio.  EXEC is all ones
// before and after (whole waves, uniform control flow); the s_nop completes the five wait states a DPP
// needs after a VALU write of EXEC, which the compiler does not track across inline assembly.
__device__ __forceinline__ void scale_mismatch(double (&a)[1], const double (&ratio)[1], uint32_t hb,
                                               const uint32_t (&base)[1]) {
    asm("v_cmpx_ne_u32_e32 vcc, %2, %3\n\t"
        "v_mul_f64 %0, %0, %1\n\t"
        "s_mov_b64 exec, -1\n\t"
        "s_nop 2"
        : "+&v"(a[0])
        : "v"(ratio[0]), "v"(hb), "v"(base[0])
        : "vcc");
}
__device__ __forceinline__ void scale_mismatch(double (&a)[2], const double (&ratio)[2], uint32_t hb,
                                               const uint32_t (&base)[2]) {
    asm("v_cmpx_ne_u32_e32 vcc, %4, %5\n\t"
        "v_mul_f64 %0, %0, %2\n\t"
        "s_mov_b64 exec, -1\n\t"
        "v_cmpx_ne_u32_e32 vcc, %4, %6\n\t"
        "v_mul_f64 %1, %1, %3\n\t"
        "s_mov_b64 exec, -1\n\t"
        "s_nop 2"
        : "+&v"(a[0]), "+&v"(a[1])
        : "v"(ratio[0]), "v"(ratio[1]), "v"(hb), "v"(base[0]), "v"(base[1])
        : "vcc");
}
__device__ __forceinline__ void scale_mismatch(double (&a)[4], const double (&ratio)[4], uint32_t hb,
                                               const uint32_t (&base)[4]) {
    asm("v_cmpx_ne_u32_e32 vcc, %8, %9\n\t"
        "v_mul_f64 %0, %0, %4\n\t"
        "s_mov_b64 exec, -1\n\t"
        "v_cmpx_ne_u32_e32 vcc, %8, %10\n\t"
        "v_mul_f64 %1, %1, %5\n\t"
        "s_mov_b64 exec, -1\n\t"
        "v_cmpx_ne_u32_e32 vcc, %8, %11\n\t"
        "v_mul_f64 %2, %2, %6\n\t"
        "s_mov_b64 exec, -1\n\t"
        "v_cmpx_ne_u32_e32 vcc, %8, %12\n\t"
        "v_mul_f64 %3, %3, %7\n\t"
        "s_mov_b64 exec, -1\n\t"
        "s_nop 2"
        : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
        : "v"(ratio[0]), "v"(ratio[1]), "v"(ratio[2]), "v"(ratio[3]), "v"(hb), "v"(base[0]), "v"(base[1]),
          "v"(base[2]), "v"(base[3])
        : "vcc");
}

// Rows per lane of the stripe that starts with `left` rows to go.
__device__ __forceinline__ int f64_stripe_rows(int left) {
    return left > 3 * kWave ? 4 : left > kWave ? 2 : 1;
}

// What a row's M is multiplied with along a lane (fast path): g = pm' MM' g' of the row below it in the
// lane, 1 for the lane's last row and above a pass-through row.  The row below takes A with pm' g'
// folded in, so M's term in it has the factor 1 and costs no product.
template <int kRows>
__device__ __forceinline__ void f64_scales(const RowTrans<double> (&w)[kRows], const bool (&real)[kRows],
                                           double (&g)[kRows]) {
    g[kRows - 1] = 1.0;
#pragma unroll
    for (int j = kRows - 2; j >= 0; --j) g[j] = real[j + 1] ? w[j + 1].pm * w[j + 1].MM * g[j + 1] : 1.0;
}

// The factor folded into the sums that reach the row at read position p, the first of its lane in a
// stripe of `rows` rows per lane (wave-uniform arguments).
__device__ __forceinline__ double f64_first_fold(int p, int rows, int R, const uint8_t *__restrict__ rb,
                                                 const uint8_t *__restrict__ rq, const uint8_t *__restrict__ ri,
                                                 const uint8_t *__restrict__ rd, const uint8_t *__restrict__ rg,
                                                 const DeviceTables &tab) {
    double f = 1.0;
    for (int j = 0; j < rows && p + j < R; ++j) {
        const RowTrans<double> w = row_trans<double>(p + j, R, rb, rq, ri, rd, rg, tab);
        f *= j == 0 ? w.pm : w.pm * w.MM;
    }
    return f;
}

// One stripe: rows of read positions p0 + kRows lane .. + kRows - 1.
template <int kRows, bool kGeneric>
__device__ __forceinline__ void f64_stripe(double *P, __attribute__((address_space(3))) double *const ring,
                                           const volatile __attribute__((address_space(3))) uint8_t *hp, int lane,
                                           int steps, int p0, int R, const uint8_t *__restrict__ rb,
                                           const uint8_t *__restrict__ rq, const uint8_t *__restrict__ ri,
                                           const uint8_t *__restrict__ rd, const uint8_t *__restrict__ rg,
                                           const DeviceTables &tab) {
    using lds_f64 = __attribute__((address_space(3))) double;
    constexpr int kLag = kWave - 1;
    int zoff;
    asm volatile("v_mov_b32 %0, 0" : "=v"(zoff));
    const double *r0 = P + 2 * kLdsPad + zoff;
    // Copy-out: lane handles column offset v of the block's finished columns.
    const int v = lane & (kUnroll - 1);
    // Row j's own MD, DD and priors; the transitions of the row below it (n).  Generic: px is the
    // mismatch prior.  Fast: pm is folded into the sums, px is px / pm, M carries the factor g.
    double MD[kRows], DD[kRows], pm[kRows], px[kRows], MMn[kRows], GMn[kRows], MIn[kRows], IIn[kRows];
    uint32_t base[kRows];
    {
        RowTrans<double> w[kRows];
        bool real[kRows];
        double g[kRows];
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            w[j] = row_trans<double>(p0 + kRows * lane + j, R, rb, rq, ri, rd, rg, tab);
            real[j] = p0 + kRows * lane + j < R;
        }
        f64_scales(w, real, g);
        const int p_next = p0 + kRows * kWave;
        double fold = 1.0;
        if constexpr (!kGeneric) {
            fold = f64_first_fold(p_next, f64_stripe_rows(R - p_next), R, rb, rq, ri, rd, rg, tab);
            fold = wave_shl1(fold, real[0] ? w[0].pm * g[0] : 1.0);
        }
        const RowTrans<double> below = row_trans<double>(p0 + kRows * lane + kRows, R, rb, rq, ri, rd, rg, tab);
#pragma unroll
        for (int j = 0; j < kRows; ++j) {
            const RowTrans<double> wn = j + 1 < kRows ? w[j + 1 < kRows ? j + 1 : 0] : below;
            const double f = kGeneric ? 1.0 : j + 1 < kRows ? wn.pm * g[j + 1 < kRows ? j + 1 : 0] : fold;
            const double inv_g = kGeneric || j + 1 == kRows ? 1.0 : 1.0 / g[j];
            MMn[j] = wn.MM * f;
            GMn[j] = wn.GM * f;
            MIn[j] = wn.MI * inv_g;
            IIn[j] = wn.II;
            MD[j] = w[j].MD * inv_g;
            DD[j] = w[j].DD;
            pm[j] = w[j].pm;
            px[j] = kGeneric ? w[j].px : real[j] ? w[j].px / w[j].pm : 0.0;
            base[j] = kGeneric || real[j] ? w[j].base : 0x1FFu;  // a pass-through row matches nothing: M = 0
        }
    }
    // dd = D / MD: D(c) = D(c-1) DD + M(c-1) MD becomes dd(c) = dd(c-1) DD + M(c-1), and
    // S = I + D = I + MD dd, one FMA each (rows past R have MD = DD = 0, so S = I there).
    double m[kRows] = {}, dd[kRows] = {};
    double an1[kRows] = {}, an2 = 0, bn1 = 0;  // sums for the row below; the last row's two steps back
    // The previous stripe's (or the initial) stores complete before this stripe reads them.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    double ab[2 * kUnroll];
    __builtin_memcpy(ab, __builtin_assume_aligned(r0, 16), sizeof(ab));
    for (int t0 = 0; t0 < steps; t0 += kUnroll) {
        lds_f64 *wr = ring + 2 * ((t0 - lane) & 127);
        uint32_t hbs[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) hbs[u] = hp[t0 + u];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) {
            const uint32_t hb = hbs[u];
            double a[kRows];
            double i = wave_shr1(ab[2 * u + 1], bn1);  // lane 0 keeps its plane values
            a[0] = wave_shr1(ab[2 * u], an2);
#pragma unroll
            for (int j = 1; j < kRows; ++j) a[j] = an1[j - 1];
            an2 = an1[kRows - 1];
            if constexpr (!kGeneric) scale_mismatch(a, px, hb, base);
            double an = 0, bn = 0;
#pragma unroll
            for (int j = 0; j < kRows; ++j) {
                if constexpr (kGeneric) a[j] *= (hb == base[j] || hb == 'N') ? pm[j] : px[j];
                dd[j] = fma(dd[j], DD[j], m[j]);
                m[j] = a[j];
                const double sx = fma(dd[j], MD[j], i);
                an = fma(sx, GMn[j], kGeneric || j + 1 == kRows ? m[j] * MMn[j] : m[j]);
                bn = fma(i, IIn[j], m[j] * MIn[j]);
                an1[j] = an;
                i = bn;
            }
            bn1 = bn;
            wr[2 * u] = bn;
            wr[2 * u + 1] = an;
            // Holds this step's stores before the next one's (store_order), as the address may be any other one from
            // here on; a barrier would hold the loads too (75 pairs, one after another's latency: 143 and 146 us).
            asm("" : "+v"(wr));
            // The next block's halves, loaded unconditionally (the slice has slots past the last
            // block): with a fixed count of loads in the loop, the wait for a half is a counted
            // one instead of a full drain at the block start.
            if (u == kUnroll / 2 - 1)
                __builtin_memcpy(ab, __builtin_assume_aligned(r0 + 2 * (t0 + kUnroll), 16), sizeof(ab) / 2);
            if (u == kUnroll - 1)
                __builtin_memcpy(ab + kUnroll, __builtin_assume_aligned(r0 + 2 * (t0 + kUnroll) + kUnroll, 16),
                                 sizeof(ab) / 2);
        }
        __builtin_amdgcn_wave_barrier();
        // Lane 63 finished columns t0 - 63 .. t0 - 56 in this block, at ring slots
        // ((t0 - 63) mod 128) + v: (B(c), A(c + 1)) as they go to the plane.
        {
            const lds_f64 *rs = ring + 2 * (((t0 - kLag) & 127) + v);
            const double ba[2] = {rs[0], rs[1]};
            __builtin_memcpy(P + 2 * (kLdsPad + t0 - kLag + v) + 1, ba, sizeof(ba));
        }
        __builtin_amdgcn_wave_barrier();
    }
    __builtin_amdgcn_wave_barrier();
}

template <int kCols, bool kGeneric>
__device__ double forward_pair_f64(const WaveLds<double> &L, int lane, int H, int R, const uint8_t *__restrict__ rb,
                                   const uint8_t *__restrict__ rq, const uint8_t *__restrict__ ri,
                                   const uint8_t *__restrict__ rd, const uint8_t *__restrict__ rg,
                                   const DeviceTables &tab) {
    const int steps = round_up(H + kWave, kUnroll);
    double *P = L.bm;  // A(c) at 2 (kLdsPad + c), B(c) at 2 (kLdsPad + c) + 1
    using lds_u8 = const volatile __attribute__((address_space(3))) uint8_t;
    lds_u8 *hp = (lds_u8 *)(L.hap + kLdsPad - 1 - lane);  // address-space cast: C-style only
    using lds_f64 = __attribute__((address_space(3))) double;
    lds_f64 *const ring = (lds_f64 *)L.ring;  // slot k: B at 2 k, A at 2 k + 1
    for (int p0 = 0; p0 < R;) {
        const int rows = f64_stripe_rows(R - p0);
        if (rows == 4)
            f64_stripe<4, kGeneric>(P, ring, hp, lane, steps, p0, R, rb, rq, ri, rd, rg, tab);
        else if (rows == 2)
            f64_stripe<2, kGeneric>(P, ring, hp, lane, steps, p0, R, rb, rq, ri, rd, rg, tab);
        else
            f64_stripe<1, kGeneric>(P, ring, hp, lane, steps, p0, R, rb, rq, ri, rd, rg, tab);
        p0 += rows * kWave;
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last stripe's B values are complete
    double acc = 0.0;
    for (int c = 1 + lane; c <= H; c += kWave) acc += P[2 * (kLdsPad + c) + 1];
    return wave_sum(acc);
}

// kGeneric: the haplotype has an 'N' (FP64: or the read a base quality of 0).
template <typename T, int kCols, bool kGeneric>
__device__ __forceinline__ double forward_pair(const WaveLds<T> &L, int lane, int H, int R, const uint8_t *rb,
                                               const uint8_t *rq, const uint8_t *ri, const uint8_t *rd,
                                               const uint8_t *rg, const DeviceTables &tab) {
    if constexpr (sizeof(T) == sizeof(double))
        return forward_pair_f64<kCols, kGeneric>(L, lane, H, R, rb, rq, ri, rd, rg, tab);
    else
        return forward_pair_f32<T, kCols, kGeneric>(L, lane, H, R, rb, rq, ri, rd, rg, tab);
}

template <typename T, int kCols>
__device__ void process_pair(const DeviceBatch &b, const DeviceTables &tab, const RescueSink &rs, const WaveLds<T> &L,
                             int lane, uint32_t pair) {
    int r, h;
    if (b.pair_read) {
        r = b.pair_read[pair];
        h = b.pair_hap[pair];
    } else {
        r = static_cast<int>(pair / static_cast<uint32_t>(b.n_haps));
        h = static_cast<int>(pair % static_cast<uint32_t>(b.n_haps));
    }
    const int H = b.hap_len[h];
    const int R = b.rd_len[r];
    const uint8_t *hap = b.hap_bases + b.hap_off[h];
    const int64_t ro = b.rd_off[r];

    // Stage the haplotype (zero padded) and the row-0 boundary: M = I = 0, D = 2^S / H
    // (LoglessPairHMM.java:30-36).
    int has_n = 0;
    for (int j = lane; j < kCols; j += kWave) {
        const int c = j - kLdsPad + 1;  // hap byte j belongs to column c
        uint8_t v = 0;
        if (c >= 1 && c <= H) {
            v = hap[c - 1];
            has_n |= (v == 'N');
        }
        L.hap[j] = v;
    }
    const T d0 = static_cast<T>(__builtin_ldexp(1.0, Scale<T>::kExp) / static_cast<double>(H));
    // Row 1's sums over row 0 (M = I = 0, D = 2^S / H from column 0 on): A(c) = d0 GM_1 for c >= 1,
    // B(c) = 0 (FP32: A in the M plane, B in the I plane; FP64: interleaved, A at 2 j, B at 2 j + 1).
    const RowTrans<T> row1 = row_trans<T>(0, R, b.rd_bases + ro, b.rd_quals + ro, b.rd_ins + ro, b.rd_del + ro,
                                          b.rd_gcp + ro, tab);
    bool generic = __any(has_n);
    T gm1 = row1.GM;
    if constexpr (sizeof(T) == sizeof(double)) {
        // The fast path divides by match priors and MM: base quality 0 (pm = 0) and gap-open qualities
        // under 4 (from there on MM >= 0.2) take the generic one.
        int low = 0;
        for (int p = lane; p < R; p += kWave)
            low |= b.rd_quals[ro + p] == 0 || b.rd_ins[ro + p] < 4 || b.rd_del[ro + p] < 4;
        generic = generic || __any(low);
        if (!generic)
            gm1 *= f64_first_fold(0, f64_stripe_rows(R), R, b.rd_bases + ro, b.rd_quals + ro, b.rd_ins + ro,
                                  b.rd_del + ro, b.rd_gcp + ro, tab);
    }
    for (int j = lane; j < kCols; j += kWave) {
        const T a0 = j >= kLdsPad + 1 ? d0 * gm1 : T(0);
        if constexpr (sizeof(T) == sizeof(float)) {
            L.bm[j] = a0;
            L.bi[j] = 0;
        } else {
            L.bm[2 * j] = a0;
            L.bm[2 * j + 1] = 0;
        }
    }
    double sum;
    if (generic)
        sum = forward_pair<T, kCols, true>(L, lane, H, R, b.rd_bases + ro, b.rd_quals + ro, b.rd_ins + ro, b.rd_del + ro,
                                    b.rd_gcp + ro, tab);
    else
        sum = forward_pair<T, kCols, false>(L, lane, H, R, b.rd_bases + ro, b.rd_quals + ro, b.rd_ins + ro, b.rd_del + ro,
                                     b.rd_gcp + ro, tab);
    // Every lane holds the same sum (butterfly reduction), so the result and the rescue decision are
    // wave-uniform; all lanes store the same value to the same address rather than branching on
    // the lane id (a lane-divergent branch here would sit next to the convergent work fetch below).
    const double scale_log10 = static_cast<double>(Scale<T>::kExp) * 0.30102999566398119521;
    b.out[pair] = log10(sum) - scale_log10;
    if (rs.list != nullptr) {
        const int need = __builtin_amdgcn_readfirstlane(static_cast<int>(!(sum >= rs.threshold)));
        if (need) {
            const uint32_t slot = __builtin_amdgcn_readfirstlane(atomicAdd(rs.count, lane == 0 ? 1u : 0u));
            rs.list[slot] = pair;
        }
    }
}

template <typename T, int kCols>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(sizeof(T) == sizeof(double) ? 3 : 1)))
void forward_kernel(DeviceBatch b, DeviceTables tab, WorkSource ws, RescueSink rs) {
    extern __shared__ __align__(16) uint8_t lds_raw[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const int waves_per_block = blockDim.x / kWave;
    constexpr size_t kPerWave = lds_per_wave<T, kCols>();
    const size_t gwave = static_cast<size_t>(blockIdx.x) * waves_per_block + wave;
    // FP64 waves past the planes' capacity stay idle (queue launches only; grid-stride launches are
    // sized to the capacity by the host).
    if (sizeof(T) == sizeof(double) && gwave >= b.f64_plane_waves) return;
    const WaveLds<T> L = carve<T, kCols>(lds_raw + kPerWave * wave, b, gwave);
    const uint32_t n_items = ws.n_items_dev ? *ws.n_items_dev : ws.n_items;
    if (ws.head) {
        // A wave's first item is the one of its own number; the next ones come from the queue head.  So
        // surplus waves of a rescue pass leave without touching the head (one address for the whole GPU,
        // about 14 ns an atomic: 60 us for a launch's 4,096 waves, whatever the rescued pairs).
        const uint32_t waves = std::min<uint32_t>(
            gridDim.x * waves_per_block, sizeof(T) == sizeof(double) ? b.f64_plane_waves : 0xFFFFFFFFu);
        for (uint32_t it = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(gwave)); it < n_items;) {
            process_pair<T, kCols>(b, tab, rs, L, lane, ws.items ? ws.items[it] : it);
            if (n_items <= waves) break;
            // All lanes issue the atomic (lane 0 adds 1, the rest add 0), so the fetch has no
            // lane-divergent branch; lane 0's pre-increment value is the wave's next item.
            it = waves + __builtin_amdgcn_readfirstlane(atomicAdd(ws.head, lane == 0 ? 1u : 0u));
        }
    } else {
        // The wave's index is wave-uniform; readfirstlane tells the compiler so, which keeps the
        // pair, its lengths and every loop over them scalar (uniform branches, no exec masking).
        const uint32_t stride = gridDim.x * waves_per_block;
        for (uint32_t it = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(gwave)); it < n_items; it += stride)
            process_pair<T, kCols>(b, tab, rs, L, lane, ws.items ? ws.items[it] : it);
    }
}

// ---- packed stripes (FP32) --------------------------------------------------------------------
//
// The aligned schedule above gives every pair whole 64-row stripes, so a read of R rows pays for
// 64 ceil(R/64) rows.  Packed stripes stream the rows of successive pairs through a wave's lanes
// instead: a stripe holds the end of one pair and the start of the next.  Each pair contributes
// R + 3 rows to the stream, in order
//   CONST  a row whose S = I + D is 1 in every column (M = I = 0, D' = 1 from the stripe start);
//   ZERO   the pair's row 0: M is d0 = 2^120/H in column -1 only (its prior is d0 on the marker
//          byte staged at column -1, 0 elsewhere, times the CONST row's S = 1), so its D, the running
//          sum of M (DD = MD = 1), is d0 from column 0 on: D(0, c) = 2^120/H as LoglessPairHMM.java:
//          30-36 sets it;
//   READ   rows 1..R, with the read's own transitions, except that row 1 takes MM = MI = 0 (its
//          row above has M = I = 0 in the model, so the terms vanish; here they hold the spike) and
//          row R takes MD = 0 (D(R, .) adds nothing to the result, and S(R, .) = I(R, .) then feeds
//          the summing row);
//   SUM    M(c) = (M + I)(R, c - 1) on columns 2..H+1 (prior 1 on real haplotype bytes read one
//          column to the left, 0 on padding), I = 0, and D' with DD = 1 is the running sum of M: at
//          column H + 2 it holds sum_c (M + I)(R, c) and stays there (M = 0 on padding).  The sum is
//          FP32 in column order, whatever stripe position and neighbours the pair gets, so results
//          are identical from run to run; its relative error is at most (H - 1) 2^-24 and in
//          practice a few ulps, since a last row's terms fall off fast away from the alignment.
// Every value stays a sub-probability times 2^120, so no product of a zeroed transition with a
// neighbour's value can be inf or NaN.  Rows need no other case: the step loop is the aligned
// schedule's, with per-lane haplotype pointers and transitions.  A stripe holds rows of at most two
// pairs (lanes past the second pair's rows idle), whose haplotypes sit in two LDS buffers; it runs
// max(H) + 66 steps, so the SUM row reaches column H + 2 and lane 63 writes every column lane 0 of
// the next stripe needs.  Haplotype bytes 0 (padding) and 1 (the row-0 marker) are reserved; the
// host uses the aligned schedule for batches whose haplotypes contain them.  Waves take the queue in
// fixed chunks (see packed_fetch).

constexpr uint32_t kPadByte = 0;      // haplotype bytes outside 1..H
constexpr uint32_t kZeroRowMark = 1;  // staged at column -1
constexpr uint32_t kNoByte = 0x1FF;   // compares equal to no byte

enum RowKind : int { kRowIdle = 0, kRowConst = 1, kRowZero = 2, kRowRead = 3, kRowSum = 4 };

// A pair in flight on a wave (wave-uniform).
struct PackedPair {
    uint32_t pair;
    int R, H;
    int64_t ro;  // read offset
    int hap_n;   // the haplotype has an 'N'
};

// LDS of a packed wave: a guard (the SUM row's prior reads one byte left of buffer 0 at lane 63's
// first step), two haplotype buffers, the two boundary planes.
constexpr int kHapGuard = 16;

template <int kCols>
constexpr size_t packed_lds_per_wave() {
    return kHapGuard + 2 * static_cast<size_t>(kCols) +
           kPlanes * static_cast<size_t>(plane_stride<kCols>()) * sizeof(float);
}

// A wave takes the queue in chunks of ws.chunk consecutive items, each chunk by one atomic on the
// queue head, and streams a chunk's pairs through its stripes in queue order.  A chunk always
// starts at lane 0 of a fresh stripe and no chunk shares a stripe with another, because a pair's
// bits depend on where its rows fall in the stripes (a row fed through the side pass rounds
// differently from one fed by DPP): chunks are fixed by the queue and the launch, so every run gives
// the same results while the waves still balance their load dynamically.  The launch sets the chunk
// (packed_chunk): at most kPackedChunk items, and few enough that every wave of the grid gets about
// four chunks, so a small queue (one region's pairs) still spreads over the whole GPU.
struct ChunkCursor {
    uint32_t next = 0, end = 0;  // items [next, end) of the wave's current chunk
    uint32_t wave = 0, waves = 0;  // this wave's number in the launch, and their count
    bool first = true;             // the wave's first chunk is the one of its own number
};

// Takes the next pair of the wave's current chunk; with new_chunk, first takes a new chunk when the
// current one is used up.  A pair with an empty read has L = 0 (log10 L = -inf): it is written at
// once and, as in the aligned schedule, listed for the FP64 pass.
__device__ bool packed_fetch(const DeviceBatch &b, const WorkSource &ws, uint32_t n_items, const RescueSink &rs,
                             int lane, PackedPair &p, ChunkCursor &cc, bool new_chunk) {
    for (;;) {
        if (cc.next >= cc.end) {
            if (!new_chunk) return false;
            // All lanes issue the atomic (lane 0 adds 1): the fetch has no lane-divergent branch.  A wave's
            // first chunk needs none: thousands of waves starting on one address take about 14 ns each.
            const uint32_t c = cc.first
                                   ? cc.wave
                                   : cc.waves + __builtin_amdgcn_readfirstlane(atomicAdd(ws.head, lane == 0 ? 1u : 0u));
            cc.first = false;
            const uint64_t first = static_cast<uint64_t>(c) * ws.chunk;
            if (first >= n_items) return false;
            cc.next = static_cast<uint32_t>(first);
            cc.end = static_cast<uint32_t>(first + ws.chunk < n_items ? first + ws.chunk : n_items);
        }
        const uint32_t it = cc.next++;
        const uint32_t pair = __builtin_amdgcn_readfirstlane(ws.items ? ws.items[it] : it);
        int r, h;
        if (b.pair_read) {
            r = b.pair_read[pair];
            h = b.pair_hap[pair];
        } else {
            r = static_cast<int>(pair / static_cast<uint32_t>(b.n_haps));
            h = static_cast<int>(pair % static_cast<uint32_t>(b.n_haps));
        }
        p.pair = pair;
        p.R = __builtin_amdgcn_readfirstlane(b.rd_len[r]);
        p.H = __builtin_amdgcn_readfirstlane(b.hap_len[h]);
        const int64_t ro = b.rd_off[r];
        p.ro = (static_cast<int64_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(ro >> 32))) << 32) |
               static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(ro)));
        p.hap_n = 0;
        if (p.R > 0) return true;
        b.out[pair] = -__builtin_inf();
        if (rs.list != nullptr) {
            const uint32_t slot = __builtin_amdgcn_readfirstlane(atomicAdd(rs.count, lane == 0 ? 1u : 0u));
            rs.list[slot] = pair;
        }
    }
}

// Stages pair p's haplotype in LDS buffer `hb`: byte of column c at kLdsPad + c - 1, the row-0 marker
// at column -1, padding everywhere else (the SUM row's prior needs padding up to the stripe's end).
template <int kCols>
__device__ void packed_stage(const DeviceBatch &b, uint8_t *hbuf, int lane, PackedPair &p) {
    // An explicit LDS pointer: through a generic one these become FLAT stores, which count on both
    // wait counters out of order and turn every LDS wait of the step loop into lgkmcnt(0).
    using lds_u8w = __attribute__((address_space(3))) uint8_t;
    lds_u8w *hb = (lds_u8w *)hbuf;  // address-space cast: C-style only
    const int h = b.pair_read ? b.pair_hap[p.pair] : static_cast<int>(p.pair % static_cast<uint32_t>(b.n_haps));
    const uint8_t *hap = b.hap_bases + b.hap_off[h];
    int has_n = 0;
    for (int j = lane; j < kCols; j += kWave) {
        const int c = j - kLdsPad + 1;
        uint8_t v = kPadByte;
        if (c >= 1 && c <= p.H) {
            v = hap[c - 1];
            has_n |= (v == 'N');
        } else if (c == -1) {
            v = kZeroRowMark;
        }
        hb[j] = v;
    }
    p.hap_n = __any(has_n) ? 1 : 0;
}

// Transitions, priors and starting state of one lane's row.
struct PackedRow {
    RowTrans<float> w;
    uint32_t nval;           // second byte the prior treats as a match ('N' for read rows)
    int shift;               // haplotype column offset of the lane's prior (-1 for SUM)
    float m1, s1, d1, s2;    // state left of the lane's first column (columns -k-1 and -k-2)
    int kind;
};

__device__ __forceinline__ PackedRow packed_row(int kind, int idx, const PackedPair &p, const DeviceBatch &b,
                                                const DeviceTables &tab, int lane) {
    PackedRow x;
    x.w = RowTrans<float>{0, 0, 0, 0, 0, 0, 0, 0, kNoByte};
    x.nval = kNoByte;
    x.shift = 0;
    x.m1 = x.s1 = x.d1 = x.s2 = 0.f;
    x.kind = kind;
    if (kind == kRowRead) {
        const int r = idx - 1;  // 1-based read row
        const int64_t ro = p.ro;
        x.w = row_trans<float>(r - 1, p.R, b.rd_bases + ro, b.rd_quals + ro, b.rd_ins + ro, b.rd_del + ro,
                               b.rd_gcp + ro, tab);
        if (r == 1) {
            x.w.MM = 0.f;
            x.w.MI = 0.f;
        }
        if (r == p.R) x.w.MD = 0.f;
        x.nval = 'N';
    } else if (kind == kRowConst) {
        x.w.MD = 1.f;
        x.w.DD = 1.f;
        x.d1 = 1.f;
        x.s1 = 1.f;
        x.s2 = 1.f;
    } else if (kind == kRowZero) {
        const float d0 = static_cast<float>(__builtin_ldexp(1.0, Scale<float>::kExp) / static_cast<double>(p.H));
        x.w.GM = 1.f;
        x.w.MD = 1.f;
        x.w.DD = 1.f;
        x.w.pm = d0;
        x.w.base = kZeroRowMark;
        if (lane == 0) x.m1 = d0;  // column -1 lies left of lane 0's first column
    } else if (kind == kRowSum) {
        x.w.MM = 1.f;
        x.w.GM = 1.f;
        x.w.DD = 1.f;
        x.w.px = 1.f;
        x.w.base = kPadByte;
        x.shift = -1;
    }
    return x;
}

// A lane's cell one step back (1) and two steps back (2); d1 is D' = D / MD.
struct PackedState {
    float m1, i1, d1, s1, m2, s2;
};

__device__ __forceinline__ PackedState packed_start(const PackedRow &x) {
    return PackedState{x.m1, 0.f, x.d1, x.s1, 0.f, x.s2};
}

// kU steps (the aligned schedule's step, per-lane haplotype bytes and 'N' bytes): lane 0's sums in av, bv,
// the lanes' haplotype bytes in hbs, M and I to wm, wi.  kNop: wait states before the DPP products.
template <bool kHapHasN, int kU, int kNop>
__device__ __forceinline__ void packed_block(PackedState &st, const RowTrans<float> &w, uint32_t nval,
                                             const float (&av)[kU], const float (&bv)[kU], const uint32_t (&hbs)[kU],
                                             __attribute__((address_space(3))) float *wm,
                                             __attribute__((address_space(3))) float *wi) {
#pragma unroll
    for (int u = 0; u < kU; ++u) {
        const uint32_t hb = hbs[u];
        const bool match = (hb == w.base) || (kHapHasN && hb == nval);
        const float prior = match ? w.pm : w.px;
        float a = av[u], i = bv[u];
        dpp_upper2<kNop>(a, st.m2, w.MM, st.s2, w.GM, i, st.m1, w.MI, st.i1, w.II);
        const float m = a * prior;
        const float d = fmaf(st.d1, w.DD, st.m1);
        const float sx = fmaf(w.MD, d, i);
        wm[u] = m;
        wi[u] = i;
        if (u % 2 == 1) store_order();
        st.m2 = st.m1;
        st.s2 = st.s1;
        st.m1 = m;
        st.i1 = i;
        st.d1 = d;
        st.s1 = sx;
    }
}

// A lane's haplotype bytes in LDS, four columns a word: aligned words, shifted to the lane's own byte.  Byte
// loads, one a step, were a third of a packed launch's LDS instructions (0.23 a VALU instruction, 0.15 with
// words), and VALU and LDS each waited for the other: 300 regions 39.7 ms with them, 36.7 ms with words; 128,000
// pairs of one region 6.40 ms, 5.87 ms; 5,265 pairs on the split kernel, whole call 293 us, 280 us.
struct HapWords {
    using lds_u32 = const __attribute__((address_space(3))) uint32_t;
    uint32_t at, word;
    lds_u32 *next;

    __device__ __forceinline__ explicit HapWords(const uint8_t *first) {  // the byte of step 0
        using lds_u8 = const __attribute__((address_space(3))) uint8_t;
        at = (uint32_t)(uintptr_t)(lds_u8 *)first;  // address-space cast: C-style only
        lds_u32 *w = (lds_u32 *)(uintptr_t)(at & ~3u);
        word = w[0];
        next = w + 1;
    }
    // The bytes of the kU steps from t0, of successive blocks.
    template <int kU>
    __device__ __forceinline__ void block(int t0, uint32_t (&hbs)[kU]) {
#pragma unroll
        for (int q = 0; q < kU / 4; ++q) {
            const uint32_t w = next[t0 / 4 + q];
            const uint32_t four = __builtin_amdgcn_alignbyte(w, word, at);
            word = w;
#pragma unroll
            for (int u = 0; u < 4; ++u) hbs[4 * q + u] = (four >> (8 * u)) & 0xFFu;
        }
    }
};

// One stripe of steps.  Returns the lane's D' after the last step (a SUM row's last-row sum).
template <int kCols, bool kHapHasN, int kU>
__device__ __forceinline__ float packed_steps(const WaveLds<float> &L, const uint8_t *hap, int lane,
                                              const PackedRow &x, int steps) {
    PackedState st = packed_start(x);
    HapWords bytes(hap + kLdsPad - 1 - lane + x.shift);
    // Every lane stores its M and I at its own column c = t - lane at step t, so the step has no
    // one-lane exec mask (no exec writes, no branch).  Lane 63 writes column c last, at step c + 63,
    // so the planes end with its row; lane 0 has read A and B of column c by step c, before any lane
    // overwrites it.
    using lds_f32 = __attribute__((address_space(3))) float;
    int lane_w = lane;
    asm volatile("" : "+v"(lane_w));
    lds_f32 *wm = (lds_f32 *)(L.bm + kLdsPad) - lane_w, *wi = (lds_f32 *)(L.bi + kLdsPad) - lane_w;
    // No scalar load may be in flight at the loop head: they complete out of order, and one pending
    // there makes every LDS wait in the loop a full lgkmcnt(0) instead of waiting for the first reads.
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    for (int t0 = 0; t0 < steps; t0 += kU) {
        float av[kU], bv[kU];
        __builtin_memcpy(av, __builtin_assume_aligned(L.bm + kLdsPad + t0, 16), sizeof(av));
        __builtin_memcpy(bv, __builtin_assume_aligned(L.bi + kLdsPad + t0, 16), sizeof(bv));
        uint32_t hbs[kU];
        bytes.block(t0, hbs);
        __builtin_amdgcn_wave_barrier();
        packed_block<kHapHasN, kU, 4>(st, x.w, x.nval, av, bv, hbs, wm + t0, wi + t0);
    }
    __builtin_amdgcn_wave_barrier();
    return st.d1;
}

// The packed-stripe FP32 pass of one wave over its share of a queue, kU wave-steps per unrolled
// loop body.
template <int kCols, int kU>
__device__ void packed_wave(const DeviceBatch &b, const DeviceTables &tab, const WorkSource &ws, uint32_t n_items,
                            const RescueSink &rs, uint8_t *lds, int lane, uint32_t gwave, uint32_t waves) {
    ChunkCursor cc;
    cc.wave = gwave;
    cc.waves = waves;
    WaveLds<float> L;
    // Haplotype buffer k at lds + kHapGuard + k kCols (chosen by arithmetic, not by indexing an array
    // of pointers, so the compiler keeps them LDS pointers).
    auto hapbuf = [&](int k) { return lds + kHapGuard + (k ? kCols : 0); };
    L.hap = hapbuf(0);
    L.bm = reinterpret_cast<float *>(lds + kHapGuard + 2 * kCols);
    L.bi = L.bm + plane_stride<kCols>();
    for (int j = lane; j < plane_stride<kCols>(); j += kWave) {
        L.bm[j] = 0.f;
        L.bi[j] = 0.f;
    }
    const double scale_log10 = static_cast<double>(Scale<float>::kExp) * 0.30102999566398119521;
    PackedPair cur{}, nxt{};
    bool have_cur = false;
    int cur_next = 0;  // next row of cur: 0 CONST, 1 ZERO, 2..R+1 READ, R+2 SUM
    int buf_cur = 0;
    bool first = true;
    float md63 = 0.f, dd63 = 0.f, cd63 = 0.f;  // lane 63's row of the previous stripe (side pass)
    int wend = 0;                              // plane slots [1, wend) lane 63 wrote in that stripe
    for (;;) {
        if (!have_cur) {
            if (!packed_fetch(b, ws, n_items, rs, lane, cur, cc, true)) break;
            have_cur = true;
            cur_next = 0;
            buf_cur = 0;
            packed_stage<kCols>(b, hapbuf(buf_cur), lane, cur);
        }
        const int rows_cur = cur.R + 3 - cur_next;
        bool two = false;
        if (rows_cur < kWave) {
            if (packed_fetch(b, ws, n_items, rs, lane, nxt, cc, false)) {
                two = true;
                packed_stage<kCols>(b, hapbuf(buf_cur ^ 1), lane, nxt);
            }
        }
        // This lane's row.
        const bool in_cur = lane < rows_cur;
        const int idx = in_cur ? cur_next + lane : lane - rows_cur;
        const PackedPair &pp = in_cur ? cur : nxt;
        int kind = kRowIdle;
        if (in_cur || (two && idx < nxt.R + 3)) {
            const int R = in_cur ? cur.R : nxt.R;
            kind = idx == 0 ? kRowConst : idx == 1 ? kRowZero : idx == R + 2 ? kRowSum : kRowRead;
        }
        const PackedRow x = packed_row(kind, idx, pp, b, tab, lane);
        const uint8_t *hap = hapbuf(in_cur ? buf_cur : buf_cur ^ 1);
        const int hmax = two && nxt.H > cur.H ? nxt.H : cur.H;
        // Wave-uniform by construction; readfirstlane makes it a scalar, so the step loop stays a
        // uniform loop (a vector trip count turns it into a divergent loop with exec masking).
        const int steps = __builtin_amdgcn_readfirstlane(round_up(hmax + kWave + 2, kU));
        if (!first)
            side_pass_f32<kCols>(L.bm, L.bi, lane, rfl(x.w.MM), rfl(x.w.GM), rfl(x.w.MI), rfl(x.w.II), md63, dd63,
                                 plane_span<kCols>(steps), cd63, wend);
        first = false;
        wend = kLdsPad - (kWave - 1) + steps;
        md63 = lane63(x.w.MD);
        dd63 = lane63(x.w.DD);
        cd63 = lane63(x.kind == kRowConst ? 1.f : 0.f);
        const float dfin = (cur.hap_n || (two && nxt.hap_n)) ? packed_steps<kCols, true, kU>(L, hap, lane, x, steps)
                                                            : packed_steps<kCols, false, kU>(L, hap, lane, x, steps);
        // SUM rows that ended here: every lane takes the SUM lane's total, so the result and the
        // rescue decision are wave-uniform.  Unscaling and log10 are FP64.
        const double total = static_cast<double>(dfin);
        const bool cur_done = rows_cur <= kWave;
        const bool nxt_done = two && nxt.R + 3 <= kWave - rows_cur;
        for (int q = 0; q < 2; ++q) {
            if (q == 0 ? !cur_done : !nxt_done) continue;
            const int sl = q == 0 ? rows_cur - 1 : rows_cur + nxt.R + 2;
            const uint64_t tb = __builtin_bit_cast(uint64_t, total);
            const uint32_t lo = __builtin_amdgcn_readlane(static_cast<int>(tb), sl);
            const uint32_t hi = __builtin_amdgcn_readlane(static_cast<int>(tb >> 32), sl);
            const double sum = __builtin_bit_cast(double, (static_cast<uint64_t>(hi) << 32) | lo);
            const uint32_t pair = q == 0 ? cur.pair : nxt.pair;
            b.out[pair] = log10(sum) - scale_log10;
            if (rs.list != nullptr && !(sum >= rs.threshold)) {
                const uint32_t slot = __builtin_amdgcn_readfirstlane(atomicAdd(rs.count, lane == 0 ? 1u : 0u));
                rs.list[slot] = pair;
            }
        }
        if (!cur_done) {
            cur_next += kWave;
        } else if (two && !nxt_done) {
            cur = nxt;
            cur_next = kWave - rows_cur;
            buf_cur ^= 1;
        } else {
            have_cur = false;
        }
    }
}

template <int kCols, int kU>
__global__ __launch_bounds__(512) void forward_kernel_packed(DeviceBatch b, DeviceTables tab, WorkSource ws,
                                                             RescueSink rs) {
    extern __shared__ __align__(16) uint8_t lds_raw[];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    const uint32_t n_items = ws.n_items_dev ? *ws.n_items_dev : ws.n_items;
    const uint32_t waves_per_block = blockDim.x / kWave;
    packed_wave<kCols, kU>(b, tab, ws, n_items, rs, lds_raw + packed_lds_per_wave<kCols>() * wave, lane,
                           __builtin_amdgcn_readfirstlane(blockIdx.x * waves_per_block + wave),
                           gridDim.x * waves_per_block);
}

// ---- split stripes (FP32) ---------------------------------------------------------------------
//
// A small queue (one region's pairs) gives a packed wave one pair (ws.chunk = 1), whose stripes it then
// computes one after another: the launch lasts as long as the longest pair's stripes in a row on a SIMD
// that got five of them, and with fewer pairs than SIMDs most of the GPU waits for single waves.  Here
// a workgroup of four waves works through pairs together, the unit of work being a stripe: the stripes of
// the group's pairs, in order, go to its waves in turn.  The wave of stripe s + 1 follows the wave of
// stripe s at the distance at which lane 63 has finished a 64-column chunk, runs the side pass over that
// chunk and then 64 steps.  Stripes, rows and the operations on every cell are those of a packed wave
// with a chunk of one pair, so results are the same bit for bit.
//
// The stripes of a pair share one pair of LDS planes: along the columns, from right to left, lie the
// columns stripe s is writing, its finished row, the same row as stripe s + 1's sums A and B, the columns
// stripe s + 1 is writing, and so on; no stripe passes the one before it.  A group holds kSlots pairs.
// Every wait is for work that does not depend on the waiting wave, by waves of the same workgroup, which
// are resident together: a stripe for the stripe before it, a reader of a pair's record for the wave that
// takes its first stripe, and that wave, to reuse a slot, for all waves to have gone past the slot's pair
// (so its stripes are done and its record is read).  A wave's LDS operations complete in the order they
// are issued, so a word published after its data needs no further wait.
//
// Bound by the latency of a pair's stripes in small queues (about 100 cycles a step for a lone wave: LDS
// round trips, dependent products) and by VALU issue in large ones.  8 steps per block (81 VGPRs, 20 waves
// per CU) against 16 (105, 16 waves): 288 and 303 us at 5,265 pairs, equal at 1,024.
constexpr int kSplitWaves = 4;
constexpr uint32_t kSplitEnd = 0xFFFFFFFFu;  // n_stripes of the record that ends the queue

using lds_u32 = volatile __attribute__((address_space(3))) uint32_t;

// A pair's record, after its haplotype and planes.
struct SplitRecord {
    uint32_t seq;  // pair number + 1 once the record is valid
    uint32_t n_stripes, pair, R, H, ro_lo, ro_hi, hap_n;
    uint32_t done[kSplitWaves];  // split_progress of the latest stripe s with s mod 4 = k
};

template <int kCols>
constexpr size_t split_slot_bytes() {
    return kHapGuard + static_cast<size_t>(kCols) + kPlanes * static_cast<size_t>(plane_stride<kCols>()) * sizeof(float) +
           sizeof(SplitRecord);
}
// Slots per group: four, or two where the longer haplotypes' planes would leave a CU less than its share
// of groups.
template <int kCols>
constexpr int split_slots() { return kCols <= 1024 ? 4 : 2; }
template <int kCols>
constexpr size_t split_lds_bytes() { return split_slots<kCols>() * split_slot_bytes<kCols>() + kSplitWaves * sizeof(uint32_t); }

__device__ __forceinline__ uint32_t lds_get(lds_u32 *p) {
    return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(*p)));
}

// Stages a haplotype as packed_stage does, one wave, four bases a load.  Returns whether it has an 'N'.
template <int kCols>
__device__ __forceinline__ bool split_stage(const uint8_t *hap, int H, uint8_t *hbuf, int lane) {
    using lds_w32 = __attribute__((address_space(3))) uint32_t;
    using lds_w8 = __attribute__((address_space(3))) uint8_t;
    lds_w32 *w = (lds_w32 *)hbuf;  // address-space casts: C-style only
    for (int k = lane; k < kCols / 4; k += kWave) w[k] = 0u;
    __builtin_amdgcn_wave_barrier();
    int has_n = 0;
    for (int c = 4 * lane; c < H; c += 4 * kWave) {
        if (c + 4 <= H) {
            uint32_t v;
            __builtin_memcpy(&v, hap + c, 4);
            w[kLdsPad / 4 + c / 4] = v;
#pragma unroll
            for (int k = 0; k < 4; ++k) has_n |= ((v >> (8 * k)) & 0xFFu) == 'N';
        } else {
            for (int k = c; k < H; ++k) {
                ((lds_w8 *)hbuf)[kLdsPad + k] = hap[k];
                has_n |= hap[k] == 'N';
            }
        }
    }
    if (lane == 0) ((lds_w8 *)hbuf)[kLdsPad - 2] = kZeroRowMark;  // column -1
    return __any(has_n);
}

// One stripe on one wave.  Returns the lane's D' after the last step.
template <int kCols, bool kHapHasN, int kU>
__device__ __forceinline__ float split_stripe(const DeviceBatch &b, const DeviceTables &tab, const PackedPair &p,
                                              const WaveLds<float> &L, lds_u32 *done, int lane, int s) {
    const int idx = s * kWave + lane;
    const int kind = idx == 0 ? kRowConst : idx == 1 ? kRowZero : idx == p.R + 2 ? kRowSum : idx < p.R + 2 ? kRowRead : kRowIdle;
    const PackedRow x = packed_row(kind, idx, p, b, tab, lane);
    // Lane 63's row of the stripe before (a read row), wave-uniform.
    const PackedRow up = packed_row(s > 0 ? kRowRead : kRowIdle, s * kWave - 1, p, b, tab, lane);
    SidePass side(lane, rfl(x.w.MM), rfl(x.w.GM), rfl(x.w.MI), rfl(x.w.II), up.w.MD, up.w.DD, 0.f);
    const int steps = __builtin_amdgcn_readfirstlane(round_up(p.H + kWave + 2, kU));
    const int wend = kLdsPad - (kWave - 1) + steps;
    const int jmax = plane_span<kCols>(steps);
    PackedState st = packed_start(x);
    HapWords bytes(L.hap + kLdsPad - 1 - lane + x.shift);
    using lds_f32 = __attribute__((address_space(3))) float;
    int lane_w = lane;
    asm volatile("" : "+v"(lane_w));
    lds_f32 *wm = (lds_f32 *)(L.bm + kLdsPad) - lane_w, *wi = (lds_f32 *)(L.bi + kLdsPad) - lane_w;
    auto follow = [&](int need) {  // until the stripe before has done `need` steps
        const uint32_t want = split_progress(static_cast<uint32_t>(s - 1), static_cast<uint32_t>(need < steps ? need : steps));
        while (!split_reached(lds_get(done + (s - 1) % kSplitWaves), want)) __builtin_amdgcn_s_sleep(1);
        asm volatile("" ::: "memory");
    };
    if (s > 0) {
        follow(kWave);
        side.chunk(L.bm, L.bi, lane, 0, wend);
    }
    for (int t1 = 0; t1 < steps; t1 += kWave) {
        if (s > 0 && t1 + kWave < jmax) {
            follow(t1 + 2 * kWave - 1);
            side.chunk(L.bm, L.bi, lane, t1 + kWave, wend);
        }
        const int end = t1 + kWave < steps ? t1 + kWave : steps;
        for (int t0 = t1; t0 < end; t0 += kU) {
            float av[kU], bv[kU];
            if (s > 0) {
                __builtin_memcpy(av, __builtin_assume_aligned(L.bm + kLdsPad + t0, 16), sizeof(av));
                __builtin_memcpy(bv, __builtin_assume_aligned(L.bi + kLdsPad + t0, 16), sizeof(bv));
            } else {  // above the CONST row
#pragma unroll
                for (int u = 0; u < kU; ++u) av[u] = bv[u] = 0.f;
            }
            uint32_t hbs[kU];
            bytes.block(t0, hbs);
            __builtin_amdgcn_wave_barrier();
            packed_block<kHapHasN, kU, 1>(st, x.w, x.nval, av, bv, hbs, wm + t0, wi + t0);
            asm volatile("" ::: "memory");  // a wave's LDS operations complete in the order they are issued
            done[s % kSplitWaves] = split_progress(static_cast<uint32_t>(s), static_cast<uint32_t>(t0 + kU));
        }
    }
    return st.d1;
}

template <int kCols, int kU>
__global__ __launch_bounds__(kSplitWaves * kWave) void forward_kernel_split(DeviceBatch b, DeviceTables tab, WorkSource ws,
                                                                            RescueSink rs) {
    extern __shared__ __align__(16) uint8_t lds_raw[];
    constexpr int kSlots = split_slots<kCols>();
    constexpr size_t kSlotBytes = split_slot_bytes<kCols>();
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    lds_u32 *const view = (lds_u32 *)(lds_raw + kSlots * kSlotBytes);  // the pair each wave has come to
    auto record = [&](int slot) {
        return (volatile __attribute__((address_space(3))) SplitRecord *)(lds_raw + (slot + 1) * kSlotBytes -
                                                                         sizeof(SplitRecord));
    };
    const double scale_log10 = static_cast<double>(Scale<float>::kExp) * 0.30102999566398119521;
    if (wave == 0) {
        for (int k = 0; k < kSlots; ++k) record(k)->seq = 0u;
        for (int k = 0; k < kSplitWaves; ++k) view[k] = 0u;
    }
    __syncthreads();
    uint32_t j = 0, first = 0;  // pair number and the task number of its first stripe
    for (uint32_t task = wave;; task += kSplitWaves) {
        uint8_t *base;
        volatile __attribute__((address_space(3))) SplitRecord *rec;
        uint32_t n_stripes;
        // The pair of this task, walking on from the wave's last one.
        for (;;) {
            const int slot = static_cast<int>(j % kSlots);
            base = lds_raw + slot * kSlotBytes;
            rec = record(slot);
            if (task == first) {
                // This wave takes the pair's first stripe: it fetches the pair and fills the slot.
                for (int k = 0; k < kSplitWaves; ++k)
                    while (lds_get(view + k) + kSlots <= j) __builtin_amdgcn_s_sleep(1);
                // The group's first pair is the one of its own number; the next ones come from the queue head.
                uint32_t it = blockIdx.x;
                if (j > 0)
                    it = ws.n_items <= gridDim.x
                             ? ws.n_items
                             : gridDim.x + static_cast<uint32_t>(
                                               __builtin_amdgcn_readfirstlane(atomicAdd(ws.head, lane == 0 ? 1u : 0u)));
                if (it < ws.n_items) {
                    const uint32_t pair = __builtin_amdgcn_readfirstlane(ws.items ? ws.items[it] : it);
                    int r, h;
                    if (b.pair_read) {
                        r = b.pair_read[pair];
                        h = b.pair_hap[pair];
                    } else {
                        r = static_cast<int>(pair / static_cast<uint32_t>(b.n_haps));
                        h = static_cast<int>(pair % static_cast<uint32_t>(b.n_haps));
                    }
                    const int R = b.rd_len[r], H = b.hap_len[h];
                    const int64_t ro = b.rd_off[r];
                    const bool hap_n = split_stage<kCols>(b.hap_bases + b.hap_off[h], H, base + kHapGuard, lane);
                    rec->n_stripes = R > 0 ? static_cast<uint32_t>((R + 3 + kWave - 1) / kWave) : 0u;
                    rec->pair = pair;
                    rec->R = static_cast<uint32_t>(R);
                    rec->H = static_cast<uint32_t>(H);
                    rec->ro_lo = static_cast<uint32_t>(ro);
                    rec->ro_hi = static_cast<uint32_t>(ro >> 32);
                    rec->hap_n = hap_n ? 1u : 0u;
                    for (int k = 0; k < kSplitWaves; ++k) rec->done[k] = 0u;
                    if (R <= 0) {  // an empty read: L = 0, listed for the FP64 pass
                        b.out[pair] = -__builtin_inf();
                        if (rs.list != nullptr)
                            rs.list[__builtin_amdgcn_readfirstlane(atomicAdd(rs.count, lane == 0 ? 1u : 0u))] = pair;
                    }
                } else {
                    rec->n_stripes = kSplitEnd;
                }
                asm volatile("" ::: "memory");
                rec->seq = j + 1;
            } else {
                while (lds_get(&rec->seq) != j + 1) __builtin_amdgcn_s_sleep(1);
            }
            asm volatile("" ::: "memory");
            n_stripes = lds_get(&rec->n_stripes);
            if (n_stripes == kSplitEnd || task - first < n_stripes) break;
            first += n_stripes;
            ++j;
            view[wave] = j;
        }
        if (n_stripes == kSplitEnd) break;
        PackedPair p{};
        p.pair = lds_get(&rec->pair);
        p.R = static_cast<int>(lds_get(&rec->R));
        p.H = static_cast<int>(lds_get(&rec->H));
        p.ro = static_cast<int64_t>((static_cast<uint64_t>(lds_get(&rec->ro_hi)) << 32) | lds_get(&rec->ro_lo));
        WaveLds<float> L;
        L.hap = base + kHapGuard;
        L.bm = reinterpret_cast<float *>(base + kHapGuard + kCols);
        L.bi = L.bm + plane_stride<kCols>();
        const int s = static_cast<int>(task - first);
        lds_u32 *const done = (lds_u32 *)rec->done;
        const float dfin = lds_get(&rec->hap_n) ? split_stripe<kCols, true, kU>(b, tab, p, L, done, lane, s)
                                                : split_stripe<kCols, false, kU>(b, tab, p, L, done, lane, s);
        if (s == static_cast<int>(n_stripes) - 1) {
            // The SUM lane's total to every lane; unscaling and log10 are FP64.
            const float f = __builtin_bit_cast(
                float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, dfin), (p.R + 2) & (kWave - 1)));
            const double sum = static_cast<double>(f);
            b.out[p.pair] = log10(sum) - scale_log10;
            if (rs.list != nullptr && !(sum >= rs.threshold))
                rs.list[__builtin_amdgcn_readfirstlane(atomicAdd(rs.count, lane == 0 ? 1u : 0u))] = p.pair;
        }
    }
}

__global__ void zero_counters_kernel(uint32_t *c, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) c[i] = 0u;
}

__global__ void copy_counters_kernel(uint32_t *c, const uint32_t *init, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) c[i] = init[i];
}

}  // namespace

int lds_columns(int max_hap_len) {
    const int need = max_hap_len + 2 * kLdsPad + 32;
    for (int c : kColClasses)
        if (c >= need) return c;
    return 0;
}

int lds_class_index(int hap_len) {
    const int need = hap_len + 2 * kLdsPad + 32;
    for (int k = 0; k < kNumColClasses; ++k)
        if (kColClasses[k] >= need) return k;
    return -1;
}

size_t lds_bytes_per_wave(int max_hap_len, bool fp64, bool packed) {
    const size_t cols = static_cast<size_t>(lds_columns(max_hap_len));
    if (cols == 0) return 0;
    if (packed && !fp64)
        return kHapGuard + 2 * cols + kPlanes * sizeof(float) * static_cast<size_t>(lds_plane_stride(static_cast<int>(cols)));
    return cols + (fp64 ? kRing64Bytes : kPlanes * sizeof(float) * static_cast<size_t>(lds_plane_stride(static_cast<int>(cols))));
}

size_t fp64_plane_bytes_per_wave(int max_hap_len) {
    const int cols = lds_columns(max_hap_len);
    return cols == 0 ? 0 : kPlanes * sizeof(double) * static_cast<size_t>(lds_plane_stride(cols));
}

namespace {

template <typename F>
hipError_t with_kernel(bool fp64, bool packed, int cols, int unroll, F &&f) {
    return dispatch_col_class(cols, [&](auto C) -> hipError_t {
        constexpr int kC = decltype(C)::value;
        if (fp64) return f(forward_kernel<double, kC>);
        if constexpr (kC > kMaxFp32Cols) {
            return hipErrorInvalidValue;  // FP64-only class
        } else {
            if (!packed) return f(forward_kernel<float, kC>);
            return unroll == 16 ? f(forward_kernel_packed<kC, 16>) : f(forward_kernel_packed<kC, 8>);
        }
    });
}


}  // namespace

namespace {

// The split kernel, for launches of fewer than eight pairs for each wave of a resident grid (takes_split).
// Measured on one call, packed and split: 1,024 pairs 158 and 129 us, 5,265 pairs 311 and 288, 18,000 pairs
// 863 and 825, 38,400 pairs 1,189 and 1,196; 200 pairs of 250-600 rows on haplotypes of 1,500 862 and 322.
// Its groups have four waves and its loop body 8 steps; its grid is grid_percent of its own resident groups.
hipError_t launch_split(const DeviceBatch &batch, const DeviceTables &tables, const WorkSource &ws, const RescueSink &rescue,
                        int cols, int grid_percent, hipStream_t stream) {
    return dispatch_col_class(cols, [&](auto C) -> hipError_t {
        constexpr int kC = decltype(C)::value;
        if constexpr (kC > kMaxFp32Cols) {
            return hipErrorInvalidValue;
        } else {
            static_assert(split_lds_bytes<kC>() <= 163840, "a workgroup's LDS fits a CU");
            auto kernel = forward_kernel_split<kC, 8>;
            if (split_lds_bytes<kC>() > 65536)
                (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                          hipFuncAttributeMaxDynamicSharedMemorySize,
                                          static_cast<int>(split_lds_bytes<kC>()));
            static const int per_cu = [&] {
                int n = 0;
                const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, kSplitWaves * kWave,
                                                                                  split_lds_bytes<kC>());
                return e == hipSuccess && n > 0 ? n : 1;
            }();
            int dev = 0, cus = 0;
            if (hipGetDevice(&dev) != hipSuccess ||
                hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
                cus = 1;
            const int64_t groups = std::max<int64_t>(1, static_cast<int64_t>(per_cu) * cus * grid_percent / 100);
            const uint32_t grid = static_cast<uint32_t>(std::min<int64_t>(ws.n_items, groups));
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(kSplitWaves * kWave), split_lds_bytes<kC>(), stream, batch, tables,
                               ws, rescue);
            return hipGetLastError();
        }
    });
}

}  // namespace

hipError_t launch_forward(bool fp64, const DeviceBatch &batch, const DeviceTables &tables, const WorkSource &work,
                          const RescueSink &rescue, int max_hap_len, const LaunchShape &shape, int grid_blocks,
                          hipStream_t stream) {
    if (shape.waves_per_block < 1 || grid_blocks < 1) return hipErrorInvalidValue;
    // The packed schedule takes chunks from a queue with a host-known item count.
    if (shape.packed && (fp64 || work.head == nullptr || work.n_items_dev != nullptr)) return hipErrorInvalidValue;
    WorkSource ws = work;
    if (shape.packed) ws.chunk = packed_chunk(work.n_items, static_cast<int64_t>(grid_blocks) * shape.waves_per_block);
    if (takes_split(shape, work.n_items, grid_blocks))
        return launch_split(batch, tables, ws, rescue, lds_columns(max_hap_len), shape.grid_percent, stream);
    const dim3 block(kWave * shape.waves_per_block);
    return with_kernel(fp64, shape.packed, lds_columns(max_hap_len), shape.unroll, [&](auto kernel) {
        if (shape.lds_bytes > 65536)
            (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      static_cast<int>(shape.lds_bytes));
        hipLaunchKernelGGL(kernel, dim3(grid_blocks), block, shape.lds_bytes, stream, batch, tables, ws, rescue);
        return hipGetLastError();
    });
}

hipError_t launch_zero_counters(uint32_t *counters, int n, hipStream_t stream) {
    hipLaunchKernelGGL(zero_counters_kernel, dim3(1), dim3(64), 0, stream, counters, n);
    return hipGetLastError();
}

hipError_t launch_copy_counters(uint32_t *counters, const uint32_t *init, int n, hipStream_t stream) {
    hipLaunchKernelGGL(copy_counters_kernel, dim3(1), dim3(64), 0, stream, counters, init, n);
    return hipGetLastError();
}

size_t max_lds_per_block() {
    static const size_t limit = [] {
        int dev = 0, v = 0;
        size_t l = 65536;
        if (hipGetDevice(&dev) == hipSuccess &&
            hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && v > 0)
            l = static_cast<size_t>(v);
        return l < 163840 ? l : static_cast<size_t>(163840);
    }();
    return limit;
}

LaunchShape forward_shape(bool fp64, int max_hap_len, int requested_waves_per_block, bool packed, int unroll) {
    LaunchShape sh;
    const int cols = lds_columns(max_hap_len);
    if (cols == 0 || (!fp64 && cols > kMaxFp32Cols)) return sh;
    packed = packed && !fp64;
    const size_t per_wave = lds_bytes_per_wave(max_hap_len, fp64, packed);
    const size_t budget = max_lds_per_block();
    int wpb = requested_waves_per_block < 1 ? 1 : requested_waves_per_block;
    while (wpb > 1 && per_wave * static_cast<size_t>(wpb) > budget) --wpb;
    if (per_wave * static_cast<size_t>(wpb) > budget) return sh;
    sh.waves_per_block = wpb;
    sh.lds_bytes = per_wave * static_cast<size_t>(wpb);
    sh.packed = packed;
    sh.tuned = requested_waves_per_block != kWavesPerBlock || unroll != 0;
    auto occupancy = [&](int u) {
        int blocks = 0;
        const hipError_t e = with_kernel(fp64, packed, cols, u, [&](auto kernel) {
            return hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, kWave * wpb, sh.lds_bytes);
        });
        return (e == hipSuccess && blocks > 0) ? blocks : 1;
    };
    sh.unroll = packed && unroll == 16 ? 16 : 8;
    sh.blocks_per_cu = occupancy(sh.unroll);
    if (packed && unroll == 0) {
        // Automatic: the 16-step body issues fewer instructions per step but needs more VGPRs; it
        // wins where the LDS slice, not the registers, limits the waves per CU (long haplotypes).
        const int b16 = occupancy(16);
        if (b16 >= sh.blocks_per_cu) {
            sh.unroll = 16;
            sh.blocks_per_cu = b16;
        }
    }
    return sh;
}

}  // namespace gatk_pairhmm
