// readprep.hip -- HaplotypeCaller's read-quality preparation on the device, over packed read planes:
//   * the PCR indel error model: PairHMMLikelihoodCalculationEngine.applyPCRErrorModel
//     (tools/walkers/haplotypecaller/PairHMMLikelihoodCalculationEngine.java:360-371) caps the
//     insertion and deletion GOP at read positions 0 .. L-2 by a quality that falls with the tandem
//     repeat length there (ReadLikelihoodCalculationEngine.findTandemRepeatUnits,
//     ReadLikelihoodCalculationEngine.java:193-253, repeat units up to 8 bases, lengths capped at 20);
//   * the minimum-quality caps of capMinimumReadQualities (:307-320): base quality capped by the
//     read's mapping quality (unless disabled) and set to 6 below the base-quality threshold,
//     insertion / deletion quality set to 6 below 6 -- compared as Java signed bytes, so a byte of
//     128 or more counts as low.
// One wave per read, lanes over its positions; every thread writes only its own position.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pairhmm_kernels.hpp"

namespace gatk_pairhmm {
namespace {

constexpr int kMaxStrUnit = 8;
constexpr int kMaxRepeat = 20;

// Tandem copies by runs of equal bases p apart.  With e_p(k) = (s[k] == s[k + p]), F_p(u) the number of
// consecutive k >= u and B_p(u) of consecutive k < u that hold it, the unit s[u, u + p) is followed by
// floor(F_p(u) / p) copies of itself and comes after floor(B_p(u) / p).  A wave takes 64 positions' e_p as
// one 64-bit mask (a ballot); a lane's F and B are counts of ones at its bit, carried over to the
// neighbouring masks where a run reaches the mask's end.

// e_p of positions k0 .. k0 + 63 (k + p < len).
__device__ __forceinline__ uint64_t equal_mask(const uint8_t *s, int len, int k0, int p, int lane) {
    const int k = k0 + lane;
    return __ballot(k + p < len && s[k] == s[k + p]);
}

// Consecutive e_p from position k0 on, given the mask there.
__device__ __forceinline__ int run_from(const uint8_t *s, int len, int k0, int p, int lane, uint64_t mask) {
    int n = 0;
    while (mask == ~0ull) {
        n += kWave;
        k0 += kWave;
        mask = equal_mask(s, len, k0, p, lane);
    }
    return n + __builtin_ctzll(~mask);
}

// F and B at the lane's bit of `mask`; `after` ones follow the mask and `before` ones end in front of it.
__device__ __forceinline__ int ones_up(uint64_t mask, int lane, int after) {
    const uint64_t up = ~mask >> lane;
    return up ? __builtin_ctzll(up) : kWave - lane + after;
}
__device__ __forceinline__ int ones_down(uint64_t mask, int lane, int before) {
    const uint64_t down = lane ? ~mask << (kWave - lane) : 0ull;
    return down ? __builtin_clzll(down) : lane + before;
}
__device__ __forceinline__ int run_to_end(uint64_t mask, int before) {
    return mask == ~0ull ? before + kWave : __builtin_clzll(~mask);
}

// findTandemRepeatUnits(read, offset).getRight() for offset = u - 1 (ReadLikelihoodCalculationEngine.java:
// 193-253): the shortest unit of up to 8 bases that starts at u and repeats after it (else the base at u),
// its copies from u on plus its copies that end at offset.  The method's own backward unit search only
// picks which of two equal counts is taken while offset is not the read's last base, which holds for
// every position the error model changes.  Per unit length two ballots and about 25 VALU instructions for
// 64 positions, where comparing copies base by base took about 850 us for the reads of 500 regions
// (40,000 reads of 172 bases on average); 107 us now.
__global__ __launch_bounds__(256) void pcr_error_model_kernel(const uint8_t *__restrict__ bases,
                                                              const int64_t *__restrict__ read_off,
                                                              const int32_t *__restrict__ read_len, int64_t n_reads,
                                                              PcrQualTable table, uint8_t *ins, uint8_t *del) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x / kWave);
    const int64_t r0 = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    for (int64_t r = r0; r < n_reads; r += waves) {
        const int64_t o = read_off[r];
        const int len = read_len[r];
        const uint8_t *s = bases + o;
        uint64_t mask[kMaxStrUnit];
        int before[kMaxStrUnit];
#pragma unroll
        for (int p = 1; p <= kMaxStrUnit; ++p) {
            mask[p - 1] = equal_mask(s, len, 0, p, lane);
            before[p - 1] = 0;
        }
        for (int k0 = 0; k0 < len; k0 += kWave) {
            uint64_t next[kMaxStrUnit];
#pragma unroll
            for (int p = 1; p <= kMaxStrUnit; ++p) next[p - 1] = equal_mask(s, len, k0 + kWave, p, lane);
            int copies = 1 + ones_down(mask[0], lane, before[0]);
            bool found = false;
#pragma unroll
            for (int p = 1; p <= kMaxStrUnit; ++p) {
                const int up = ones_up(mask[p - 1], lane, run_from(s, len, k0 + kWave, p, lane, next[p - 1]));
                const bool now = !found && up >= p;
                if (__ballot(now) != 0) {
                    const int c = 1 + up / p + ones_down(mask[p - 1], lane, before[p - 1]) / p;
                    copies = now ? c : copies;
                    found |= now;
                }
                before[p - 1] = run_to_end(mask[p - 1], before[p - 1]);
                mask[p - 1] = next[p - 1];
            }
            const int u = k0 + lane;
            if (u >= 1 && u < len) {  // position u - 1, as in the reference loop
                const uint8_t q = table.q[copies > kMaxRepeat ? kMaxRepeat : copies];
                if (ins[o + u - 1] > q) ins[o + u - 1] = q;
                if (del[o + u - 1] > q) del[o + u - 1] = q;
            }
        }
    }
}

__device__ __forceinline__ uint8_t fixed_if_low(uint8_t v, int8_t min_q) {
    return static_cast<int8_t>(v) < min_q ? static_cast<uint8_t>(6) : v;  // QualityUtils.MIN_USABLE_Q_SCORE
}

__global__ __launch_bounds__(256) void cap_qualities_kernel(const int64_t *__restrict__ read_off,
                                                            const int32_t *__restrict__ read_len, int64_t n_reads,
                                                            const int32_t *__restrict__ mapq, int32_t bq_threshold,
                                                            int32_t disable_mapq_cap, uint8_t *quals, uint8_t *ins,
                                                            uint8_t *del) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x / kWave);
    const int8_t threshold = static_cast<int8_t>(bq_threshold);
    for (int64_t r = static_cast<int64_t>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave; r < n_reads;
         r += waves) {
        const int64_t o = read_off[r];
        const int len = read_len[r];
        const int mq = disable_mapq_cap ? 255 : mapq[r];
        for (int i = lane; i < len; i += kWave) {
            int q = quals[o + i];
            if (!disable_mapq_cap && mq < q) q = mq;
            quals[o + i] = fixed_if_low(static_cast<uint8_t>(q), threshold);
            ins[o + i] = fixed_if_low(ins[o + i], 6);
            del[o + i] = fixed_if_low(del[o + i], 6);
        }
    }
}

int read_grid(int64_t n_reads) {
    const int64_t blocks = (n_reads + 3) / 4;  // four waves (reads) per 256-thread block
    return static_cast<int>(blocks < 1 ? 1 : (blocks > 65536 ? 65536 : blocks));
}

}  // namespace

hipError_t launch_pcr_error_model(const uint8_t *bases, const int64_t *read_off, const int32_t *read_len,
                                  int64_t n_reads, const PcrQualTable &table, uint8_t *ins, uint8_t *del,
                                  hipStream_t stream) {
    if (n_reads <= 0) return hipSuccess;
    hipLaunchKernelGGL(pcr_error_model_kernel, dim3(read_grid(n_reads)), dim3(256), 0, stream, bases, read_off,
                       read_len, n_reads, table, ins, del);
    return hipGetLastError();
}

hipError_t launch_cap_qualities(const int64_t *read_off, const int32_t *read_len, int64_t n_reads, const int32_t *mapq,
                                int32_t bq_threshold, int32_t disable_mapq_cap, uint8_t *quals, uint8_t *ins,
                                uint8_t *del, hipStream_t stream) {
    if (n_reads <= 0) return hipSuccess;
    hipLaunchKernelGGL(cap_qualities_kernel, dim3(read_grid(n_reads)), dim3(256), 0, stream, read_off, read_len,
                       n_reads, mapq, bq_threshold, disable_mapq_cap, quals, ins, del);
    return hipGetLastError();
}

}  // namespace gatk_pairhmm

// ---------------------------------------------------------------------------------------------
// DRAGstr imputation on the device (DragstrPairHMMInputScoreImputator.impute,
// DragstrPairHMMInputScoreImputator.java:53-70, over the contexts of DragstrReadSTRAnalyzer,
// DragstrReadSTRAnalyzer.java:69-139).  The copy count of period p at position i is the reference
// test's brute-force definition (DragstrReadSTRAnalyzerTest.java:126-171): the longest run of equal
// adjacent p-mers through any p-mer starting in [i-p+1, i+1], one copy discounted for the p-mer at 0
// when i < p-1; the best period has the most copies, the shorter on ties.
//
// With T(u) = F_p(u) + B_p(u), the length of the run of e_p that touches u, a p-mer start u lies in
// 1 + floor(F/p) + floor(B/p) copies, and the most over the starts of the window [w0, w1] (clipped to
// [0, L-p]) is 1 + floor(max(T(w0), T(w1)) / p): a run that touches an end of the window gives all its
// copies at the run's own end if that lies in the window, else the window holds every residue; a run
// inside the window is shorter than p and gives one.  The window of a position i < p-1 begins at 0,
// whose discount is a run of T(0) - 1.
// So a wave writes T of 64 starts from one ballot, and a position reads two of them per period.
// ---------------------------------------------------------------------------------------------
namespace gatk_pairhmm {
namespace {

constexpr int kDragstrMaxRead = 4096;  // longest read taken

// The brute-force count itself, for reads over the launch's capacity (a caller's max_read_len that is
// too small).
__device__ __forceinline__ bool pmer_eq(const uint8_t *s, int a, int b, int p) {
    for (int k = 0; k < p; ++k)
        if (s[a + k] != s[b + k]) return false;
    return true;
}

__device__ int copies_at(const uint8_t *s, int L, int i, int p) {
    if (p > L) return 0;
    const int lo = i - p + 1 > 0 ? i - p + 1 : 0;
    const int hi = i + 1 < L - p ? i + 1 : L - p;
    int best = 0;
    for (int u = lo; u <= hi; ++u) {
        int f = 1;  // equal p-mers from u forward
        while (u + f * p <= L - p && pmer_eq(s, u + (f - 1) * p, u + f * p, p)) ++f;
        int b = 0;  // and backward
        while (u - (b + 1) * p >= 0 && pmer_eq(s, u - (b + 1) * p, u - b * p, p)) ++b;
        int c = f + b;
        if (u == 0 && i < p - 1) c = c - 1 > 1 ? c - 1 : 1;
        best = c > best ? c : best;
    }
    return best;
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Bound by VALU issue, about 50 instructions per period and 64 positions: the reads of 500 regions
// (40,000 of 172 bases on average), 8 periods: 163 us, against 2,580 with the brute-force count.
// A wave's LDS is sized by the longest read (7 bytes a position: bases, T, best period), so short reads
// are not held to the few waves that 4,096 positions allow (470 us at that size).
__global__ __launch_bounds__(kWave) void dragstr_impute_kernel(const uint8_t *__restrict__ bases,
                                                               const int64_t *__restrict__ read_off,
                                                               const int32_t *__restrict__ read_len, int64_t n_reads,
                                                               DragstrByteTables tables, int cap, uint8_t *out_gop,
                                                               uint8_t *out_gcp) {
    // The best period so far as copies << 10 | 1023 - period: the larger key has more copies or, on ties,
    // the shorter period (periods are at most 512).
    extern __shared__ uint32_t best[];
    uint16_t *const runs = reinterpret_cast<uint16_t *>(best + cap);
    uint8_t *const s = reinterpret_cast<uint8_t *>(runs + cap);
    const int lane = threadIdx.x;
    for (int64_t r = blockIdx.x; r < n_reads; r += gridDim.x) {
        const int64_t o = read_off[r];
        const int L = __builtin_amdgcn_readfirstlane(read_len[r]);
        if (L > kDragstrMaxRead) continue;  // the host rejects such batches up front
        wave_lds_sync();
        if (L <= cap) {
            for (int i = lane; i < L; i += kWave) {
                s[i] = bases[o + i];
                best[i] = 0u;
            }
            wave_lds_sync();
            for (int p = 1; p <= tables.max_period && p <= L; ++p) {
                uint64_t mask = equal_mask(s, L, 0, p, lane);
                int before = 0;
                for (int k0 = 0; k0 <= L - p; k0 += kWave) {
                    const uint64_t next = equal_mask(s, L, k0 + kWave, p, lane);
                    const int after = run_from(s, L, k0 + kWave, p, lane, next);
                    if (k0 + lane <= L - p)
                        runs[k0 + lane] =
                            static_cast<uint16_t>(ones_up(mask, lane, after) + ones_down(mask, lane, before));
                    before = run_to_end(mask, before);
                    mask = next;
                }
                wave_lds_sync();
                const float inv_p = 1.0f / static_cast<float>(p);
                for (int i = lane; i < L - 1; i += kWave) {
                    const int w0 = i - p + 1 > 0 ? i - p + 1 : 0, w1 = i + 1 < L - p ? i + 1 : L - p;
                    int t0 = runs[w0], t1 = runs[w1];
                    if (i < p - 1 && t0 > 0) {
                        if (t0 >= w1) t1 -= 1;  // the same run
                        t0 -= 1;
                    }
                    // floor(t / p) in FP32: (t + 0.5) / p is at least 0.5 / p from a whole number, far
                    // more than its rounding error for t <= 4096 and p <= 512.
                    const int t = t0 > t1 ? t0 : t1;
                    const uint32_t c = 1u + static_cast<uint32_t>((static_cast<float>(t) + 0.5f) * inv_p);
                    const uint32_t key = c << 10 | (1023u - static_cast<uint32_t>(p));
                    if (key > best[i]) best[i] = key;
                }
                wave_lds_sync();
            }
        }
        for (int i = lane; i < L; i += kWave) {
            if (i == L - 1) {  // DragstrPairHMMInputScoreImputator.java:22-23,69-70
                out_gop[o + i] = 45;
                out_gcp[o + i] = 10;
                continue;
            }
            int best_p = 1, best_c = 0;
            if (L <= cap) {
                best_c = static_cast<int>(best[i] >> 10);
                best_p = 1023 - static_cast<int>(best[i] & 1023u);
            } else {
                for (int p = 1; p <= tables.max_period; ++p) {
                    const int c = copies_at(bases + o, L, i, p);
                    if (c > best_c) {
                        best_c = c;
                        best_p = p;
                    }
                }
            }
            const int rep = best_c < 1 ? 1 : (best_c > tables.max_repeats ? tables.max_repeats : best_c);
            const int cell = (best_p - 1) * tables.max_repeats + rep - 1;
            out_gop[o + i] = tables.gop[cell];
            out_gcp[o + i] = tables.gcp[cell];
        }
    }
}

// Best keys, run lengths (of starts 0..L-1) and bases of `cap` positions.
constexpr size_t dragstr_lds_bytes(int cap) { return static_cast<size_t>(cap) * (4 + 2 + 1); }
static_assert(dragstr_lds_bytes(kDragstrMaxRead) <= 65536, "a read's LDS fits the default dynamic limit");

}  // namespace

hipError_t launch_dragstr_impute(const uint8_t *bases, const int64_t *read_off, const int32_t *read_len,
                                 int64_t n_reads, const DragstrByteTables &tables, uint8_t *out_gop, uint8_t *out_gcp,
                                 hipStream_t stream) {
    if (n_reads <= 0) return hipSuccess;
    const int64_t grid = n_reads < 65536 ? n_reads : 65536;
    const int longest = tables.max_read_len < kDragstrMaxRead ? tables.max_read_len : kDragstrMaxRead;
    const int cap = (longest < 1 ? 1 : (longest + kWave - 1) / kWave) * kWave;
    hipLaunchKernelGGL(dragstr_impute_kernel, dim3(static_cast<unsigned>(grid)), dim3(kWave), dragstr_lds_bytes(cap), stream,
                       bases, read_off, read_len, n_reads, tables, cap, out_gop, out_gcp);
    return hipGetLastError();
}

int dragstr_max_read_length() { return kDragstrMaxRead; }

}  // namespace gatk_pairhmm
