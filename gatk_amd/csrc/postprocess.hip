// postprocess.hip -- the likelihood post-processing that follows the PairHMM, on the device, so the
// read x haplotype matrix need not travel to the host for it
// (PairHMMLikelihoodCalculationEngine.computeReadLikelihoods,
// src/main/java/org/broadinstitute/hellbender/tools/walkers/haplotypecaller/PairHMMLikelihoodCalculationEngine.java:200-201):
//   1. the mismapping-rate cap, AlleleLikelihoods.normalizeLikelihoods
//      (src/main/java/org/broadinstitute/hellbender/utils/genotyper/AlleleLikelihoods.java:416-458):
//      per read, every likelihood below best + cap is raised to it, best being searchBestAllele's
//      (:505-533; the reference allele is skipped unless normalisation is symmetric);
//   2. the poorly-modelled read filter, filterPoorlyModeledEvidence
//      (ReadLikelihoodCalculationEngine.java:98-155, AlleleLikelihoods.java:1351-1375): a read is
//      dropped when its best likelihood is below ceil(L * rate) * -4 (at most 2 errors unless the
//      DRAGEN dynamic threshold is on, which takes the lower of that and
//      -0.1 (sum mean_q + K sqrt(sum var_q)) over the read's HMM base qualities).
// One thread per read.  A wave's 64 matrix rows are staged through LDS with coalesced loads; a lane reads
// its own qualities, 64 bytes at a time.  FP64 with contraction off, so every sum and product rounds where
// Java's do (the quality sums run in read order).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "pairhmm_kernels.hpp"

namespace gatk_pairhmm {
namespace {

// ReadLikelihoodCalculationEngine.dynamicReadQualThreshLookupTable (:161-176): mean and variance for
// base qualities 1..40, the reference's values.
__constant__ double kDynMean[40] = {
    5.996842844, 5.870018422, 5.401558531, 4.818940919, 4.218758304, 3.646319832, 3.122346753, 2.654731979,
    2.244479156, 1.88893867,  1.583645342, 1.3233807,   1.102785365, 0.916703025, 0.760361881, 0.629457387,
    0.520175654, 0.42918208,  0.353590663, 0.290923699, 0.23906788,  0.196230431, 0.160897421, 0.131795374,
    0.1078567,   0.088189063, 0.072048567, 0.058816518, 0.047979438, 0.039111985, 0.031862437, 0.025940415,
    0.021106532, 0.017163711, 0.013949904, 0.011332027, 0.009200898, 0.007467036, 0.006057179, 0.004911394};
__constant__ double kDynVar[40] = {
    0.196616587, 1.388545569, 5.641990128, 10.33176216, 14.25799688, 17.02880749, 18.64537883, 19.27521677,
    19.13584613, 18.43922003, 17.36842261, 16.07088712, 14.65952563, 13.21718577, 11.80207947, 10.45304833,
    9.194183767, 8.038657241, 6.991779595, 6.053379213, 5.219610436, 4.484302033, 3.839943445, 3.27839108,
    2.791361596, 2.370765375, 2.008921719, 1.698687797, 1.433525748, 1.207526336, 1.015402928, 0.852465956,
    0.714585285, 0.598145851, 0.500000349, 0.41742159,  0.348056286, 0.289881373, 0.241163527, 0.200422214};

constexpr int kPpWaves = 4;             // waves per workgroup, each over 64 consecutive reads
constexpr int kRowStage = 512;          // likelihoods a wave stages in LDS (64 reads x 8 haplotypes)
constexpr int kNoQual = 256;            // table entry of a byte outside the read: adds 0
constexpr int kGranules = 4;            // 16-byte granules of a lane's qualities in flight

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A lane's qualities as 16-byte granules of a span of `len` bytes (quality_lead): kGranules from granule k, those that
// hold any.
__device__ __forceinline__ void load_granules(uint4 (&g)[kGranules], const uint8_t *span, int k, int len) {
#pragma unroll
    for (int i = 0; i < kGranules; ++i)
        if (16 * (k + i) < len) __builtin_memcpy(&g[i], span + quality_granule_at(len, k + i), 16);
}

// The granule of a span of fewer than 16 bytes: the read's bytes come last, as in a longer span's last granule.
__device__ __forceinline__ uint4 load_short(const uint8_t *q, int L) {
    uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int b = 1; b < 16; ++b)
        if (b >= 16 - L) w[b / 4] |= static_cast<uint32_t>(q[b - (16 - L)]) << (8 * (b % 4));
    return uint4{w[0], w[1], w[2], w[3]};
}

// Adds the table entries of a granule's 16 bytes, in order; its first `skip` bytes add entry kNoQual.  kWhole:
// none is skipped.
template <bool kWhole>
__device__ __forceinline__ void add_granule(const uint4 &g, int skip, const double2 *tab, double &s_mean, double &s_var) {
#pragma clang fp contract(off)
    const uint32_t w[4] = {g.x, g.y, g.z, g.w};
#pragma unroll
    for (int b = 0; b < 16; ++b) {
        uint32_t e = (w[b / 4] >> (8 * (b % 4))) & 0xFFu;
        if (!kWhole) e = b >= skip ? e : kNoQual;
        const double2 mv = tab[e];
        s_mean += mv.x;
        s_var += mv.y;
    }
}

// The kernel is bound by HBM latency and by the LDS lookups, 16 bytes per quality at lane-random entries.
// Staging the qualities in LDS too held a CU to ten waves, took only spans of up to 10,240 bytes per wave
// (reads of 160 on average; longer ones went byte by byte from global memory) and ran 13 VALU instructions
// per quality; a lane's own 64-byte loads touch each line about twice and leave 6.  400,000 reads x 8
// haplotypes, 100-250 bases: a call takes 64 us, 95 with the staged qualities (63 with last granules that may end
// after the plane).
__global__ __launch_bounds__(kPpWaves * 64) void postprocess_kernel(PostprocessArgs p) {
#pragma clang fp contract(off)
    // The table in LDS by quality byte: per-base lookups differ lane to lane, which LDS serves far better
    // than gathers from global memory.
    __shared__ double2 tab[kNoQual + 1];
    // Each wave's rows are adjacent in the matrix: brought into LDS with coalesced loads, worked on there,
    // and written back coalesced.
    __shared__ double rstage[kPpWaves][kRowStage];
    if (p.dynamic) {  // the same for the whole launch; a call without it waits for no table (85 reads: 15.7 us, 15.4)
        for (int q = threadIdx.x; q <= kNoQual; q += blockDim.x) {
            const int e = q <= 1 ? 0 : (q < 40 ? q : 40) - 1;
            tab[q] = q == kNoQual ? make_double2(0.0, 0.0) : make_double2(kDynMean[e], kDynVar[e]);
        }
        __syncthreads();
    }
    const int w = static_cast<int>(threadIdx.x) / 64, lane = static_cast<int>(threadIdx.x) % 64;
    const int64_t r0 = (static_cast<int64_t>(blockIdx.x) * kPpWaves + w) * 64;
    if (r0 >= p.n_reads) return;  // the whole wave
    const int nr = p.n_reads - r0 < 64 ? static_cast<int>(p.n_reads - r0) : 64;
    const bool has = lane < nr;
    const int64_t r = r0 + lane;
    const int A = p.n_alleles;

    const bool stage_rows = static_cast<int64_t>(nr) * A <= kRowStage;
    double *const grow = p.likelihoods + r0 * A;
    const int L = has ? p.read_len[r] : 0;
    const uint8_t *q = p.base_quals + (has && p.dynamic ? p.read_off[r] : 0);
    // The wave's first HBM loads are issued before the first wait: the rows (nr * A <= kRowStage = 8 * 64, so
    // eight values per lane) and the first granules of each lane's qualities.
    double rt[kRowStage / 64];
    if (stage_rows) {
#pragma unroll
        for (int u = 0; u < kRowStage / 64; ++u) {
            const int e = lane + 64 * u;
            rt[u] = e < nr * A ? grow[e] : 0.0;
        }
    }
    const int n_quals = p.dynamic && L > 0 ? L : 0;
    const int lead = quality_lead(reinterpret_cast<uintptr_t>(q), n_quals, reinterpret_cast<uintptr_t>(p.base_quals));
    const int span_len = lead + n_quals;
    uint4 g[kGranules] = {};
    const int wide_len = span_len >= 16 ? span_len : 0;
    load_granules(g, q - lead, 0, wide_len);
    if (n_quals > 0 && span_len < 16) g[0] = load_short(q, n_quals);
    if (stage_rows) {
#pragma unroll
        for (int u = 0; u < kRowStage / 64; ++u) {
            const int e = lane + 64 * u;
            if (e < nr * A) rstage[w][e] = rt[u];
        }
        wave_lds_sync();
    }
    double *v = !has ? rstage[w] : stage_rows ? &rstage[w][lane * A] : p.likelihoods + r * A;

    if (has && p.normalize && A >= 2) {
        const bool can_ref = p.symmetric != 0;
        const int b0 = (can_ref || p.ref_index != 0) ? 0 : 1;
        double best = v[b0];
        for (int a = b0 + 1; a < A; ++a) {
            if (!can_ref && a == p.ref_index) continue;
            const double c = v[a];
            if (c > best) best = c;
        }
        const double worst = best + p.cap;
        for (int a = 0; a < A; ++a)
            if (v[a] < worst) v[a] = worst;
    }
    const double errors = ceil(static_cast<double>(L) * p.max_error_per_base);
    double t = (p.dynamic ? errors : fmin(2.0, errors)) * -4.0;
    if (p.dynamic) {
        // Sums in read order, as the reference adds them, the next granules loading meanwhile.
        double s_mean = 0.0, s_var = 0.0;
        for (int k = 0; __any(16 * k < span_len); k += kGranules) {
            uint4 next[kGranules] = {};
            load_granules(next, q - lead, k + kGranules, wide_len);
#pragma unroll
            for (int i = 0; i < kGranules; ++i) {
                const int skip = quality_granule_skip(span_len, lead, k + i);
                if (__all(skip <= 0))
                    add_granule<true>(g[i], skip, tab, s_mean, s_var);
                else if (__any(skip < 16))
                    add_granule<false>(g[i], skip, tab, s_mean, s_var);
            }
#pragma unroll
            for (int i = 0; i < kGranules; ++i) g[i] = next[i];
        }
        const double d = (s_mean + p.scale * sqrt(s_var)) * -0.1;
        if (d < t) t = d;
    }
    if (has) {
        double m = -__builtin_inf();
        for (int a = 0; a < A; ++a)
            if (v[a] > m) m = v[a];
        p.keep[r] = (m < t) ? 0 : 1;
        if (p.threshold) p.threshold[r] = t;
    }
    if (stage_rows && p.normalize && A >= 2) {
        wave_lds_sync();
        for (int e = lane; e < nr * A; e += 64) grow[e] = rstage[w][e];
    }
}

}  // namespace

hipError_t launch_postprocess(const PostprocessArgs &args, hipStream_t stream) {
    if (args.n_reads <= 0) return hipSuccess;
    const int64_t per_block = 64 * kPpWaves;
    const int64_t grid = (args.n_reads + per_block - 1) / per_block;
    hipLaunchKernelGGL(postprocess_kernel, dim3(static_cast<unsigned>(grid)), dim3(per_block), 0, stream, args);
    return hipGetLastError();
}

}  // namespace gatk_pairhmm
