"""The work that users of this engine have it do, as cases that can be timed and checked.

A variant caller hands the engine one active region at a time (reads x haplotypes through the
drop-in call), or many regions as a batch that stays on the device; around that it prepares the
reads' qualities, caps and filters the likelihoods and realigns reads to their best haplotypes; a
penalty fit needs the likelihoods' gradients.  Every case goes through the package's public entry
points.  Sizes are those of the package's workloads (gatk_amd/synth.py): regions of 2-128 haplotypes
of 150-600 bases and about 80 reads of 100-250 bases, regions of long low-quality reads on STR-rich
haplotypes of 800-1,500 bases, and the streaming mix of the two.

Kinds and what they stand for:
  region      one computeLikelihoods call, host arrays in and out (forward)
  batch       many regions resident on the device, one forward pass, likelihoods back to the host
  chunk       one chunk of a stream of regions: upload, forward, likelihoods back, free
  train       log10 likelihoods and their gradients by per-base penalties (forward and backward)
  pd_region   one partially determined computeLikelihoods call
  align       Smith-Waterman of a list of pairs in one call, host sequences in, CIGARs out
  read_prep   DRAGstr penalties, PCR indel error model and quality caps over a chunk's reads
  post        mismapping cap and read filter over a likelihood matrix on the device
"""
import math
import zlib

import numpy as np
import torch

from gatk_amd import synth
from gatk_amd.autograd import GradEngine, GradProblem, pairhmm_log10_likelihood
from gatk_amd.batch import BatchEngine, PackedBatch
from gatk_amd.dragstr import DragstrParams
from gatk_amd.pairhmm import HaplotypeDataHolder, HipPairHmm, PairHMMNativeArguments, ReadDataHolder
from gatk_amd.pdhmm import DEL_END, DEL_START, SNP, HipPDHmm
from gatk_amd.pdhmm import HaplotypeDataHolder as PDHaplotypeDataHolder
from gatk_amd.postprocess import LikelihoodPostProcessor, log10_mismapping_cap
from gatk_amd.readprep import PCRErrorModel, ReadPrep
from gatk_amd.smithwaterman import (ALIGNMENT_TO_BEST_HAPLOTYPE_SW_PARAMETERS, NEW_SW_PARAMETERS,
                                    HipSmithWatermanBinding, SWOverhangStrategy)

DEV = "cuda"

# Read and haplotype profiles: base qualities, error rates, STR content.
PROFILES = {
    "plain": synth.PLAIN_SMALL,       # short reads of good quality
    "uneven": synth.BATCHED_UNEVEN,   # base quality 10-40, 1 % substitutions, few indels
    "stress": synth.PRECISION_STRESS, # base quality 2-15, 5 % substitutions, STR-rich haplotypes
}


def listed():
    return [
        # The smallest call: a low-coverage region with few haplotypes, where launches and copies count.
        {"name": "region_small", "kind": "region", "profile": "plain", "reads": 64, "haps": 16, "hap_len": 300,
         "read_min": 150, "read_max": 150, "double": False},
        # The ordinary call: mean coverage, mean haplotype count and length, ragged reads.
        {"name": "region_typical", "kind": "region", "profile": "uneven", "reads": 81, "haps": 65, "hap_len": 377,
         "read_min": 100, "read_max": 250, "double": False},
        # The largest call: the coverage and haplotype limits on the longest window.
        {"name": "region_large", "kind": "region", "profile": "uneven", "reads": 1000, "haps": 128, "hap_len": 600,
         "read_min": 100, "read_max": 250, "double": False},
        # A batch of ordinary regions on the device: throughput of the FP32 pass.
        {"name": "batch_uneven", "kind": "batch", "profile": "uneven", "regions": 300, "stress_part": 0.0},
        # A batch of long low-quality reads, most of which need the FP64 pass.
        {"name": "batch_stress", "kind": "batch", "profile": "stress", "regions": 40, "stress_part": 0.0},
        # One chunk of a stream of regions of both kinds: every chunk is new, so the upload counts.
        {"name": "chunk_mix", "kind": "chunk", "profile": "uneven", "regions": 100, "stress_part": 0.1},
        # One step of a penalty fit: likelihoods and gradients over a batch of regions.
        {"name": "train_step", "kind": "train", "profile": "uneven", "regions": 100},
        # The ordinary call of the partially determined model.
        {"name": "pd_region", "kind": "pd_region", "reads": 81, "haps": 65, "hap_len": 377, "read_min": 100,
         "read_max": 250},
        # A region's reads against their best haplotypes.
        {"name": "align_region", "kind": "align", "pairs": 81, "what": "reads"},
        # A chunk's reads against their best haplotypes in one call.
        {"name": "align_chunk", "kind": "align", "pairs": 20000, "what": "reads"},
        # The reads of a chunk before the HMM.
        {"name": "read_prep", "kind": "read_prep", "regions": 500, "stress_part": 0.1},
        # A chunk's likelihood matrix after the HMM.
        {"name": "post", "kind": "post", "reads": 400000, "alleles": 8, "read_min": 100, "read_max": 250,
         "dynamic": True},
    ]


def _log_int(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("region", "region", "batch", "batch", "chunk", "train", "pd_region", "align", "read_prep", "post"))
    lo = rng.randint(80, 180)
    if kind == "region":
        profile = rng.choice(("plain", "uneven", "uneven", "stress"))
        if profile == "stress":
            return {"kind": kind, "profile": profile, "reads": _log_int(rng, 5, 150), "haps": _log_int(rng, 2, 64),
                    "hap_len": rng.randint(800, 1500), "read_min": 250, "read_max": rng.randint(260, 600),
                    "double": False}
        return {"kind": kind, "profile": profile, "reads": _log_int(rng, 3, 1000), "haps": _log_int(rng, 2, 128),
                "hap_len": rng.randint(150, 600), "read_min": lo, "read_max": lo + rng.randint(0, 90),
                "double": rng.random() < 0.2}
    if kind in ("batch", "chunk"):
        if kind == "batch" and rng.random() < 0.4:
            return {"kind": kind, "profile": "stress", "regions": _log_int(rng, 2, 40), "stress_part": 0.0}
        return {"kind": kind, "profile": "uneven", "regions": _log_int(rng, 5, 100),
                "stress_part": rng.choice((0.0, 0.1)) if kind == "batch" else 0.1}
    if kind == "train":
        return {"kind": kind, "profile": rng.choice(("plain", "uneven")), "regions": _log_int(rng, 3, 80)}
    if kind == "pd_region":
        return {"kind": kind, "reads": _log_int(rng, 3, 300), "haps": _log_int(rng, 2, 128),
                "hap_len": rng.randint(150, 600), "read_min": lo, "read_max": lo + rng.randint(0, 90)}
    if kind == "align":
        what = rng.choice(("reads", "reads", "haplotypes"))
        return {"kind": kind, "pairs": _log_int(rng, 5, 15000 if what == "reads" else 2000), "what": what}
    if kind == "read_prep":
        return {"kind": kind, "regions": _log_int(rng, 5, 400), "stress_part": rng.choice((0.0, 0.1))}
    return {"kind": kind, "reads": _log_int(rng, 50, 400000), "alleles": rng.randint(2, 17), "read_min": lo,
            "read_max": lo + rng.randint(0, 90), "dynamic": rng.random() < 0.7}


# ---- inputs --------------------------------------------------------------------------------------


def _sizes(case):
    """Per region (window, haplotypes, read lengths, profile): of the case alone, so that inputs of every
    seed have the same sizes."""
    rng = np.random.default_rng(zlib.crc32(repr(sorted((k, v) for k, v in case.items() if k != "name")).encode()))
    main = PROFILES[case.get("profile", "uneven")]
    part = case.get("stress_part", 0.0)
    got = []
    for k in range(case.get("regions", 1)):
        sp = synth.PRECISION_STRESS if rng.random() < part else main
        if "reads" in case:
            window, haps, reads = case["hap_len"], case["haps"], case["reads"]
            lo, hi = case["read_min"], case["read_max"]
        else:
            window = int(rng.integers(sp.window[0], sp.window[1] + 1))
            haps = sp.fixed_haps or int(rng.integers(sp.n_haps[0], sp.n_haps[1] + 1))
            reads = sp.fixed_reads or int(np.clip(rng.poisson(sp.reads_mean), *sp.reads_clamp))
            lo, hi = sp.read_len
        longest = window - sp.hap_indels[1] * sp.hap_indel_len[1]  # of the shortest haplotype
        got.append((window, haps, np.minimum(rng.integers(lo, hi + 1, reads), longest), sp))
    return got


def _window(rng, n, spec):
    """Reference bases, with short tandem repeats between random flanks where the profile has them."""
    if not spec.str_rich:
        return synth.BASES[rng.integers(0, 4, n)]
    parts, total = [], 0
    while total < n:
        motif = synth.BASES[rng.integers(0, 4, int(rng.integers(spec.str_motif[0], spec.str_motif[1] + 1)))]
        tract = np.tile(motif, int(rng.integers(spec.str_repeats[0], spec.str_repeats[1] + 1)))
        parts += [synth.BASES[rng.integers(0, 4, int(rng.integers(10, 60)))], tract]
        total += len(parts[-2]) + len(tract)
    return np.concatenate(parts)[:n]


def _with_indel(rng, seq, length):
    """`seq` with an insertion or a deletion of `length` bases at a random place."""
    p = int(rng.integers(0, len(seq) - length))
    if rng.random() < 0.5:
        return np.concatenate([seq[:p], synth.BASES[rng.integers(0, 4, length)], seq[p:]])
    return np.concatenate([seq[:p], seq[p + length:]])


def _haplotype(rng, window, spec):
    """The window with a few SNPs and indels."""
    h = window.copy()
    at = rng.integers(0, len(h), int(rng.integers(spec.hap_snps[0], spec.hap_snps[1] + 1)))
    h[at] = synth.BASES[rng.integers(0, 4, len(at))]
    for _ in range(int(rng.integers(spec.hap_indels[0], spec.hap_indels[1] + 1))):
        h = _with_indel(rng, h, int(rng.integers(spec.hap_indel_len[0], spec.hap_indel_len[1] + 1)))
    return h


def _regions(case, seed):
    """The case's regions, packed: haplotypes mutated from a window, reads sampled from them with
    substitutions and indels."""
    rng = np.random.Generator(np.random.PCG64(seed))
    haps, bases, quals, lens = [], [], [], []
    pr, ph, rpo, rro, rho = [], [], [0], [0], [0]
    for window, n_haps, R, sp in _sizes(case):
        win = _window(rng, window, sp)
        hs = [_haplotype(rng, win, sp) for _ in range(n_haps)]
        hl = np.array([len(h) for h in hs])
        cat, ho = np.concatenate(hs), np.cumsum(hl) - hl
        src = rng.integers(0, n_haps, len(R))
        start = ho[src] + (rng.random(len(R)) * (hl[src] - R + 1)).astype(np.int64)
        at = np.repeat(start - (np.cumsum(R) - R), R) + np.arange(R.sum())
        read = cat[at]
        sub = np.nonzero(rng.random(len(read)) < sp.sub_rate)[0]
        read[sub] = synth.BASES[rng.integers(0, 4, len(sub))]
        ends = np.cumsum(R)
        for k in np.nonzero(rng.random(len(R)) < sp.indel_rate * R)[0]:
            n, e = int(R[k]), int(ends[k])
            longer = np.concatenate([read[e - n:e], synth.BASES[rng.integers(0, 4, sp.indel_len[1])]])
            read[e - n:e] = _with_indel(rng, longer, int(rng.integers(sp.indel_len[0], sp.indel_len[1] + 1)))[:n]
        pr.append(np.repeat(np.arange(rro[-1], rro[-1] + len(R), dtype=np.int32), n_haps))
        ph.append(np.tile(np.arange(rho[-1], rho[-1] + n_haps, dtype=np.int32), len(R)))
        haps += hs
        bases.append(read)
        quals.append(rng.integers(sp.base_q[0], sp.base_q[1] + 1, len(read)).astype(np.uint8))
        lens.append(R)
        rpo.append(rpo[-1] + len(R) * n_haps)
        rro.append(rro[-1] + len(R))
        rho.append(rho[-1] + n_haps)
    bases, rl, hl = np.concatenate(bases), np.concatenate(lens).astype(np.int32), np.array([len(h) for h in haps], np.int32)
    n = len(bases)
    return PackedBatch(
        read_bases=bases, read_quals=np.concatenate(quals), read_ins=np.full(n, 45, np.uint8),
        read_del=np.full(n, 45, np.uint8), read_gcp=np.full(n, 10, np.uint8),
        read_off=np.cumsum(rl, dtype=np.int64) - rl, read_len=rl, hap_bases=np.concatenate(haps),
        hap_off=np.cumsum(hl, dtype=np.int64) - hl, hap_len=hl, pair_read=np.concatenate(pr), pair_hap=np.concatenate(ph),
        region_pair_off=np.array(rpo, np.int64), region_read_off=np.array(rro, np.int64),
        region_hap_off=np.array(rho, np.int64))


def _pd_bytes(b, seed):
    """Per haplotype three SNP columns with one to four alternatives and one optional deletion of one
    to eight bases."""
    rng = np.random.default_rng(seed)
    pd = np.zeros(len(b.hap_bases), np.uint8)
    for o, n in zip(b.hap_off.tolist(), b.hap_len.tolist()):
        for j in rng.choice(n, 3, replace=False):
            pd[o + j] = SNP | (int(rng.integers(1, 16)) << 3)
        s = int(rng.integers(0, n - 8))
        pd[o + s] |= DEL_START
        pd[o + s + int(rng.integers(0, 8))] |= DEL_END
    return pd


def _penalties(b, seed):
    """Phred values of a fit in progress, one per read base: the base qualities, and penalties around
    the usual gap-open 45 and gap-continuation 10."""
    rng = np.random.default_rng(seed)
    n = len(b.read_bases)
    return {"qb": b.read_quals.astype(np.float32), "qi": rng.uniform(35, 45, n).astype(np.float32),
            "qd": rng.uniform(35, 45, n).astype(np.float32), "qc": rng.uniform(9, 12, n).astype(np.float32)}


def _pairs_to_align(case, seed):
    """Reads with the haplotype of their region that they go to, or haplotypes with their region's
    padded reference."""
    n = case["pairs"]
    rng = np.random.default_rng(seed)
    if case["what"] == "haplotypes":
        refs, alts = [], []
        for k in range(-(-n // 30)):
            ref = synth.BASES[rng.integers(0, 4, int(rng.integers(250, 701)))]
            alts += [_haplotype(rng, ref[50:-50], synth.BATCHED_UNEVEN).tobytes() for _ in range(30)]
            refs += [ref.tobytes()] * 30
        return refs[:n], alts[:n]
    refs, alts = [], []
    for k in range(-(-n // 81)):
        one = {"reads": 81, "haps": 8, "hap_len": int(rng.integers(150, 601)), "read_min": 100, "read_max": 250}
        b = _regions(one, seed + k)
        reads, haps = b.region(0)
        refs += [haps[h].tobytes() for h in rng.integers(0, len(haps), len(reads))]
        alts += [r[0].tobytes() for r in reads]
    return refs[:n], alts[:n]


def _matrix(case, seed):
    """Likelihoods (reads x alleles), base qualities and read extents of a chunk, on the device."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    n = case["reads"]
    lens = torch.randint(case["read_min"], case["read_max"] + 1, (n,), generator=g, device=DEV, dtype=torch.int32)
    off = torch.cumsum(lens, 0, dtype=torch.int64) - lens
    quals = torch.randint(2, 41, (int(lens.sum()),), generator=g, device=DEV, dtype=torch.uint8)
    u = torch.rand((n, case["alleles"]), generator=g, device=DEV, dtype=torch.float64)
    return 15.0 * torch.log(u.clamp_min(1e-300)), quals, off, lens


# ---- what a program keeps ------------------------------------------------------------------------

_kept = {}


def _handle(name, make):
    """The engine handle of a kind, made once, as a program does."""
    if name not in _kept:
        _kept[name] = make()
    return _kept[name]


def _hmm(double):
    h = HipPairHmm()
    if not h.load():
        raise RuntimeError("no gfx950 device")
    h.initialize(PairHMMNativeArguments(use_double_precision=double))
    return h


def _pdhmm():
    h = HipPDHmm()
    if not h.load():
        raise RuntimeError("no gfx950 device")
    h.initialize()
    return h


def _aligner():
    h = HipSmithWatermanBinding()
    if not h.load():
        raise RuntimeError("no gfx950 device")
    return h


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind in ("region", "pd_region"):
        b = _regions(case, seed)
        reads, haps = b.region(0)
        s["reads"] = [ReadDataHolder(*r) for r in reads]
        s["out"] = np.empty(len(reads) * len(haps))
        if kind == "region":
            s["haps"] = [HaplotypeDataHolder(h) for h in haps]
            s["hmm"] = _handle("hmm64" if case["double"] else "hmm", lambda: _hmm(case["double"]))
        else:
            pd = _pd_bytes(b, seed)
            s["haps"] = [PDHaplotypeDataHolder(h, pd[o:o + len(h)]) for h, o in zip(haps, b.hap_off.tolist())]
            s["hmm"] = _handle("pdhmm", _pdhmm)
    elif kind in ("batch", "chunk"):
        b = _regions(case, seed)
        s["engine"] = _handle("batch", BatchEngine)
        s["out"] = np.empty(b.n_pairs)
        if kind == "batch":
            s["batch"] = s["engine"].upload(b)
        else:
            s["regions"] = b
    elif kind == "train":
        b = _regions(case, seed)
        s["problem"] = GradProblem.from_batch(b, DEV)
        s["q"] = {k: torch.from_numpy(v).to(DEV).requires_grad_() for k, v in _penalties(b, seed).items()}
        s["engine"] = _handle("grad", GradEngine)
    elif kind == "align":
        s["refs"], s["alts"] = _pairs_to_align(case, seed)
        s["params"] = NEW_SW_PARAMETERS if case["what"] == "haplotypes" else ALIGNMENT_TO_BEST_HAPLOTYPE_SW_PARAMETERS
        s["aligner"] = _handle("align", _aligner)
    elif kind == "read_prep":
        b = _regions(case, seed)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
        mapq = np.random.default_rng(seed).integers(20, 61, len(b.read_len)).astype(np.int32)
        s.update(bases=dev(b.read_bases), off=dev(b.read_off), len=dev(b.read_len.astype(np.int32)), mapq=dev(mapq),
                 quals=dev(b.read_quals), ins=dev(b.read_ins), dele=dev(b.read_del), params=DragstrParams.default(),
                 max_len=int(b.read_len.max()))
        s["gop"], s["gcp"] = torch.empty_like(s["bases"]), torch.empty_like(s["bases"])
        s["prep"] = _handle("prep", ReadPrep)
    elif kind == "post":
        s["lk"], s["quals"], s["off"], s["len"] = _matrix(case, seed)
        s["keep"] = torch.empty(case["reads"], dtype=torch.uint8, device=DEV)
        s["threshold"] = torch.empty(case["reads"], dtype=torch.float64, device=DEV)
        s["cap"] = log10_mismapping_cap(45)
        s["dynamic"] = case["dynamic"]
        s["post"] = _handle("post", LikelihoodPostProcessor)
    else:
        raise ValueError(kind)
    torch.cuda.synchronize()  # the engines work on streams of their own
    return s


def run(s):
    kind = s["kind"]
    if kind in ("region", "pd_region"):
        s["hmm"].compute_likelihoods(s["reads"], s["haps"], s["out"])
        return s["out"]
    if kind == "batch":
        s["batch"].forward(out=s["out"])
        return s["out"]
    if kind == "chunk":
        dev = s["engine"].upload(s["regions"])
        dev.forward(out=s["out"])
        dev.free()
        return s["out"]
    if kind == "train":
        q = s["q"]
        for t in q.values():
            t.grad = None
        lk = pairhmm_log10_likelihood(s["problem"], q["qb"], q["qi"], q["qd"], q["qc"], s["engine"])
        lk.sum().backward()
        return {"log10_likelihood": lk.detach(), **{k: t.grad for k, t in q.items()}}
    if kind == "align":
        got = s["aligner"].align_batch(s["refs"], s["alts"], s["params"], SWOverhangStrategy.SOFTCLIP)
        text = "\n".join([c for c, _ in got]).encode()
        cigars = np.zeros(64 * len(got), np.uint8)
        cigars[:len(text)] = np.frombuffer(text, np.uint8)
        return {"cigars": cigars, "offsets": np.array([o for _, o in got], np.int32)}
    if kind == "read_prep":
        s["prep"].dragstr_impute(s["params"], s["bases"], s["off"], s["len"], s["gop"], s["gcp"], s["max_len"])
        # In place; a second pass leaves every byte as the first one did.
        s["prep"].modify_read_qualities(s["bases"], s["off"], s["len"], s["quals"], s["ins"], s["dele"],
                                        PCRErrorModel.CONSERVATIVE, mapping_quality=s["mapq"])
        return {"gop": s["gop"], "gcp": s["gcp"], "quals": s["quals"], "ins": s["ins"], "del": s["dele"]}
    # In place; a second cap leaves every value as the first one did.
    s["post"].normalize_and_filter(s["lk"], s["len"], 0, s["cap"], False, s["quals"], s["off"], 0.02, s["dynamic"], 1.0,
                                   s["keep"], s["threshold"])
    return {"likelihoods": s["lk"], "keep": s["keep"], "threshold": s["threshold"]}


# ---- the work a pass cannot do without -----------------------------------------------------------


def work(case):
    """Means over the case's distributions.  Floating operations per cell (read base x haplotype base):
    12 of the forward recurrence (M 6, I 3, D 3), 24 more of its adjoint; integer work counts its
    scores' additions and comparisons (10 a cell)."""
    kind = case["kind"]
    if kind == "post":
        n, a, length = case["reads"], case["alleles"], (case["read_min"] + case["read_max"]) / 2
        return {"bytes": n * (16 * a + length * case["dynamic"] + 21), "flops": n * (3 * a + 2 * length * case["dynamic"])}
    if kind == "align":
        a, r = (175, 363) if case["what"] == "reads" else (375, 475)
        return {"bytes": case["pairs"] * (a + r + 16), "flops": case["pairs"] * a * r * 10}
    part = case.get("stress_part", 0.0)
    if kind in ("region", "pd_region"):
        stress = case.get("profile") == "stress"
        reads, haps, length, regions = case["reads"], case["haps"], (case["read_min"] + case["read_max"]) / 2, 1
        sizes = [(1.0, min(length, case["hap_len"]), case["hap_len"])]
    else:
        stress = case.get("profile") == "stress"
        reads, haps, regions = 80, 65, case["regions"]
        if case.get("profile") == "plain":
            reads, haps, sizes = 64, 16, [(1.0, 150, 300)]
        else:
            sizes = [(1.0 - part if not stress else 0.0, 172, 375), (part if not stress else 1.0, 425, 1150)]
    cells = regions * reads * haps * sum(p * r * h for p, r, h in sizes)
    read_bytes = regions * reads * sum(p * r for p, r, _ in sizes)
    hap_bytes = regions * haps * sum(p * h for p, _, h in sizes)
    pairs = regions * reads * haps
    if kind == "read_prep":
        # Bases read twice, three quality planes read and written, two planes written.
        return {"bytes": 10 * read_bytes, "flops": 0}
    if kind == "train":
        return {"bytes": read_bytes * (1 + 2 * 4 * 4) + hap_bytes + 16 * pairs, "flops": 36 * cells}
    return {"bytes": 5 * read_bytes + hap_bytes + 8 * pairs, "flops": 12 * cells}


# ---- the same in 64 bits, by plain torch -----------------------------------------------------------


def _match_to_match():
    """MM by the two gap-open qualities: 1 - e(ins) - e(del) through the model's table of log sums (step
    1e-4, differences of 8 and more dropped)."""
    q = np.arange(128) * -0.1
    hi, diff = np.maximum(q[:, None], q[None]), np.abs(q[:, None] - q[None])
    step = np.floor(diff * 1e4 + 0.5) * 1e-4
    s = np.minimum(1.0, 10.0 ** (hi + np.where(diff < 8.0, np.log10(1.0 + 10.0 ** -step), 0.0)))
    return torch.from_numpy(np.exp(np.log1p(-np.minimum(s, 1 - 1e-16)))).to(DEV)


def _groups(R, H, elements):
    """Pairs in groups of near lengths, each of at most about `elements` (row, pair) places."""
    order = torch.argsort(R // 16 * 100000 + H, stable=True)
    at, n = 0, len(order)
    Rs = R[order].cpu().numpy()
    while at < n:
        take = max(1, int(elements // (int(Rs[min(n - 1, at + 1)]) + 17)))
        yield order[at:at + take]
        at += take


class _Group:
    """Bases and row parameters of a group of pairs: rows x pairs, haplotypes end first."""

    def __init__(self, rd, hp, r, h, rows):
        self.R, self.H = rd["len"][r].long(), hp["len"][h].long()
        self.n, self.m, self.p = int(self.R.max()), int(self.H.max()), len(r)
        i = torch.arange(self.n, device=DEV)[:, None]
        self.at = (rd["off"][r][None] + i).clamp_max(len(rd["bases"]) - 1)
        self.on = i < self.R[None]
        j = torch.arange(self.m, device=DEV).flip(0)[:, None]
        self.hat = (hp["off"][h][None] + j).clamp_max(len(hp["bases"]) - 1)
        self.hon = j < self.H[None]
        self.x = rd["bases"][self.at]
        self.y = torch.where(self.hon, hp["bases"][self.hat], torch.zeros((), dtype=torch.uint8, device=DEV))
        for k, v in rows(self.at).items():
            setattr(self, k, v)

    def rows_of(self, d):
        """Rows (from 1) and the haplotype slice of anti-diagonal d = row + column."""
        lo, hi = max(1, d - self.m), min(self.n, d - 1)
        return lo, hi + 1, self.m - d + lo, self.m - d + hi + 1


def _zeros(g, k):
    return [torch.zeros(g.n + 1, g.p, dtype=torch.float64, device=DEV) for _ in range(k)]


def _forward(g, keep=None):
    """Scaled last-row sums of a group by anti-diagonals; `keep` takes each diagonal's M, I, D, sum before
    the prior and match mask."""
    d0 = 2.0 ** 1020 / g.H.double()
    M, S, I, D = _zeros(g, 3), _zeros(g, 3), _zeros(g, 2), _zeros(g, 2)
    for s in S:
        s[0] = d0
    acc = torch.zeros(g.p, dtype=torch.float64, device=DEV)
    for d in range(2, g.n + g.m + 1):
        lo, hi, a, b = g.rows_of(d)
        up, own, q = slice(lo - 1, hi - 1), slice(lo, hi), slice(lo - 1, hi - 1)
        M0, M1, M2, S0, S2 = M[d % 3], M[(d - 1) % 3], M[(d - 2) % 3], S[d % 3], S[(d - 2) % 3]
        I0, I1, D0, D1 = I[d % 2], I[(d - 1) % 2], D[d % 2], D[(d - 1) % 2]
        hit = g.x[q] == g.y[a:b]
        pre = (M2[up] * g.MM[q]).addcmul_(S2[up], g.GM[q])
        torch.mul(pre, torch.where(hit, g.pm[q], g.px[q]), out=M0[own])
        torch.mul(M1[up], g.MI[q], out=I0[own]).addcmul_(I1[up], g.II[q])
        torch.mul(M1[own], g.MD[q], out=D0[own]).addcmul_(D1[own], g.II[q])
        torch.add(I0[own], D0[own], out=S0[own])
        if keep is not None:
            keep.append((M0[own].clone(), I0[own].clone(), D0[own].clone(), pre, hit))
        c = d - g.R
        last = (M0.gather(0, g.R[None]) + I0.gather(0, g.R[None]))[0]
        acc += torch.where((c >= 1) & (c <= g.H), last, torch.zeros_like(last))
    return acc


def _planes(b, names):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    rd = {"bases": t(b.read_bases), "off": t(b.read_off), "len": t(b.read_len)}
    rd.update({k: t(getattr(b, v)).long() for k, v in names.items()})
    return rd, {"bases": t(b.hap_bases), "off": t(b.hap_off), "len": t(b.hap_len)}, t(b.pair_read).long(), t(b.pair_hap).long()


def _qualities(rd):
    """Row parameters from byte qualities."""
    err = 10.0 ** (torch.arange(256, dtype=torch.float64, device=DEV) / -10.0)
    mm = _match_to_match()

    def rows(at):
        q, i, d, c = (rd[k][at] for k in ("q", "i", "d", "c"))
        return {"MM": mm[i, d], "MI": err[i], "MD": err[d], "II": err[c], "GM": 1.0 - err[c], "pm": 1.0 - err[q],
                "px": err[q] / 3.0}
    return rows


_BYTES = {"q": "read_quals", "i": "read_ins", "d": "read_del", "c": "read_gcp"}


def _exact_likelihoods(b):
    rd, hp, pr, ph = _planes(b, _BYTES)
    out = torch.empty(len(pr), dtype=torch.float64, device=DEV)
    for k in _groups(rd["len"][pr].long(), hp["len"][ph].long(), 4e6):
        out[k] = torch.log10(_forward(_Group(rd, hp, pr[k], ph[k], _qualities(rd)))) - 1020 * math.log10(2.0)
    return out.cpu().numpy()


def _exact_gradients(b, q):
    """log10 likelihoods and the sums over pairs of their derivatives by each base's four Phred values."""
    rd, hp, pr, ph = _planes(b, {})
    q = {k: torch.from_numpy(v).to(DEV).double() for k, v in q.items()}
    e = {k: 10.0 ** (-v / 10.0) for k, v in q.items()}

    def rows(at):
        eb, ei, ed, ec = (e[k][at] for k in ("qb", "qi", "qd", "qc"))
        return {"MM": 1.0 - ei - ed, "MI": ei, "MD": ed, "II": ec, "GM": 1.0 - ec, "pm": 1.0 - eb, "px": eb / 3.0}

    out = torch.empty(len(pr), dtype=torch.float64, device=DEV)
    grad = {k: torch.zeros(len(rd["bases"]), dtype=torch.float64, device=DEV) for k in q}
    for k in _groups(rd["len"][pr].long(), hp["len"][ph].long(), 1.5e6):
        g, kept = _Group(rd, hp, pr[k], ph[k], rows), []
        total = _forward(g, kept)
        out[k] = torch.log10(total) - 1020 * math.log10(2.0)
        # Rows from 1 as before, with a row of zeros after the last one; adjoints of a unit last-row sum.
        X, GI, GD = ([torch.zeros(g.n + 2, g.p, dtype=torch.float64, device=DEV) for _ in range(n)] for n in (3, 2, 2))
        s = {n: torch.zeros(g.n + 1, g.p, dtype=torch.float64, device=DEV) for n in ("MM", "GM", "MI", "II", "MD", "DD", "E")}
        d0 = 2.0 ** 1020 / g.H.double()
        row = torch.arange(g.n + 1, device=DEV)[:, None]
        for d in range(g.n + g.m, 1, -1):
            lo, hi, _, _ = g.rows_of(d)
            own, q1, below = slice(lo, hi), slice(lo - 1, hi - 1), slice(lo + 1, hi + 1)

            def par(v):  # parameters of the row below, none below the last row
                w = v[lo:hi]
                return w if len(w) == hi - lo else torch.cat([w, torch.zeros(1, g.p, dtype=w.dtype, device=DEV)])

            m, i, dd, pre, hit = kept[d - 2]
            x2, gi1, gd1 = X[(d + 2) % 3][below], GI[(d + 1) % 2][below], GD[(d + 1) % 2][own]
            c = d - row[own]
            seed = ((row[own] == g.R[None]) & (c >= 1) & (c <= g.H[None])).double()
            gs = par(g.GM) * x2
            gm = (par(g.MM) * x2).addcmul_(par(g.MI), gi1).addcmul_(g.MD[q1], gd1).add_(seed)
            gi = torch.addcmul(gs, par(g.II), gi1).add_(seed)
            gd = torch.addcmul(gs, g.II[q1], gd1)
            x = gm * torch.where(hit, g.pm[q1], g.px[q1])
            for buf, v in ((X[d % 3], x), (GI[d % 2], gi), (GD[d % 2], gd)):
                buf[own] = v
            s["E"][own].add_(gm * pre * (hit.double() * (-4.0 / 3.0) + 1.0 / 3.0))
            # Products with the values these adjoints came from: rows above on diagonals d-1 and d-2.
            if d - 2 >= 2:
                l2, h2, _, _ = g.rows_of(d - 2)
                M, I, D = kept[d - 4][:3]
                a, z = max(lo, l2 + 1), min(hi, h2 + 1)
                s["MM"][a:z].addcmul_(x[a - lo:z - lo], M[a - 1 - l2:z - 1 - l2])
                s["GM"][a:z].addcmul_(x[a - lo:z - lo], I[a - 1 - l2:z - 1 - l2] + D[a - 1 - l2:z - 1 - l2])
            if lo == 1:
                s["GM"][1] += x[0] * d0
            if d - 1 >= 2:
                l1, h1, _, _ = g.rows_of(d - 1)
                M, I, D = kept[d - 3][:3]
                a, z = max(lo, l1 + 1), min(hi, h1 + 1)
                s["MI"][a:z].addcmul_(gi[a - lo:z - lo], M[a - 1 - l1:z - 1 - l1])
                s["II"][a:z].addcmul_(gi[a - lo:z - lo], I[a - 1 - l1:z - 1 - l1])
                a, z = max(lo, l1), min(hi, h1)
                s["MD"][a:z].addcmul_(gd[a - lo:z - lo], M[a - l1:z - l1])
                s["DD"][a:z].addcmul_(gd[a - lo:z - lo], D[a - l1:z - l1])
        norm = (1.0 / total)[None] / math.log(10.0) * (-math.log(10.0) / 10.0)
        at = g.at[g.on]
        for name, v in (("qb", s["E"]), ("qi", s["MI"] - s["MM"]), ("qd", s["MD"] - s["MM"]),
                        ("qc", s["II"] + s["DD"] - s["GM"])):
            grad[name].index_add_(0, at, (v[1:] * norm * e[name][g.at])[g.on])
    return {"log10_likelihood": out, **grad}


def _exact_pd(b, pd):
    """The partially determined model: branch values bM, bI, bD beside M, I, D; E is what a cell hands on,
    max(branch, value) where a deletion ends and the value elsewhere."""
    rd, hp, pr, ph = _planes(b, _BYTES)
    first, later, alt = np.zeros(len(pd), bool), np.zeros(len(pd), bool), np.where(pd & SNP, pd & 0x78, 0)
    for o, n in zip(b.hap_off.tolist(), b.hap_len.tolist()):
        state = 0  # inside a deletion: 1, just after one: 2; a row begins as the one before ended
        for inside in (first, later):
            for j in range(o, o + n):
                inside[j] = state == 1
                state = 0 if state == 2 else state
                state = 1 if pd[j] & DEL_START else state
                state = 2 if pd[j] & DEL_END else state
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)  # noqa: E731
    first, later, ends, alt = t(first), t(later), t((pd & DEL_END) != 0), t(alt.astype(np.uint8))
    bit = torch.zeros(256, dtype=torch.uint8, device=DEV)
    for k, c in enumerate(b"ACGT"):
        bit[c] = 8 << k
    g = _Group(rd, hp, pr, ph, _qualities(rd))
    at_hap = lambda v: torch.where(g.hon, v[g.hat], torch.zeros((), dtype=v.dtype, device=DEV))  # noqa: E731
    first, later, ends, alt, xbit = at_hap(first), at_hap(later), at_hap(ends), at_hap(alt), bit[g.x.long()]
    M, I, D = _zeros(g, 3), _zeros(g, 3), _zeros(g, 3)
    B = [_zeros(g, 2) for _ in range(3)]
    for v in D:
        v[0] = 2.0 ** 1020 / g.H.double()
    acc = torch.zeros(g.p, dtype=torch.float64, device=DEV)
    last = torch.zeros(g.n + 1, g.p, dtype=torch.float64, device=DEV)
    for d in range(2, g.n + g.m + 1):
        lo, hi, a, z = g.rows_of(d)
        up, own, q = slice(lo - 1, hi - 1), slice(lo, hi), slice(lo - 1, hi - 1)
        (M0, M1, M2), (I0, I1, I2), (D0, D1, D2) = ((v[d % 3], v[(d - 1) % 3], v[(d - 2) % 3]) for v in (M, I, D))
        hit = (g.x[q] == g.y[a:z]) | ((xbit[q] & alt[a:z]) != 0)
        m = (M2[up] * g.MM[q] + (I2[up] + D2[up]) * g.GM[q]) * torch.where(hit, g.pm[q], g.px[q])
        i = M1[up] * g.MI[q] + I1[up] * g.II[q]
        dd = M1[own] * g.MD[q] + D1[own] * g.II[q]
        inside = later[a:z].clone()
        if lo == 1:
            inside[0] = first[a]
        for (b0, b1), prev, now, value in zip(((v[d % 2], v[(d - 1) % 2]) for v in B), (M1, I1, D1), (M0, I0, D0), (m, i, dd)):
            b0[own] = torch.where(inside, b1[own], prev[own])
            now[own] = torch.where(ends[a:z], torch.maximum(b0[own], value), value)
        last[own] = m + i
        c = d - g.R
        v = last.gather(0, g.R[None])[0]
        acc += torch.where((c >= 1) & (c <= g.H), v, torch.zeros_like(v))
    return (torch.log10(acc) - 1020 * math.log10(2.0)).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("region", "batch", "chunk"):
        return _exact_likelihoods(_regions(case, seed))
    if kind == "train":
        b = _regions(case, seed)
        return _exact_gradients(b, _penalties(b, seed))
    if kind == "pd_region":
        b = _regions(case, seed)
        return _exact_pd(b, _pd_bytes(b, seed))
    if kind == "post":
        lk, _, _, lens = _matrix(case, seed)
        best = lk[:, 1:].max(1, keepdim=True).values  # allele 0 is the reference
        threshold = torch.ceil(lens.double() * 0.02).clamp_max(2.0) * -4.0
        return {"likelihoods": torch.maximum(lk, best - 4.5), "keep": None,
                "threshold": None if case["dynamic"] else threshold}
    return None
