"""Performance cases: the work that a program using libewfa has it do.

A case is a batch of synthetic sequence pairs (ewfa.Workload), the entry point
that aligns it and that entry point's options:

  entry   device  ewfa_align_device on inputs resident in device memory
          ascii   ewfa_pack_ascii on ASCII in device memory, then ewfa_align_device
          host    ewfa_align_host on pinned host buffers, PCIe included
          served  jobs submitted to the job server together and waited for
  n       pairs
  kind    0: fixed length `hi`, error `err_hi` split equally between
          substitutions, insertions and deletions; 1: log-uniform lengths
          lo..hi; 2: uniform lengths lo..hi with insertion and deletion runs.
          Kinds 1 and 2 draw each pair's error from err_lo..err_hi.
  cap     ewfa_opts_t.max_distance (0: exact; 64: the reference's own limit)
  policy  "c2" / "": the tuned policy of 1,000 bp reads, or the built-in table
  room    CIGAR bytes per pair (0: room for the case's error rate and length)

Every output is whole: each pair's result record and the CIGAR buffer.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ewfa-gpu_amd"))
import ewfa  # noqa: E402

POLICIES = {"": None, "c2": os.path.join(ROOT, "ewfa-gpu_amd", "policy", "c2_1000bp_5pct.policy")}
JOBS = 48          # jobs a served case is cut into
THREADS = 8


def case(name, entry, n, kind, lo, hi, err_lo, err_hi, cap=0, policy="", room=0):
    c = dict(entry=entry, n=n, kind=kind, lo=lo, hi=hi, err_lo=err_lo, err_hi=err_hi, cap=cap, policy=policy, room=room)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one pair as it comes up in a program: all launch and host latency
        case("one_pair", "device", 1, 0, 150, 150, 0.02, 0.02),
        # an interactive call: the reads of one locus, of mixed length
        case("few_pairs", "device", 60, 1, 100, 2_000, 0.01, 0.10),
        # a sequencer's short reads (150 bp, 2%), a small batch
        case("short_reads", "device", 10_000, 0, 150, 150, 0.02, 0.02),
        # the headline workload: a million 1,000 bp reads at 5%, with the
        # policy tuned for them and the reference's CIGAR stride
        case("reads_1kb", "device", 1_000_000, 0, 1_000, 1_000, 0.05, 0.05, policy="c2", room=1_004),
        # mixed lengths and error rates in one launch
        case("mixed", "device", 500_000, 1, 100, 10_000, 0.01, 0.10),
        # long noisy reads with insertion and deletion runs
        case("long_reads", "device", 20_000, 2, 10_000, 50_000, 0.10, 0.15),
        # a batch of a few kbp at a high error rate, odd lengths
        case("noisy_3to7kb", "device", 15_001, 2, 2_999, 7_013, 0.08, 0.15),
        # accurate long reads: a few hundred pairs, few edits, long matches
        case("accurate_15kb", "device", 400, 2, 10_000, 20_000, 0.002, 0.02),
        # the reference's own distance limit (pairs beyond 64 come back capped)
        case("capped", "device", 200_000, 1, 300, 1_200, 0.01, 0.08, cap=64),
        # ASCII reads already on the device, packed there and aligned
        case("ascii_600", "ascii", 100_000, 1, 500, 700, 0.01, 0.06),
        # host buffers in and out in one call
        case("host_250", "host", 200_000, 1, 150, 350, 0.005, 0.04),
        # a burst of jobs into the job server
        case("served", "served", 60_000, 1, 100, 5_000, 0.01, 0.10),
    ]


def draw(rng):
    """One more case: an entry point, a length range, an error range, and a
    count between one pair and what keeps it below the largest listed cases."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    entry = rng.choice(["device"] * 6 + ["ascii", "host", "served"])
    kind = rng.choice([0, 1, 2])
    hi = log(100, 30_000 if entry == "device" else 4_000)
    lo = hi if kind == 0 else max(60, int(hi / rng.choice([1.3, 2, 5])))
    err_hi = round(rng.uniform(0.01, 0.15), 3)
    err_lo = err_hi if kind == 0 else round(err_hi * rng.uniform(0.1, 0.9), 4)
    cap = 64 if entry == "device" and rng.random() < 0.2 else 0
    # bounded by bases (a gigabase), by wavefront cells and by PCIe or host work
    most = min(400_000_000 // hi, int(1.0e11 / (hi * err_hi + 30) ** 2))
    if entry != "device":
        most = min(most, 40_000_000 // hi)
    least = JOBS * 4 if entry == "served" else 1
    n = max(least, log(least, max(most, least + 1)))
    return case("", entry, n, kind, lo, hi, err_lo, err_hi, cap=cap)


def spec(c, seed):
    return ewfa.synth_spec(kind=c["kind"], seed=seed, len=c["hi"], err=c["err_hi"], len_lo=c["lo"], len_hi=c["hi"],
                           err_lo=c["err_lo"], err_hi=c["err_hi"])


def room(c):
    """CIGAR bytes per pair: at D edits a stream holds at most 2D+1 bytes and
    one more for every 127 matches."""
    return c["room"] or (2 * math.ceil(c["err_hi"] * c["hi"]) + c["hi"] // 127 + 64) // 4 * 4


class State:
    """What the program holds: its context or server, inputs and outputs."""
    handle = None

    def __del__(self):
        if self.handle is not None:
            self.handle.close()


def on_device(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1)).cuda()


def pinned(nbytes):
    """Zeroed pinned host memory (the array keeps its tensor alive)."""
    return torch.zeros(nbytes, dtype=torch.uint8, pin_memory=True).numpy()


def prepare(c, seed):
    s = State()
    s.entry, s.n = c["entry"], c["n"]
    w = ewfa.Workload(spec(c, seed), c["n"], cigar_cap=room(c), threads=THREADS)
    s.max_len = w.max_len
    opts = dict(max_distance=c["cap"], policy_path=POLICIES[c["policy"]])
    if s.entry in ("host", "served"):
        s.words = pinned(w.words.nbytes).view(np.uint64)
        s.words[:] = w.words
        s.pairs = w.pairs[:w.n].copy()
        s.results = pinned(w.n * ewfa.RESULT_DTYPE.itemsize).view(ewfa.RESULT_DTYPE)
        s.cigars = pinned(w.cigar_bytes).view(np.int8)
        s.cigar_bytes = w.cigar_bytes
        if s.entry == "host":
            s.handle = ewfa.Context(**opts)
        else:
            s.handle = ewfa.Server(arena_bytes=1 << 30, max_batch_cigar_bytes=64 << 20, **opts)
            # jobs of unequal size, each a slice of the buffers
            cuts = np.random.default_rng(seed).choice(np.arange(1, w.n), JOBS - 1, replace=False)
            cuts = [0] + sorted(int(x) for x in cuts) + [w.n]
            s.jobs = []
            for a, b in zip(cuts, cuts[1:]):
                words, pairs, cigar_bytes, _, c0 = ewfa.slice_pairs(s.words, s.pairs, a, b)
                s.jobs.append((words, pairs, b - a, cigar_bytes, s.results[a:b], s.cigars[c0:c0 + cigar_bytes]))
        return s
    pairs = w.pairs[:w.n].copy()
    if s.entry == "ascii":
        # fixed-stride ASCII slabs, patterns and texts, packed to fixed-stride words
        s.stride = w.stride
        s.wstride = int(ewfa.lib().ewfa_packed_words(w.stride))
        s.pat, s.txt = on_device(w.pat), on_device(w.txt)
        s.plen, s.tlen = on_device(w.plen), on_device(w.tlen)
        s.words = torch.zeros(2 * w.n * s.wstride * 8, dtype=torch.uint8, device="cuda")
        pairs["pattern_off"] = np.arange(w.n, dtype=np.uint64) * np.uint64(s.wstride)
        pairs["text_off"] = np.arange(w.n, 2 * w.n, dtype=np.uint64) * np.uint64(s.wstride)
    else:
        s.words = on_device(w.words)
    s.pairs = on_device(pairs)
    s.results = torch.zeros((w.n, 4), dtype=torch.int32, device="cuda")
    s.cigars = torch.zeros(w.cigar_bytes, dtype=torch.int8, device="cuda")
    s.handle = ewfa.Context(**opts)
    return s


def run(s):
    if s.entry == "host":
        s.handle.align_host(s.words, s.pairs, s.n, s.cigar_bytes, s.results, s.cigars)
    elif s.entry == "served":
        for job in [s.handle.submit(*j) for j in s.jobs]:
            job.wait()
    else:
        if s.entry == "ascii":
            half = s.n * s.wstride * 8
            for seqs, lens, to in ((s.pat, s.plen, 0), (s.txt, s.tlen, half)):
                ewfa._check(ewfa.lib().ewfa_pack_ascii(seqs.data_ptr(), s.stride, lens.data_ptr(), s.n,
                                                       s.words.data_ptr() + to, s.wstride, None))
        s.handle.align_device(s.words.data_ptr(), s.pairs.data_ptr(), s.n, s.max_len, s.results.data_ptr(),
                              s.cigars.data_ptr())
    if s.entry in ("host", "served"):
        return {"results": s.results.view(np.int32), "cigars": s.cigars}
    return {"results": s.results, "cigars": s.cigars}


def work(c):
    """Sequences, descriptors, results and streams, each once."""
    lo, hi, n = c["lo"], c["hi"], c["n"]
    mean = (hi - lo) / math.log(hi / lo) if c["kind"] == 1 and hi > lo else (lo + hi) / 2
    err = (c["err_lo"] + c["err_hi"]) / 2
    bases = 2 * mean * (1.0 if c["entry"] == "ascii" else 0.25)
    stream = min(2 * err * mean + mean / 127 + 1, room(c))
    return {"bytes": n * (bases + 40 + 16 + stream), "flops": 0}


def exact(c, seed):
    """Outputs are whole numbers and bytes: there is no value to round."""
    return None
