"""The bit-parallel pass as large calls use it, and what decides on it.

Lists of the mid-length buckets take its instance for all classes, calls of
32,768 pairs and more its narrowest groups of lanes; few long pairs take one of
two passes by a sample, also where a recorded graph is replayed over other
inputs.  Outputs are the oracle's, and where a list's way matters the call is
timed beside one with a distance cap beyond any distance, which only has the
wavefront.
"""
import ctypes

import numpy as np
import pytest

import ewfa
import oracle_py as orc
from test_gpu_bitpar import POLICY, case_pairs, mutate
from test_gpu_bound import check, policy_file
from test_gpu_limits import BASES, OnDevice, fill_pairs, median_us
from test_gpu_stress import oracle_streams

pytestmark = pytest.mark.gpu


def pool_case(rng, count, pairs):
    """`count` pairs drawn from a few with their oracle outputs."""
    P, T = [p for p, _ in pairs], [t for _, t in pairs]
    d, st = oracle_streams(P, T)
    take = rng.permutation(np.resize(np.arange(len(P)), count))
    case = OnDevice(*ewfa.from_sequences([P[i] for i in take], [T[i] for i in take]))
    return case, [d[i] for i in take], [st[i] for i in take]


def both_ways(case, d, st, label):
    """The call, checked, and its time over that of the wavefront alone."""
    took = []
    for cap in (0, 1 << 20):
        with ewfa.Context(max_distance=cap) as ctx:
            case.dc.fill_zero()
            took.append(median_us(lambda: case.align(ctx), 3))
        case.check(d, st, (label, cap))
    return took[0] / took[1]


@pytest.mark.parametrize("count,lo,hi,rate", [(2600, 4600, 4990, 0.14), (1500, 9000, 10400, 0.14),
                                              (33_000, 2600, 4900, 0.13)])
def test_mid_length_lists_of_many_edits(count, lo, hi, rate):
    """Buckets of 512 and 1,024 levels, whose lists a sample sends the
    bit-parallel way: one kernel for all classes; from 32,768 pairs on groups of
    8 and 16 lanes of up to four words."""
    print(f"case mid {count} pairs of {lo}..{hi} at {rate}", flush=True)
    rng = np.random.default_rng(count)
    pool = []
    for i in range(60):
        p = rng.choice(BASES, int(rng.integers(lo, hi))).tobytes()
        # some within the wavefront's budget, some with gaps that lose the bound
        pool.append((p, mutate(rng, p, rate if i % 5 else 0.06, 60 if i % 20 == 3 else 1)))
    pool = [(p, t[:hi]) for p, t in pool]
    case, d, st = pool_case(rng, count, pool)
    assert both_ways(case, d, st, "mid") < 0.75


@pytest.mark.parametrize("name", ["classes", "gaps", "repeats"])
def test_groups_of_lanes_of_large_calls(tmp_path, name):
    """Every class of bands in a call of 33,000 pairs: 8, 16, 32 and 64 lanes a
    pair with two to four words each, as they narrow."""
    print(f"case groups {name}", flush=True)
    P, T, rng = case_pairs(name)
    if name == "classes":  # several pairs a wave, of unequal lengths
        for n in (700, 1200, 1700, 2300, 3100, 4100, 5300, 7300):
            for _ in range(9):
                p = rng.choice(BASES, int(n * rng.uniform(0.9, 1.0))).tobytes()
                P.append(p)
                T.append(mutate(rng, p, 0.15))
    d, st = oracle_streams(P, T)
    fp, ft, fd, fst = fill_pairs(33_000 - len(P))
    case = OnDevice(*ewfa.from_sequences(P + fp, T + ft))
    with ewfa.Context(policy_path=policy_file(tmp_path, "wide", POLICY)) as ctx:
        for _ in range(2):
            case.dc.fill_zero()
            case.align(ctx).check(list(d) + fd, list(st) + fst, name)


def test_replays_of_a_sampled_choice():
    """300 pairs over several buckets, recorded once: the replays see inputs of
    few edits and of many in turn, and the sample picks another pass each time."""
    print("case sampled replays", flush=True)
    rng = np.random.default_rng(300)
    base = [rng.choice(BASES, int(n)).tobytes() for n in rng.integers(300, 14_000, 20)] + [rng.choice(BASES, 15_500).tobytes()]
    sets = []
    for rate in (0.004, 0.1):
        pairs = [(p, (mutate(rng, p, rate) + p)[:len(p)]) for p in base]  # of one length: the descriptors stay
        P, T = [p for p, _ in pairs], [t for _, t in pairs]
        d, st = oracle_streams(P, T)
        take = [i % len(P) for i in range(300)]
        sets.append((ewfa.from_sequences([P[i] for i in take], [T[i] for i in take], cigar_cap=8192),
                     [d[i] for i in take], [st[i] for i in take]))
    case = OnDevice(*sets[0][0])
    with ewfa.Context() as ctx:
        for k in (0, 0, 1, 1, 0, 1, 0):
            (words, pairs, cb, ml), d, st = sets[k]
            assert ml == case.max_len and np.array_equal(pairs, case.pairs)
            case.dw.upload(words)
            case.dc.fill_zero()
            ewfa.synchronize()
            case.align(ctx).check(d, st, k)


@pytest.mark.parametrize("named", [True, False])
def test_a_call_waits_for_what_its_stream_still_has_to_do(named):
    """Inputs still on their way when the call is made: on the stream it is
    given, and on a blocking stream beside the null stream."""
    hip = ctypes.CDLL("libamdhip64.so")
    print(f"case late inputs, {'given' if named else 'null'} stream", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=4, len_lo=100, len_hi=3000, err_lo=0.01, err_hi=0.05), 400)
    ok, d, sl, st = orc.batch_workload(w)
    case = OnDevice(w.words, w.pairs[:w.n].copy(), w.cigar_bytes, w.max_len)
    right, wrong = ewfa.DeviceBuffer.from_array(w.words), ewfa.DeviceBuffer.from_array(w.words ^ np.uint64(0x5555))
    big = [ewfa.DeviceBuffer(1 << 30) for _ in range(2)]
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(stream), ctypes.c_uint(1 if named else 0)) == 0

    def queue(dst, src, nbytes):
        assert hip.hipMemcpyAsync(ctypes.c_void_p(dst.ptr), ctypes.c_void_p(src.ptr), ctypes.c_size_t(nbytes), 3, stream) == 0

    with ewfa.Context() as ctx:
        for _ in range(3):
            ewfa.synchronize()
            queue(case.dw, wrong, w.words.nbytes)
            for _ in range(10):  # some milliseconds
                queue(big[0], big[1], 1 << 30)
            queue(case.dw, right, w.words.nbytes)
            ctx.align_device(case.dw.ptr, case.dp.ptr, case.n, case.max_len, case.dr.ptr, case.dc.ptr,
                             stream.value if named else None)
            case.check(d, st, named)
    ewfa.synchronize()
    assert hip.hipStreamDestroy(stream) == 0


def test_pairs_beyond_the_allocation_free_calls_levels():
    """What its last pass defers is marked, the rest is aligned."""
    print("case allocation-free, too distant", flush=True)
    fp, ft, fd, fst = fill_pairs(50)
    case = OnDevice(*ewfa.from_sequences([b"A" * 60_000] + fp, [b"C" * 60_000] + ft))
    with ewfa.Context() as ctx:
        ctx.align_device_noalloc(case.dw.ptr, case.dp.ptr, case.n, case.max_len, case.dr.ptr, case.dc.ptr, None)
    res, cig = case.dr.download(ewfa.RESULT_DTYPE, case.n), case.dc.download(np.int8)
    assert int(res[0]["status"]) == ewfa.PAIR_TOO_DISTANT
    check(res[1:], case.pairs[1:], cig, fd, fst, "beside")
