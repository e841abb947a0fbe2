"""The bit-parallel pass (bitpar.hip) against the oracle, bit for bit.

A policy whose only bucket has a budget above 2,048 levels weighs the pass for
every call of more than 1,024 pairs: here mostly short ones, so that the oracle
stays quick, around the pairs of the case.  From 8,192 pairs on the distance
bounds come from the lane-per-pair search, and from 32,768 on the groups of lanes
are at their narrowest.
"""
import numpy as np
import pytest

import ewfa
import oracle_py as orc
from test_gpu_bound import check, policy_file
from test_gpu_stress import oracle_streams, stress_pairs

pytestmark = pytest.mark.gpu

POLICY = "4000000000 8 1048576 0 1\n"
BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


def mutate(rng, p, rate, gap=1):
    """p with `rate` of its bases edited, a third of the edits each kind,
    insertions and deletions in runs of up to `gap`."""
    out, i = [], 0
    while i < len(p):
        if rng.random() < rate:
            kind, run = rng.integers(3), int(rng.integers(1, gap + 1))
            if kind == 0:
                out.append(int(rng.choice(BASES)))
                i += 1
            elif kind == 1:
                out.extend(rng.choice(BASES, run).tolist())
            else:
                i += run
        else:
            out.append(p[i])
            i += 1
    return bytes(out)


def case_pairs(name):
    rng = np.random.default_rng(sum(map(ord, name)))
    rand = lambda n: rng.choice(BASES, n).tobytes()  # noqa: E731
    P, T = [], []
    if name == "edges":  # either side of whole words and of whole 32-column blocks
        for n in (1, 2, 31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 255, 256, 257, 511, 512, 513):
            for d in (-33, -32, -1, 0, 1, 31, 32, 33):
                if n + d > 0:
                    p = rand(n)
                    P.append(p)
                    T.append((mutate(rng, p, 0.15) + rand(64))[:n + d])
        P += [b"A" * 200, b"A" * 64, rand(300), rand(300), b"", rand(40), b"A" * 33]
        T += [b"C" * 200, b"A" * 96, rand(300), rand(260), rand(40), b"", b"T" * 31]
    elif name == "classes":  # distances over every band width, to the widest
        for n, rate in ((900, .15), (1400, .16), (2600, .16), (3500, .15), (5000, .15), (6600, .15), (8000, .15),
                        (10500, .15), (14000, .15), (21000, .15), (29000, .15), (42000, .15), (52000, .16)):
            for _ in range(2):
                p = rand(n)
                P.append(p)
                T.append(mutate(rng, p, rate))
    elif name == "gaps":  # the bound search can lose these paths
        for n in (400, 1500, 4000, 9000):
            for gap in (8, 40, 90):
                p = rand(n)
                P.append(p)
                T.append(mutate(rng, p, 0.02, gap))
        for extra in (40, 200, 700):
            p = rand(2000)
            P += [p, p + rand(extra), rand(extra) + p]
            T += [p[:900] + rand(extra) + p[900:], p, p]
    else:
        P, T = stress_pairs(77, 500)
    return P, T, rng


@pytest.mark.parametrize("name,count", [("edges", 2100), ("classes", 2100), ("gaps", 8300), ("repeats", 2100),
                                        ("edges", 33000)])
def test_equals_the_oracle(tmp_path, name, count):
    P, T, rng = case_pairs(name)
    pool = []
    for _ in range(400):
        p = rng.choice(BASES, int(rng.integers(40, 420))).tobytes()
        pool.append((p, mutate(rng, p, float(rng.uniform(0.05, 0.18)))))
    fill = [pool[i % len(pool)] for i in range(count - len(P))]
    P, T = P + [p for p, _ in fill], T + [t for _, t in fill]
    print(f"case bit-parallel {name}: {len(P)} pairs", flush=True)
    d, st = oracle_streams(P, T)
    words, pairs, cb, ml = ewfa.from_sequences(P, T)
    with ewfa.Context(policy_path=policy_file(tmp_path, "wide", POLICY)) as ctx:
        dw, dp = ewfa.DeviceBuffer.from_array(words), ewfa.DeviceBuffer.from_array(pairs)
        dr, dc = ewfa.DeviceBuffer(len(P) * 16), ewfa.DeviceBuffer(cb)
        for _ in range(2):  # and a replay
            dc.fill_zero()
            ctx.align_device(dw.ptr, dp.ptr, len(P), ml, dr.ptr, dc.ptr)
            check(dr.download(ewfa.RESULT_DTYPE, len(P)), pairs, dc.download(np.int8), d, st, name)


def test_streams_end_at_their_region(tmp_path):
    """Streams longer than their region: cut at it, whole length reported; one
    whose region is not in whole dwords: refused with its distance."""
    print("case bit-parallel overflow: 2100 pairs, 16-byte regions", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=1, seed=9, len_lo=40, len_hi=300, err_lo=0.02, err_hi=0.2), 2100, cigar_cap=16)
    ok, d, sl, st = orc.batch_workload(w)
    pairs = w.pairs[:w.n].copy()
    pairs["cigar_off"][::50] += 1
    dw, dp = ewfa.DeviceBuffer.from_array(w.words), ewfa.DeviceBuffer.from_array(pairs)
    dr, dc = ewfa.DeviceBuffer(w.n * 16), ewfa.DeviceBuffer(w.cigar_bytes + 4)
    dc.upload(np.full(w.cigar_bytes + 4, 7, dtype=np.int8))
    with ewfa.Context(policy_path=policy_file(tmp_path, "wide", POLICY)) as ctx:
        ctx.align_device(dw.ptr, dp.ptr, w.n, w.max_len, dr.ptr, dc.ptr)
    res, cig = dr.download(ewfa.RESULT_DTYPE, w.n), dc.download(np.int8)
    for i in range(w.n):
        assert int(res[i]["distance"]) == int(d[i]), i
        region = cig[16 * i: 16 * i + 16]
        if i % 50 == 0:
            assert int(res[i]["status"]) == ewfa.PAIR_BADARG and (region == 7).all(), i
            continue
        full = len(st[i])
        assert int(res[i]["cigar_len"]) == full, i
        assert int(res[i]["status"]) == (ewfa.PAIR_OVERFLOW if full > 16 else ewfa.PAIR_OK), i
        # whole dwords up to the terminator's, the rest untouched
        end = min((full & ~3) + 4, 16)
        expect = np.full(16, 7, dtype=np.int8)
        expect[:end] = 0
        expect[:min(full, 16)] = st[i][:16]
        assert np.array_equal(region, expect), i


@pytest.mark.parametrize("stride", [1, 31, 32, 33, 65, 735])
def test_pack_strides_and_last_words(stride):
    """ewfa_pack_ascii at strides and lengths around whole words, the last
    sequence ending where the buffer does."""
    print(f"case pack stride {stride}", flush=True)
    rng = np.random.default_rng(stride)
    n = 70
    lens = rng.integers(0, stride + 1, n).astype(np.uint32)
    lens[:4] = [0, stride, max(stride - 1, 0), min(stride, 32)]
    text = rng.choice(np.frombuffer(b"ACGTNacgtU", dtype=np.uint8), size=(n - 1) * stride + int(lens[-1]))
    ws = int(ewfa.lib().ewfa_packed_words(stride))
    expect = np.zeros(n * ws, dtype=np.uint64)
    for j in range(n):
        e = orc.pack_u64(text[j * stride: j * stride + int(lens[j])].tobytes())
        expect[j * ws: j * ws + len(e)] = e
    da, dl = ewfa.DeviceBuffer.from_array(text), ewfa.DeviceBuffer.from_array(lens)
    dw = ewfa.DeviceBuffer.from_array(np.full(n * ws, 0xFFFFFFFFFFFFFFFF, dtype=np.uint64))
    assert ewfa.lib().ewfa_pack_ascii(da.ptr, stride, dl.ptr, n, dw.ptr, ws, None) == 0
    ewfa.synchronize()
    assert np.array_equal(dw.download(np.uint64), expect)


@pytest.mark.parametrize("lo,hi", [(1, 400), (2500, 3300), (200, 11000)])
def test_cap_of_64_is_one_banded_pass(lo, hi):
    """Calls under the reference's cap at any length, also beyond one pass."""
    print(f"case cap 64, {lo}..{hi} bp", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=lo, len_lo=lo, len_hi=hi, err_lo=0.0, err_hi=0.08), 300)
    ok, d, sl, st = orc.batch_workload(w, max_distance=64)
    with ewfa.Context(max_distance=64) as ctx:
        res, cig = ctx.align_host(w.words, w.pairs, w.n, w.cigar_bytes)
    check(res, w.pairs, cig, d, st, "cap 64", capped_ok=True)


@pytest.mark.parametrize("count", [1, 2, 257, 8191, 8193, 16385, 20011])
def test_short_lists_over_the_grid(count):
    """Work shares of the banded pass around its grid and its first items."""
    print(f"case shares {count} pairs", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=0, seed=count, len=60, err=0.05), count)
    ok, d, sl, st = orc.batch_workload(w)
    dw, dp = ewfa.DeviceBuffer.from_array(w.words), ewfa.DeviceBuffer.from_array(w.pairs[:w.n])
    dr, dc = ewfa.DeviceBuffer.from_array(np.full(w.n * 4, -1, np.int32)), ewfa.DeviceBuffer(w.cigar_bytes)
    dc.fill_zero()
    with ewfa.Context() as ctx:
        ctx.align_device(dw.ptr, dp.ptr, w.n, w.max_len, dr.ptr, dc.ptr)
    check(dr.download(ewfa.RESULT_DTYPE, w.n), w.pairs[:w.n], dc.download(np.int8), d, st, count)


@pytest.mark.parametrize("name,count,near,far", [("wavefront", 1500, 3000, 0), ("bit-parallel", 1500, 0, 600),
                                                 ("both", 16000, 400, 400)])
def test_a_list_goes_one_way_or_both(tmp_path, name, count, near, far):
    """Lists of pairs of a few edits (the wavefront's), of many (bit-parallel),
    and of half and half, enough of them that both ways pay."""
    print(f"case ways {name}: {count} pairs", flush=True)
    rng = np.random.default_rng(count + near)
    pool = []
    for i in range(200):
        n = near if near and (not far or i % 2) else far
        p = rng.choice(BASES, n - int(rng.integers(40))).tobytes()
        pool.append((p, mutate(rng, p, 0.15 if n == far and not (near and i % 2) else 0.0005)))
    P, T = [pool[i % 200][0] for i in range(count)], [pool[i % 200][1] for i in range(count)]
    d, st = oracle_streams([p for p, _ in pool], [t for _, t in pool])
    d, st = [d[i % 200] for i in range(count)], [st[i % 200] for i in range(count)]
    words, pairs, cb, ml = ewfa.from_sequences(P, T)
    with ewfa.Context(policy_path=policy_file(tmp_path, "ways", POLICY)) as ctx:
        dw, dp = ewfa.DeviceBuffer.from_array(words), ewfa.DeviceBuffer.from_array(pairs)
        dr, dc = ewfa.DeviceBuffer(count * 16), ewfa.DeviceBuffer(cb)
        dc.fill_zero()
        ctx.align_device(dw.ptr, dp.ptr, count, ml, dr.ptr, dc.ptr)
        check(dr.download(ewfa.RESULT_DTYPE, count), pairs, dc.download(np.int8), d, st, name)


@pytest.mark.parametrize("count,lo,hi", [(2, 4100, 9000), (256, 2600, 4100), (257, 1300, 6000), (1025, 1300, 2600)])
def test_few_pairs_share_levels_over_more_waves(count, lo, hi):
    """Calls around a pair, and four pairs, per CU: 16, 8 and 2 waves a pair."""
    print(f"case few {count} pairs {lo}..{hi} bp", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=count, len_lo=lo, len_hi=hi, err_lo=0.02, err_hi=0.1), count)
    ok, d, sl, st = orc.batch_workload(w)
    with ewfa.Context() as ctx:
        res, cig = ctx.align_host(w.words, w.pairs, w.n, w.cigar_bytes)
    check(res, w.pairs, cig, d, st, "few")


@pytest.mark.parametrize("count,lo,hi,err", [(257, 640, 700, 0.15), (9000, 420, 440, 0.17), (700, 600, 700, 0.30)])
def test_deferred_banded_pairs_end_in_four_chunks(count, lo, hi, err):
    """Around 63 and 127 edits: what the banded pass defers, a wave's worth and
    more at a time, and what the register pass after it defers again."""
    print(f"case deferred {count} pairs {lo}..{hi} bp {err}", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=count, len_lo=lo, len_hi=hi, err_lo=err / 3, err_hi=err), count)
    ok, d, sl, st = orc.batch_workload(w)
    assert max(d) > 63
    with ewfa.Context() as ctx:
        res, cig = ctx.align_host(w.words, w.pairs, w.n, w.cigar_bytes)
    check(res, w.pairs, cig, d, st, "deferred")


@pytest.mark.parametrize("lo,hi,err", [(200, 16000, 0.01), (200, 16000, 0.08)])
def test_few_long_pairs_with_and_without_bounds(lo, hi, err):
    """Between one and four pairs per CU, of few edits and of many."""
    print(f"case few long {lo}..{hi} bp {err}", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=7, len_lo=lo, len_hi=hi, err_lo=err / 2, err_hi=err), 300)
    ok, d, sl, st = orc.batch_workload(w)
    with ewfa.Context() as ctx:
        for _ in range(3):  # eager, recorded, replayed
            res, cig = ctx.align_host(w.words, w.pairs, w.n, w.cigar_bytes)
            check(res, w.pairs, cig, d, st, "few long")


@pytest.mark.parametrize("order", ["abab", "aacaaba", "bdadbca"])
def test_control_words_between_calls(order):
    """Calls of one context that leave its counters at zero, or not: one pass
    (a), one that defers (b), several buckets (c), longer pairs than before (d)."""
    print(f"case calls {order}", flush=True)
    shapes = {"a": (300, 100, 150, 0.03), "b": (300, 640, 700, 0.16), "c": (900, 100, 3000, 0.05), "d": (40, 2000, 5000, 0.1)}
    made = {}
    for k, (n, lo, hi, err) in shapes.items():
        w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=n + lo, len_lo=lo, len_hi=hi, err_lo=err / 2, err_hi=err), n)
        made[k] = (w, orc.batch_workload(w))
    with ewfa.Context() as ctx:
        for k in order:
            w, (ok, d, sl, st) = made[k]
            dw, dp = ewfa.DeviceBuffer.from_array(w.words), ewfa.DeviceBuffer.from_array(w.pairs[:w.n])
            dr, dc = ewfa.DeviceBuffer(w.n * 16), ewfa.DeviceBuffer(w.cigar_bytes)
            dc.fill_zero()
            ctx.align_device(dw.ptr, dp.ptr, w.n, w.max_len, dr.ptr, dc.ptr)
            check(dr.download(ewfa.RESULT_DTYPE, w.n), w.pairs[:w.n], dc.download(np.int8), d, st, order + k)
