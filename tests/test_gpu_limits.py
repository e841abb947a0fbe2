"""Calls at the limits of what their passes hold, against the oracle."""
import ctypes
import time

import numpy as np
import pytest

import ewfa
import oracle_py as orc
from test_gpu_bitpar import POLICY, mutate
from test_gpu_bound import check, policy_file
from test_gpu_stress import oracle_streams

pytestmark = pytest.mark.gpu

BASES = np.frombuffer(b"ACGT", dtype=np.uint8)


class OnDevice:
    """Sequences, descriptors and outputs in device memory."""

    def __init__(self, words, pairs, cigar_bytes, max_len):
        self.pairs, self.n, self.max_len = pairs, len(pairs), max_len
        self.dw, self.dp = ewfa.DeviceBuffer.from_array(words), ewfa.DeviceBuffer.from_array(pairs)
        self.dr, self.dc = ewfa.DeviceBuffer(self.n * 16), ewfa.DeviceBuffer(cigar_bytes)
        self.dc.fill_zero()

    def align(self, ctx):
        ctx.align_device(self.dw.ptr, self.dp.ptr, self.n, self.max_len, self.dr.ptr, self.dc.ptr)
        return self

    def check(self, d, st, label):
        check(self.dr.download(ewfa.RESULT_DTYPE, self.n), self.pairs, self.dc.download(np.int8), d, st, label)


def fill_pairs(count, lo=40, hi=260, seed=3):
    """Short pairs of a few substitutions, and their oracle outputs."""
    rng = np.random.default_rng(seed)
    pool = []
    for _ in range(200):
        p = rng.choice(BASES, int(rng.integers(lo, hi)))
        t = p.copy()
        t[rng.integers(0, len(t), 3)] = rng.choice(BASES, 3)
        pool.append((p.tobytes(), t.tobytes()))
    d, st = oracle_streams([p for p, _ in pool], [t for _, t in pool])
    take = [i % len(pool) for i in range(count)]
    return [pool[i][0] for i in take], [pool[i][1] for i in take], [d[i] for i in take], [st[i] for i in take]


@pytest.mark.parametrize("count", [300, 8300])
def test_distances_beyond_the_narrow_slots_and_the_widest_band(tmp_path, count):
    """One bucket whose budget exceeds any distance: pairs beyond what its
    narrow slots hold (9,600 levels at this length), and beyond the widest
    band of the bit-parallel pass (8,129), which defer them."""
    print(f"case beyond the bands: {count} pairs", flush=True)
    # nothing in common: as many substitutions as bases
    P, T = [b"A" * n for n in (9700, 9500, 8200, 9400)], [b"C" * n for n in (9700, 9500, 8200, 9400)]
    d, st = [len(p) for p in P], [np.full(len(p), ord("X"), dtype=np.int8) for p in P]
    fp, ft, fd, fst = fill_pairs(count - len(P))
    case = OnDevice(*ewfa.from_sequences(P + fp, T + ft))
    with ewfa.Context(policy_path=policy_file(tmp_path, "one", POLICY)) as ctx:
        case.align(ctx).check(d + fd, st + fst, "beyond the bands")


def test_outputs_are_pinned_only_within_one_allocation():
    """Buffers the device may write as they are: parts of one pinned
    allocation, and nothing that reaches past its end into another."""
    print("case pinned ranges", flush=True)
    mapped = ewfa.lib()._ZN4ewfa11mapped_hostEPvm
    mapped.restype, mapped.argtypes = ctypes.c_void_p, [ctypes.c_void_p, ctypes.c_size_t]
    size = 3 << 20
    held = [ewfa.PinnedArray(size, np.uint8) for _ in range(2)]
    a, b = sorted(h.array.ctypes.data for h in held)
    assert mapped(a, size) and mapped(a + 4096, size - 4096) and mapped(a + size - 4, 4) and mapped(b, 0)
    assert not mapped(a, b - a + size)  # both ends pinned, and what lies between not known to be
    assert not mapped(a + 4, size)
    plain = np.zeros(size, dtype=np.uint8)
    assert not mapped(plain.ctypes.data, size)
    dev = ewfa.DeviceBuffer(size)
    assert not mapped(dev.ptr, size)


@pytest.mark.parametrize("flags", [0, 0x40000000, 0x80000000])  # default, coherent, non-coherent
def test_streams_in_pinned_memory_of_every_kind(flags):
    """Calls one after the other into the same pinned buffers, read by the host
    after each."""
    hip = ctypes.CDLL("libamdhip64.so")

    def pinned(nbytes):
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(nbytes), ctypes.c_uint(flags)) == 0
        return p, np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_int8)), (nbytes,))

    print(f"case pinned memory {flags:#x}", flush=True)
    ewfa.synchronize()
    loads = []
    for seed in range(3):
        w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=seed, len_lo=100, len_hi=700, err_lo=0.01, err_hi=0.1), 3000,
                          cigar_cap=160)
        ok, d, sl, st = orc.batch_workload(w)
        loads.append((w, d, st))
    pr, res = pinned(3000 * 16)
    pc, cig = pinned(3000 * 160)
    res = res.view(ewfa.RESULT_DTYPE)
    with ewfa.Context() as ctx:
        for k in (0, 1, 2, 0, 1, 2):
            w, d, st = loads[k]
            cig[:] = 1
            ctx.align_host(w.words, w.pairs, w.n, w.cigar_bytes, results=res, cigars=cig)
            check(res, w.pairs[:w.n], cig, d, st, (flags, k))
    for p in (pr, pc):
        assert hip.hipHostFree(p) == 0


@pytest.mark.parametrize("entry", ["ewfa_upload_words", "ewfa_upload_words_async"])
def test_uploaded_words_have_room_for_the_last_pad_word(entry):
    """The last sequence's pad word, which kernels read, may lie just past the
    words given: the context's buffer holds it."""
    n = 1 << 18  # whole pages of words
    print(f"case pad word {entry}", flush=True)
    words = np.zeros(n, dtype=np.uint64)
    with ewfa.Context() as ctx:
        before = ctx.memory_bytes()
        assert getattr(ewfa.lib(), entry)(ctx.handle, ctypes.c_void_p(words.ctypes.data), ctypes.c_size_t(n)) == 0
        ewfa.synchronize()
        assert ctx.memory_bytes() - before >= (n + 1) * 8


def test_short_pairs_beside_one_beyond_lds_are_not_served_in_turn():
    """A call of few pairs, one of which needs its slot in HBM: the others run
    beside it, so that the call takes little longer than that pair alone."""
    print("case 60 pairs of 10 kbp and one of 400 kbp", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=5, len_lo=9000, len_hi=10000, err_lo=0.01, err_hi=0.02), 60)
    P, T = [bytes(w.pattern(i)) for i in range(60)], [bytes(w.text(i)) for i in range(60)]
    rng = np.random.default_rng(4)
    p = rng.choice(BASES, 400_000)
    t = p.copy()
    at = rng.choice(400_000, 300, replace=False)
    t[at] = BASES[(np.searchsorted(BASES, t[at]) + 1) % 4]
    d, st = oracle_streams(P + [p.tobytes()], T + [t.tobytes()])
    took = []
    for a, b, dd, ss in (([], [], [], []), (P, T, list(d[:60]), list(st[:60]))):
        case = OnDevice(*ewfa.from_sequences(a + [p.tobytes()], b + [t.tobytes()]))
        with ewfa.Context() as ctx:
            case.align(ctx).check(dd + [d[60]], ss + [st[60]], "beside 400 kbp")
            times = []
            for _ in range(7):
                t0 = time.perf_counter()
                case.align(ctx)
                times.append(time.perf_counter() - t0)
        took.append(sorted(times)[3])
    assert took[1] < 1.6 * took[0], took


def median_us(call, reps=7):
    call()
    times = []
    for _ in range(reps):
        t0 = time.perf_counter()
        call()
        times.append(time.perf_counter() - t0)
    return sorted(times)[reps // 2] * 1e6


def test_a_list_beyond_its_budget_goes_on_to_the_next(tmp_path):
    """2,210 pairs of 4,760 bp at 12.6%: 540 to 600 edits, beyond their bucket's
    512 levels and within the 1,024 that follow, which hold them at twice the
    occupancy of a budget of the whole length."""
    print("case 2210 pairs of 4760 bp, all deferred", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=0, seed=5, len=4760, err=0.126), 2210)
    few = ewfa.Workload(ewfa.synth_spec(kind=0, seed=5, len=4760, err=0.126), 24)
    ok, d, sl, st = orc.batch_workload(few)
    case = OnDevice(w.words, w.pairs[:w.n].copy(), w.cigar_bytes, w.max_len)
    out, took = [], []
    for path in (policy_file(tmp_path, "enough", "4000000000 2 1024 0 1\n"), None):
        with ewfa.Context(policy_path=path) as ctx:
            case.dc.fill_zero()
            took.append(median_us(lambda: case.align(ctx)))
        res, cig = case.dr.download(ewfa.RESULT_DTYPE, case.n), case.dc.download(np.int8)
        check(res[:24], case.pairs[:24], cig, d, st, path)
        assert (res["status"] == ewfa.PAIR_OK).all() and res["distance"].max() > 512
        out.append((res, cig))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert took[1] < 2.2 * took[0], took


def test_the_allocation_free_call_takes_what_its_per_pair_buffers_hold():
    """Short pairs fill its scratch to the last pair: no pass refuses what is
    left of it."""
    print("case allocation-free, scratch full of 150 bp pairs", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=0, seed=5, len=150, err=0.02), 1000)
    ok, d, sl, st = orc.batch_workload(w)
    n = 1_400_000
    pairs = np.resize(w.pairs[:w.n], n)
    pairs["cigar_off"] = np.arange(n, dtype=np.uint64) * 64
    pairs["cigar_cap"] = 64
    case = OnDevice(w.words, pairs, 64 * n, w.max_len)

    def call(m):
        ctx.align_device_noalloc(case.dw.ptr, case.dp.ptr, m, case.max_len, case.dr.ptr, case.dc.ptr, None)

    with ewfa.Context() as ctx:
        lo, hi = 1_000_000, n
        while lo < hi:
            m = (lo + hi + 1) // 2
            try:
                call(m)
                lo = m
            except ewfa.EwfaError as e:
                hi, why = m - 1, str(e)
        call(lo)
        res, cig = case.dr.download(ewfa.RESULT_DTYPE, n), case.dc.download(np.int8)
        assert "before any pass" in why, (lo, why)
        check(res[lo - 1000:lo], pairs[lo - 1000:lo], cig, [d[i % 1000] for i in range(lo - 1000, lo)],
              [st[i % 1000] for i in range(lo - 1000, lo)], lo)


def test_the_allocation_free_call_over_few_long_pairs():
    """200 pairs, whose longest have room for a few blocks only, take no longer
    than 300 of the same lengths."""
    took = []
    for n in (200, 300):
        print(f"case allocation-free, {n} pairs of 1..12 kbp", flush=True)
        w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=5, len_lo=1000, len_hi=12000, err_lo=0.025, err_hi=0.05), n)
        ok, d, sl, st = orc.batch_workload(w)
        case = OnDevice(w.words, w.pairs[:w.n].copy(), w.cigar_bytes, w.max_len)
        with ewfa.Context() as ctx:
            took.append(median_us(lambda: ctx.align_device_noalloc(case.dw.ptr, case.dp.ptr, n, case.max_len,
                                                                   case.dr.ptr, case.dc.ptr, None)))
        case.check(d, st, "allocation-free")
    assert took[0] < 1.2 * took[1], took


def test_bit_parallel_slots_leave_others_room():
    """With 44 GiB of the device free, a call whose bit-parallel slots could
    take 40 (its wavefront's own take 21) holds about half of them."""
    gib = 44
    hip = ctypes.CDLL("libamdhip64.so")

    def free_bytes():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    fp, ft, fd, fst = fill_pairs(5000)
    rng = np.random.default_rng(gib)
    P = [rng.choice(BASES, n).tobytes() for n in (24_000, 49_000)]
    T = [bytes(BASES[(np.searchsorted(BASES, np.frombuffer(p, np.uint8)) + (np.arange(len(p)) % 25 == 7)) % 4]) for p in P]
    d, st = oracle_streams(P, T)
    case = OnDevice(*ewfa.from_sequences(P + fp, T + ft))
    ewfa.synchronize()
    print(f"case {gib} GiB free", flush=True)
    held = ewfa.DeviceBuffer(free_bytes() - (gib << 30))
    try:
        with ewfa.Context() as ctx:
            for _ in range(2):
                case.align(ctx).check(list(d) + fd, list(st) + fst, gib)
            assert ctx.memory_bytes() < 0.6 * (gib << 30)
            assert free_bytes() > 0.35 * (gib << 30)
    finally:
        held.free()


@pytest.mark.parametrize("policy", [None, "500 1 200 1 2\n1500 1 40 1 2\n4000000000 4 300 0 1\n"])
def test_deferred_pairs_of_every_bucket(tmp_path, policy):
    """A list in which every bucket defers pairs: each goes untried through the
    deferral passes that hold no more than its bucket's did, and ends in a
    later one.  Also where a shorter bucket has the larger budget."""
    print("case deferred from every bucket", flush=True)
    rng = np.random.default_rng(8)
    P, T = [], []
    for n, rate in ((250, .40), (480, .30), (650, .25), (690, .12), (1100, .14), (1400, .08), (2400, .40), (3000, .14),
                    (4900, .16), (9000, .15), (10400, .13)):
        for _ in range(4):
            p = rng.choice(BASES, n).tobytes()
            P.append(p)
            T.append(mutate(rng, p, rate))
    d, st = oracle_streams(P, T)
    fp, ft, fd, fst = fill_pairs(600)
    order = rng.permutation(len(P) + 600)
    P, T, d, st = P + fp, T + ft, list(d) + fd, list(st) + fst
    P, T, d, st = ([x[i] for i in order] for x in (P, T, d, st))
    case = OnDevice(*ewfa.from_sequences(P, T))
    with ewfa.Context(policy_path=policy_file(tmp_path, "some", policy) if policy else None) as ctx:
        for _ in range(2):
            case.dc.fill_zero()
            case.align(ctx).check(d, st, policy)


@pytest.mark.parametrize("err", [0.01, 0.12])
@pytest.mark.parametrize("count", [10_240, 10_241, 32_768, 32_769])
def test_streams_by_wave_and_by_lane(tmp_path, count, err):
    """Lists on either side of 40 and 128 pairs per CU: a wave a pair, as a
    sample of the results says, and a lane a pair."""
    print(f"case streams {count} pairs {err}", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=2, seed=count, len_lo=100, len_hi=200, err_lo=err / 2, err_hi=err), count)
    ok, d, sl, st = orc.batch_workload(w)
    case = OnDevice(w.words, w.pairs[:w.n].copy(), w.cigar_bytes, w.max_len)
    with ewfa.Context(policy_path=policy_file(tmp_path, "block", "4000000000 2 256 0 1\n")) as ctx:
        for _ in range(2):
            case.dc.fill_zero()
            case.align(ctx).check(d, st, (count, err))


class EmitArgs(ctypes.Structure):
    _fields_ = [(k, ctypes.c_void_p) for k in ("words", "pairs", "results", "ops")] + [
        ("ops_stride", ctypes.c_uint32), ("cigars", ctypes.c_void_p), ("list", ctypes.c_void_p),
        ("count", ctypes.c_uint32), ("count_ptr", ctypes.c_void_p), ("per_wave", ctypes.c_uint32)]


@pytest.mark.parametrize("count,distance,waves", [(15_000, 50, True), (15_000, 80, False), (30_000, 30, True),
                                                  (30_000, 40, False), (300, 900, True), (1, 1000, True), (0, 0, True)])
def test_a_sample_of_the_results_picks_the_emit(count, distance, waves):
    """At 256 CUs a list of 1,500 bp pairs goes by waves while its pairs per CU
    times its edits a base stay within 2.5."""
    print(f"case pick {count} pairs of {distance} edits", flush=True)
    n = max(count, 1)
    pairs, res = np.zeros(2 * n, dtype=ewfa.PAIR_DTYPE), np.zeros(2 * n, dtype=ewfa.RESULT_DTYPE)
    pairs["tlen"] = 1500
    res["distance"], res["status"] = distance, ewfa.PAIR_OK
    res["distance"][::2], res["status"][1::14] = 1500, ewfa.PAIR_BADARG  # not of the list, and not aligned
    lst = np.arange(n, dtype=np.uint32) * 2 + 1
    bufs = [ewfa.DeviceBuffer.from_array(x) for x in (pairs, res, lst, np.array([count, 7, 7], dtype=np.uint32))]
    args = EmitArgs(pairs=bufs[0].ptr, results=bufs[1].ptr, list=bufs[2].ptr, count=3 * n, count_ptr=bufs[3].ptr)
    pick = ewfa.lib()._ZN4ewfa16launch_emit_pickERKNS_8EmitArgsEfPjP12ihipStream_t
    pick.argtypes = [ctypes.c_void_p, ctypes.c_float, ctypes.c_void_p, ctypes.c_void_p]
    at = bufs[3].ptr.value if isinstance(bufs[3].ptr, ctypes.c_void_p) else bufs[3].ptr
    assert pick(ctypes.byref(args), 2.5 * 256, at + 4, None) == 0
    ewfa.synchronize()
    got = bufs[3].download(np.uint32, 3)
    assert got.tolist() == [count, count if waves else 0, 0 if waves else count]


@pytest.mark.parametrize("count,kind,lo,hi,err,bits", [
    (2500, 2, 4350, 8700, 0.06, False),   # 0.86 ms by the wavefront, 2.36 bit-parallel
    (2500, 2, 2500, 5000, 0.09, False),   # 0.71 and 1.49
    (1450, 2, 4832, 24162, 0.06, False),  # 3.6 and 8.6: weighed by its bounds
    (6000, 0, 8700, 8700, 0.13, True),    # 92 (beyond its budget) and 4.1
    (15000, 0, 5000, 5000, 0.13, True),   # 36 and 3.0
])
def test_a_sample_sends_a_list_the_faster_way(count, kind, lo, hi, err, bits):
    """Lists whose two ways are far apart, beside the same call with a distance
    cap beyond any distance, which only has the wavefront."""
    print(f"case sampled {count} pairs of {lo}..{hi} at {err}", flush=True)
    w = ewfa.Workload(ewfa.synth_spec(kind=kind, seed=5, len=hi, err=err, len_lo=lo, len_hi=hi, err_lo=err / 2,
                                      err_hi=err), count)
    case = OnDevice(w.words, w.pairs[:w.n].copy(), w.cigar_bytes, w.max_len)
    out, took = [], []
    for cap in (0, 1 << 20):
        with ewfa.Context(max_distance=cap) as ctx:
            case.dc.fill_zero()
            took.append(median_us(lambda: case.align(ctx), 5))
        out.append((case.dr.download(ewfa.RESULT_DTYPE, count), case.dc.download(np.int8)))
    assert (out[0][0]["status"] == ewfa.PAIR_OK).all()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert took[0] < (0.5 if bits else 1.35) * took[1], took
