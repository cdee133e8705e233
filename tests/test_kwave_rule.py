"""The rule that puts a launch on the tiles whose K the waves share
(kernels::kwave_plan_shape and launch_bytes_wanted, through the hostsim
library): over seeded shapes of every form a plan's ranges cover K in multiples
of 32, its tile is one the form has, no chain of a sum is longer than the ranges
of the split rule nor than 1024, a launch
given exactly the partials its plan wants takes the same plan and one byte less
another that fits, and the partials of any launch fit the allocation-free
entry's 128 MiB."""
import ctypes
import time

import numpy as np

import xvram_amd as xv

from gemm_cases import route

ANY = (1 << 64) - 1
RUN = (32, 32, 32, 32, 128, 0, 0)


def fns():
    dll = xv.load(hostsim=True).dll
    i64, pint = ctypes.c_int64, ctypes.POINTER(ctypes.c_int)
    dll.xvram_hostsim_kwave_plan.argtypes = [i64] * 3 + [ctypes.c_int, ctypes.c_uint64] + [pint] * 3
    dll.xvram_hostsim_split_shape.argtypes = [i64] * 3 + [ctypes.c_int] * 2 + [ctypes.c_uint64, pint, pint]
    dll.xvram_hostsim_launch_bytes_wanted.argtypes = [ctypes.c_int] * 5 + [i64] * 2
    dll.xvram_hostsim_launch_bytes_wanted.restype = ctypes.c_uint64
    dll.xvram_hostsim_k_remainder_shape.argtypes = [i64] * 3 + [ctypes.c_int]
    dll.xvram_hostsim_k_remainder_shape.restype = i64
    return dll


def test_plan_properties():
    dll = fns()

    def plan(m, n, k, nt, ws=ANY):
        s, d, f = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
        t = dll.xvram_hostsim_kwave_plan(m, n, k, nt, ws, ctypes.byref(s), ctypes.byref(d), ctypes.byref(f))
        return t, s.value, d.value, f.value

    rng = np.random.default_rng(41)
    tiles, split = set(), 0
    for _ in range(4000):
        m, n = (int(2 ** v) for v in rng.uniform(0, 13, 2))
        k = int(2 ** rng.uniform(0, 16))
        nt = int(rng.integers(0, 2))
        tile, s, depth, fold = plan(m, n, k, nt)
        fits = k >= 8 and -(-m // 256) * -(-n // 256) < 256
        old = ctypes.c_int(), ctypes.c_int()
        olds = dll.xvram_hostsim_split_shape(m, n, k, nt, 1, ANY, ctypes.byref(old[0]), ctypes.byref(old[1]))
        if tile < 0:
            ring = olds > 1 and not old[1].value and old[0].value >= 4096
            assert not fits or ring
            continue
        tiles.add((tile, nt))
        assert fits and (tile < 5 or nt)
        assert (s == 1 and depth == k) or (depth % 32 == 0 and (s - 1) * depth < k <= s * depth)
        chain = min(old[0].value if olds > 1 else k, 1024)
        if (depth + 3) // 4 > chain:
            assert fold % RUN[tile] == 0 and RUN[tile] <= fold <= chain
        partial = (m + 3) // 4 * 4 * n * 4
        if s > 1:
            split += 1
            assert s * partial <= 64 << 20
            assert plan(m, n, k, nt, s * partial) == (tile, s, depth, fold)
            less = plan(m, n, k, nt, s * partial - 1)
            assert less[1] == 1 or less[1] * partial < s * partial
        assert plan(m, n, k, nt, 0)[1] == 1
    assert tiles >= {(t, nt) for t in range(5) for nt in (0, 1)} | {(6, 1)} and split > 500


def test_many_tiles():
    """Launches of 256 tiles of 256 x 256 and more (kernels::many_shape): whole
    rounds of interior tiles stay on the ring kernels; shallow K and K that is no
    multiple of their step below 512 go to small tiles and want no partials; a
    rectangle of whole rounds is whole 256 x 256 tiles inside C that fill at least
    19/20 of their rounds, smaller than C, needs K of the ring kernels' step from
    1024 on and runs on those kernels."""
    dll = fns()
    i64, pint = ctypes.c_int64, ctypes.POINTER(ctypes.c_int)
    dll.xvram_hostsim_kwave_many.argtypes = [i64] * 3 + [ctypes.c_int, pint] + [ctypes.POINTER(i64)] * 2

    def many(m, n, k, nt):
        mi, ni = i64(), i64()
        t = dll.xvram_hostsim_kwave_many(m, n, k, nt, None, ctypes.byref(mi), ctypes.byref(ni))
        return t, mi.value, ni.value

    for whole in ((4096, 4096, 256, 1), (8192, 8192, 8192, 1), (8192, 8192, 1024, 0)):
        assert many(*whole) == (-1, 0, 0)
    assert many(5000, 5000, 5000, 0) == many(5000, 5000, 5000, 1) == (-1, 4096, 4096)
    # The best rectangle of all would be one round of 252 or 255 tiles: small tiles. Where
    # only the chains leave it fewer (14 of 18 tile rows), it is taken.
    assert many(5586, 3566, 3344, 0)[0] == many(4352, 4352, 2048, 0)[0] == 2
    assert many(4608, 4608, 2048, 0) == (-1, 3584, 4608)
    assert many(3712, 4590, 503, 1)[0] == many(6379, 2968, 32, 1)[0] == 6
    # K no multiple of the ring kernels' step and no K remainder: the general kernel,
    # against which the small tiles are rated (a rectangle runs on neither).
    assert route(4096, 4096, 4099, "NN") == route(8192, 8192, 4099, "NT") == "general"
    assert route(17152, 7936, 10711, "NN").startswith("small 64x64 ranges 1 ")
    # A grid of 2^24 workgroups of 256 threads is past what one launch holds.
    assert many(1 << 17, 1 << 18, 9, 0)[0] == 2 and many(1 << 19, 1 << 19, 9, 0)[0] == -1
    rng = np.random.default_rng(47)
    small = rect = 0
    for _ in range(3000):
        m, n = (int(2 ** v) for v in rng.uniform(8, 14, 2))
        k, nt = int(2 ** rng.uniform(0, 13)), int(rng.integers(0, 2))
        k = k // 8 * 8 if rng.random() < 0.5 else k
        tile, mi, ni = many(m, n, k, nt)
        if -(-m // 256) * -(-n // 256) < 256 or k < 8:
            assert (tile, mi, ni) == (-1, 0, 0)
        elif k < 512 and k % (4 if nt else 8):
            assert tile >= 0
        lda, ldb = (m + 3) // 4 * 4, ((n if nt else k) + 3) // 4 * 4
        if tile >= 0:
            small += 1
            assert mi == 0 and dll.xvram_hostsim_launch_bytes_wanted(m, n, k, 0, nt, lda, ldb) == 0
        if mi:
            rect += 1
            assert mi % 256 == ni % 256 == 0 and 0 < mi <= m and 0 < ni <= n and (mi < m or ni < n)
            groups = mi // 256 * (ni // 256)
            assert 20 * groups >= 19 * -(-groups // 256) * 256
            how = route(m, n, k, ("NN", "NT")[nt])
            assert how.startswith(f"rectangle[{mi}x{ni}x")
            assert all(part.endswith(" ring") for part in how[10:-1].split("; ")
                       if part.startswith(f"{mi}x{ni}x"))
            assert k >= 1024 and k % (4 if nt else 8) == 0
    assert small > 100 and rect > 30


def test_no_chain_is_longer_than_the_large_kernels_make_it():
    """Over seeded launches of 256 tiles and more, elements at the corners, on both
    sides of the interior's edges and anywhere: small tiles, rectangles and strips
    add no more k values in one accumulator than the rules of the large kernels
    alone would for that element (a split tail's ranges, an edge strip's)."""
    dll = fns()
    fn = dll.xvram_hostsim_longest_chain
    fn.restype = ctypes.c_int64
    fn.argtypes = [ctypes.c_int] * 5 + [ctypes.c_int64] * 4 + [ctypes.c_int]
    rng = np.random.default_rng(53)
    rect = passes = edges = 0
    for _ in range(6000):
        m, n = (int(2 ** v) for v in rng.uniform(10, 14, 2))
        k = int(2 ** rng.uniform(8, 13))
        if rng.random() < 0.5:
            k = k // 8 * 8
        if rng.random() < 0.3:
            m, n = m // 256 * 256, n // 256 * 256
        if -(-m // 256) * -(-n // 256) < 256:
            continue
        form = ("NN", "NT", "TN", "TT")[int(rng.integers(0, 4))]
        ak, bn = form[0] == "T", form[1] == "T"
        lda, ldb = ((k if ak else m) + 3) // 4 * 4, ((n if bn else k) + 3) // 4 * 4
        how = route(m, n, k, form)
        rect += how.startswith("rectangle")
        first = how[10:].split(";") if how.startswith("rectangle") else ["", ""]
        passes += len(first) > 1 and first[0].split("x")[:2] == first[1].strip().split("x")[:2]
        edges += " edge " in how and "edge split" not in how
        rows = {0, m - 1, m // 256 * 256 - 1, *(int(v) for v in rng.integers(0, m, 4))}
        cols = {0, n - 1, n // 256 * 256 - 1, *(int(v) for v in rng.integers(0, n, 4))}
        for i in rows:
            for j in cols:
                now, before = (fn(m, n, k, ak, bn, lda, ldb, i, j, large) for large in (0, 1))
                assert now <= before, (m, n, k, form, i, j, now, before, how)
    assert rect > 100 and passes > 20 and edges > 100, (rect, passes, edges)
    # The rectangle reaches past the head of the rules' tail split (13 of its 16 tile
    # rows), whose tail's ranges are 2528 deep: two passes.
    assert route(5000, 5000, 5000, "TT").startswith("rectangle[4096x4096x2528 ring; 4096x4096x2472 ring;")
    # 13 x 19 tiles in one pass leave strips that end in a nearly empty round.
    assert route(5000, 5000, 2048, "NN").startswith("rectangle[4096x4096x1024 ring; 4096x4096x1024 ring;")
    # Rows that lie in a tail of 320-deep ranges.
    assert fn(2304, 8512, 2080, 0, 0, 2304, 2080, 1800, 0, 0) <= 320


def test_odd_k_runs_on_the_kernel_rated_faster():
    """Interior launches of an odd K: without a K remainder they run on the general
    kernel or on small tiles, whichever models faster (up to K = 1200 the small
    tiles up to 4 % behind), and never on neither because a rectangle that no K
    remainder will run modelled faster still."""
    dll = fns()
    dll.xvram_hostsim_odd_k_times.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] + \
        [ctypes.POINTER(ctypes.c_double)] * 2
    small, general = ctypes.c_double(), ctypes.c_double()
    rng = np.random.default_rng(59)
    seen = {"general": 0, "small": 0, "k remainder": 0}
    for _ in range(1500):
        m, n = (256 * int(2 ** v) for v in rng.uniform(3, 6.2, 2))
        k, form = int(rng.integers(520, 12000)) | 1, ("NN", "NT")[int(rng.integers(0, 2))]
        if m // 256 * (n // 256) < 256:
            continue
        how = route(m, n, k, form)
        kind = next(r for r in seen if how.startswith(r))
        seen[kind] += 1
        dll.xvram_hostsim_odd_k_times(m, n, k, form == "NT", ctypes.byref(small), ctypes.byref(general))
        limit = 1.04 if k < 1200 else 1.0
        if kind == "general":
            assert small.value >= limit * general.value, (m, n, k, form)
        elif dll.xvram_hostsim_k_remainder_shape(m, n, k, form == "NT") == 0:
            assert small.value < limit * general.value, (m, n, k, form)
    assert min(seen.values()) > 20, seen


def test_rule_is_quick_for_many_tiles():
    """The rule runs on every enqueue: over 512 x 512 tiles it takes microseconds
    (a search of rounds x tile rows took 2 ms; the bound leaves a slow machine room)."""
    dll = fns()
    start = time.perf_counter()
    for _ in range(20):
        dll.xvram_hostsim_launch_bytes_wanted(131072, 131072, 1032, 0, 0, 4, 4)
    assert (time.perf_counter() - start) / 20 < 0.5e-3


def test_partials_fit_the_scratch():
    dll = fns()
    rng = np.random.default_rng(43)
    split = 0
    for _ in range(8000):
        scale = int(rng.choice([512, 4096, 16384]))
        m, n = (int(v) for v in rng.integers(1, scale + 1, 2))
        k = int(rng.integers(1, 3 * scale))
        if rng.random() < 0.5:
            m, n = 256 * max(1, m // 256), 256 * max(1, n // 256)
        ak, bn = (int(v) for v in rng.integers(0, 2, 2))
        lda, ldb = ((k if ak else m) + 3) // 4 * 4, ((n if bn else k) + 3) // 4 * 4
        wanted = dll.xvram_hostsim_launch_bytes_wanted(m, n, k, ak, bn, lda, ldb)
        split += wanted > 0
        assert wanted <= 128 << 20, (m, n, k, ak, bn)
    assert split > 300


def test_planner_gives_the_partials_frame_to_a_larger_block(oracle_mod):
    """1024 x 1024 x 8192 N/T under 12 frames of 2 MiB: 2 x 2 C tiles of 512 x
    512 and 8 K panels. Its launches run on small tiles, so the plan takes all
    four C tiles in one block instead of keeping a frame for partials: A and B
    cross the link once, and the product is exact on the analytic pattern."""
    from gemm_cases import pattern_operands
    from xvram_amd import abi

    m, n, k = 1024, 1024, 8192
    a_op, b_op = pattern_operands(m, n, k)
    lib = xv.load(hostsim=True)
    lib.dll.xvram_hostsim_reset()
    with xv.Session(lib, chunk_size_bytes=2 << 20, cache_target_bytes=24 << 20, workspace_cap_bytes=0,
                    device_headroom_bytes=0, max_transaction_ms=600000) as s:
        A, B, C = s.allocation(4 * m * k), s.allocation(4 * n * k), s.allocation(4 * m * n)
        A.write(np.ascontiguousarray(a_op.T, dtype=np.float32))
        B.write(np.ascontiguousarray(b_op, dtype=np.float32))
        plan = xv.GemmPlan(s, xv.matrix(A, m, k, m), xv.matrix(B, n, k, n), xv.matrix(C, m, n, m),
                           abi.OP_N, abi.OP_T)
        info = plan.info()
        plan.execute()
        out = C.read(dtype=np.float32).reshape(n, m).T
        h2d = s.telemetry().bytes_h2d
        plan.release()
    assert (info.tile_m, info.tile_n, info.tile_count) == (512, 512, 32)
    assert info.maximum_working_set_bytes == 3 * (2 << 20)
    assert h2d == 4 * (m * k + n * k)
    assert np.array_equal(out.astype(np.float64), oracle_mod.pattern_expected_matrix(m, n, k))
