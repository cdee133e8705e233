"""Tiles whose K the waves of a workgroup share (sgemm_kwave.hip) on the MI355X,
through the extension's sgemm_device: each tile of the rule in each form at the
edges of its range -- one tile, tiles cut by m and n, K tails, fewer slots than
waves, chains that fold, K split over workgroups -- with alpha,
beta, a row or column bias and ReLU over operands whose padding is NaN. Every
element is within 4*K*2^-24*(|alpha||A||B| + |beta C0| + |bias|) of the FP64
result, the padding of C keeps its bits, and a second run gives the same bits."""
import ctypes

import numpy as np
import pytest

import xvram_amd as xv
from xvram_amd import abi

from gemm_cases import route
from test_gpu_sgemm_device import FORMS, Hip, desc_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    return xv.load()


@pytest.fixture()
def hip(lib):
    h = Hip()
    yield h
    h.close()


def plan(m, n, k, form):
    """(tile, K ranges, fold) of the rule, given any workspace."""
    fn = xv.load(hostsim=True).dll.xvram_hostsim_kwave_plan
    fn.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.c_uint64] + [ctypes.POINTER(ctypes.c_int)] * 3
    s, d, f = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    t = fn(m, n, k, int(form == "NT"), (1 << 64) - 1, ctypes.byref(s), ctypes.byref(d), ctypes.byref(f))
    return t, s.value, f.value


def many(m, n, k, form):
    fn = xv.load(hostsim=True).dll.xvram_hostsim_kwave_many
    fn.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int, ctypes.POINTER(ctypes.c_int), ctypes.c_void_p,
                                          ctypes.c_void_p]
    f = ctypes.c_int()
    return fn(m, n, k, int(form == "NT"), ctypes.byref(f), None, None), 1, f.value


def padded_nan(mat, extra):
    rows, cols = mat.shape
    ld = (rows + 3) // 4 * 4 + extra
    buf = np.full((cols, ld), np.nan, dtype=np.float32)
    buf[:, :rows] = mat.T
    return buf, ld


# (m, n, k): the tile, whether K splits over workgroups and whether chains fold
# in the N/N, T/N and T/T forms, and in N/T.
CASES = [
    ((1, 1, 8), (0, False, False), None),
    ((33, 31, 9), (0, False, False), None),
    ((100, 84, 260), (0, False, False), None),
    ((5, 3751, 406), (0, False, True), None),
    ((9, 36, 7124), (0, True, False), None),
    ((4, 3353, 2220), (0, True, True), None),
    ((391, 2806, 212), (1, False, False), None),
    ((1450, 973, 410), (1, False, True), None),
    ((4910, 7, 2046), (1, True, False), None),
    ((433, 70, 12283), (1, True, True), None),
    ((5405, 740, 59), (2, False, False), (6, False, False)),
    ((3582, 2666, 9), (1, False, False), (6, False, False)),
    ((1557, 506, 729), (2, False, True), None),
    ((5417, 43, 1723), (2, True, False), None),
    ((666, 434, 1525), (2, True, True), None),
    ((41, 2771, 4028), (2, True, True), (6, True, False)),
    ((4085, 3, 13738), (3, True, False), None),
    ((4630, 3, 12564), (3, True, True), None),
    ((5470, 5, 2545), (4, False, True), None),
    ((6, 194, 16278), (4, True, False), None),
    ((2313, 1, 10837), (4, True, True), None),
]
# The same for launches of 256 tiles of 256 x 256 and more.
MANY = [
    ((100, 65401, 41), (2, False, False), (6, False, False)),
    ((4098, 4099, 31), (1, False, False), (6, False, False)),
    ((1501, 15842, 1730), (2, False, False), (5, False, False)),
]


# Launches of many tiles whose sums may not be added in longer chains than the
# large kernels' rules add them in, and how they run.
BOUNDED = [
    ((4762, 5194, 1208), "rectangle[4096x4096x608 ring; 4096x4096x600 ring; 4096x1098x1208 small"),
    ((2304, 8512, 2080), "small 64x64 ranges 1 fold 320 edge 96"),
]


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("shape,how", BOUNDED, ids=["x".join(map(str, c[0])) for c in BOUNDED])
def test_bounded_chains(lib, hip, oracle_mod, shape, how, form):
    assert route(*shape, form).startswith(how)
    check(lib, hip, oracle_mod, shape, form)


@pytest.mark.parametrize("form", sorted(FORMS))
@pytest.mark.parametrize("shape,want,want_nt", CASES + MANY,
                         ids=["x".join(map(str, c[0])) for c in CASES + MANY])
def test_tile(lib, hip, oracle_mod, shape, want, want_nt, form):
    m, n, k = shape
    rule = many if -(-m // 256) * -(-n // 256) >= 256 else plan
    tile, splits, fold = rule(m, n, k, form)
    assert (tile, splits > 1, 0 < fold < 1 << 27) == (want_nt if want_nt and form == "NT" else want)
    print(f"[kwave] tile {tile}, {splits} ranges, fold {fold}", flush=True)
    check(lib, hip, oracle_mod, shape, form)


def check(lib, hip, oracle_mod, shape, form):
    m, n, k = shape
    ops = FORMS[form]
    seed = m + 3 * n + 7 * k
    bias_axis = abi.BIAS_PER_ROW if (m + n) % 2 else abi.BIAS_PER_COLUMN
    relu = k % 2 == 1
    a = oracle_mod.fill_uniform(m * k, seed).reshape(m, k)
    b = oracle_mod.fill_uniform(k * n, seed + 1).reshape(k, n)
    c0 = oracle_mod.fill_uniform(m * n, seed + 2).reshape(m, n)
    bias = oracle_mod.fill_uniform(m if bias_axis == abi.BIAS_PER_ROW else n, seed + 3).astype(np.float32)
    fa, lda = padded_nan(a if ops[0] == abi.OP_N else a.T, 4)
    fb, ldb = padded_nan(b if ops[1] == abi.OP_N else b.T, 0)
    fc, ldc = padded_nan(c0, 8)
    print(f"[kwave] {form} {shape}: {route(m, n, k, form)}", flush=True)
    ptrs = [hip.alloc(x.nbytes) for x in (fa, fb, fc, bias)]
    s = hip.stream()
    outs = []
    try:
        hip.put(ptrs[0], fa)
        hip.put(ptrs[1], fb)
        hip.put(ptrs[3], bias)
        d = desc_for(ptrs[:3], m, n, k, ops,
                     (lda, ldb, ldc), 1.5, -0.5, ptrs[3], bias_axis, relu)
        for _ in range(2):
            hip.put(ptrs[2], fc)
            assert lib.ext.sgemm_device(ctypes.byref(d), s) == abi.SUCCESS
            hip.sync(s)
            outs.append(hip.get(ptrs[2], fc.size).reshape(n, ldc))
    finally:
        for p in ptrs:
            hip.free(p)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    assert np.array_equal(outs[0][:, m:].view(np.uint32), fc[:, m:].view(np.uint32))
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    add = bias[:, None] if bias_axis == abi.BIAS_PER_ROW else bias[None, :]
    ref = 1.5 * (a64 @ b64) - 0.5 * c0 + add
    ref = np.maximum(ref, 0.0) if relu else ref
    bound = 4 * k * 2.0 ** -24 * (1.5 * (np.abs(a64) @ np.abs(b64)) + 0.5 * np.abs(c0) + np.abs(add)) + 1e-30
    assert np.all(np.abs(outs[0][:, :m].T - ref) <= bound)
