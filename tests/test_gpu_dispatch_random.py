"""Seeded random shapes across the launch rules, on the MI355X through the C
ABI (the extension's sgemm_device on device memory), every element checked.

Shapes are drawn until each route of a launch (kernels::route) has two of them:
small tiles unsplit and with K split over workgroups, deep interior launches
split on the ring kernels, the tail split, the edge split with its interior on
the ring kernels and on small tiles, the rectangle of whole rounds in one pass
of K and in several, the K remainder, whole ragged launches on the ring kernels'
edge instances, whole rounds on the ring kernels and odd K on the general kernel;
in random N/T forms.
Operands are the analytic pattern (examples' gemm_bench pattern: exact in FP32
for these K), so every element of C must equal its closed form bit for bit,
whichever split, order of ranges or part computed it."""
import ctypes

import numpy as np
import pytest

import xvram_amd as xv
from xvram_amd import abi

from gemm_cases import route
from test_gpu_sgemm_device import FORMS, Hip, desc_for, padded
from test_gpu_tail_split import pattern_stored, synth  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu


def log(msg):
    print(f"[dispatch] {msg}", flush=True)


ROUTES = ["small unsplit", "small split", "many small", "ring split", "tail split",
          "edge split ring", "edge split small", "rectangle", "rectangle in passes", "k remainder",
          "edge ring", "ring", "general"]


def kind_of(m, n, k, form):
    how = route(m, n, k, form)
    if how.startswith("small"):
        if -(-m // 256) * -(-n // 256) >= 256:
            return "many small"
        return "small unsplit" if " ranges 1 " in how else "small split"
    if how.startswith("rectangle["):
        parts = how[10:].split("; ")
        return "rectangle in passes" if parts[1].split("x")[:2] == parts[0].split("x")[:2] else "rectangle"
    if how.startswith("edge split["):
        return "edge split " + how[11:].split(" ")[1].rstrip(";")
    return how.split("[")[0] if "[" in how else " ".join(w for w in how.split(" ") if w.isalpha())


def make_cases(seed=4242, each=2):
    rng = np.random.default_rng(seed)
    wanted = {r: each for r in ROUTES}
    cases = []
    while any(wanted.values()):
        if wanted["ring split"] and rng.random() < 0.2:  # at least 4096 deep on nearly every CU
            m, n, k = 256 * int(rng.integers(24, 33)), 256 * int(rng.integers(2, 5)), 8 * int(rng.integers(1024, 1300))
        elif rng.random() < 0.2:
            m, n, k = (int(v) for v in rng.integers(300, 3500, 3))
        else:
            m, n, k = (int(v) for v in rng.integers(2048, 5600, 3))
            k //= 2
        if rng.random() < 0.4:
            m, n = m // 256 * 256, n // 256 * 256
        if rng.random() < 0.6:
            k = k // 8 * 8
        if min(m, n, k) == 0:
            continue
        form = sorted(FORMS)[int(rng.integers(0, 4))]
        kind = kind_of(m, n, k, form)
        if wanted.get(kind):
            wanted[kind] -= 1
            cases.append((kind, m, n, k, form))
    return cases


CASES = make_cases()


@pytest.fixture(scope="module")
def lib():
    return xv.load()


@pytest.mark.parametrize("kind,m,n,k,form", CASES,
                         ids=[f"{c[0].replace(' ', '-')}-{c[1]}x{c[2]}x{c[3]}-{c[4]}" for c in CASES])
def test_dispatch_pattern_exact(lib, synth, oracle_mod, kind, m, n, k, form):
    ops = FORMS[form]
    a_st = pattern_stored(synth, "a", *((m, k) if ops[0] == abi.OP_N else (k, m)),
                          ops[0] == abi.OP_T)
    b_st = pattern_stored(synth, "b", *((k, n) if ops[1] == abi.OP_N else (n, k)),
                          ops[1] == abi.OP_T)
    a_flat, lda = padded(a_st)
    b_flat, ldb = padded(b_st)
    c_flat, ldc = padded(np.full((m, n), np.nan, np.float32))  # beta 0: C is never read
    hip = Hip()
    pa, pb, pc = hip.alloc(a_flat.nbytes), hip.alloc(b_flat.nbytes), hip.alloc(c_flat.nbytes)
    s = hip.stream()
    try:
        hip.put(pa, a_flat)
        hip.put(pb, b_flat)
        hip.put(pc, c_flat)
        d = desc_for((pa, pb, pc), m, n, k, ops, (lda, ldb, ldc))
        assert lib.ext.sgemm_device(ctypes.byref(d), ctypes.c_void_p(s)) == abi.SUCCESS
        hip.sync(s)
        got = hip.get(pc, c_flat.size).reshape(n, ldc)[:, :m].T
    finally:
        for p in (pa, pb, pc):
            hip.free(p)
        hip.close()
    expect = oracle_mod.pattern_expected_matrix(m, n, k).astype(np.float32)
    bad = int(np.count_nonzero(got != expect))
    log(f"{kind} {m}x{n}x{k} {form}: {bad} of {m * n} differ")
    assert bad == 0
