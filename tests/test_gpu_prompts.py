"""The matrix cores' prompt tiles (gemm.hip) above the token counts that the few-token tiles take (128 of int8 and int6, 400
of ternary and binary), through hq_phase: several jobs a launch, of more than one row tile each, both correction forms, rows
of one group to many rounds of a tile's ring, and both ways of loading the scales; and these, the few-token tiles (few.hip)
and the token kernel with infinite and NaN scales, of which none may reach a row or token beside its own."""
import numpy as np
import pytest

from gpu_util import Arena, first_difference, same_bits
from models import F
from test_gpu_few import matrix

pytestmark = pytest.mark.gpu
SIGNS = ("matmul_t2r", "matmul_b1r")


@pytest.fixture(scope="module")
def arena():
    return Arena(1 << 28)


@pytest.fixture(autouse=True)
def fresh(arena):
    arena.reset()
    yield


def plain_nan(v):
    """any NaN as one"""
    v = np.array(v, F)
    v[np.isnan(v)] = np.nan
    return v


def check(pkg, arena, oracle, kind, n, tokens, rows, shift=0, special=False):
    from pyodide_llm_amd import jobs
    signs = kind in SIGNS
    rng = np.random.default_rng(n * 7 + tokens + special)
    ng = n // 32
    x = (rng.standard_normal((tokens, n)) * np.exp(rng.uniform(-3, 3, (tokens, 1)))).astype(F)
    frame = (n + 8 * ng + 16 + 15) // 16 * 16
    acts = np.zeros((tokens, frame), np.uint8)
    ready = []
    for t in range(tokens):
        q, s = oracle.quantize_x(x[t], 0 if signs else 64)
        if special and t in (1, 2):
            s[0 if t == 2 else ng - 1] = np.nan if t == 2 else np.inf
        if signs:
            q, s = oracle.interleave(q.view(np.int8), s)
        ready.append((q, s))
        acts[t, :n] = q.view(np.uint8)
        acts[t, n + shift:n + shift + s.nbytes] = np.ascontiguousarray(s).view(np.uint8)
    a = arena.put(acts)
    table, checks = [], []
    for i, r in enumerate(rows):
        w, ws, wc, product = matrix(rng, oracle, kind, r, n)
        if special:  # (the product holds ws itself)
            of = ws.view(np.float16) if signs else ws
            of = of.reshape(r, -1)
            of[1::4, 0], of[2::4, -1], of[3::8, 0] = np.inf, np.nan, -np.inf
        os = 4 * r + 8
        out = arena.alloc(tokens * os + 64, fill=np.full((tokens * os + 64) // 4, -7, F))
        wsa = arena.alloc(ws.nbytes + 16) + (0 if signs else shift)
        arena.write(wsa, ws)
        c = None if signs or i % 2 else (wc + rng.integers(-9, 9, wc.size)).astype(np.int32)
        table.append(jobs.job(kind, out, a, a + n + shift, arena.put(w), wsa, arena.put(c) if c is not None else 0, n, rows=r,
                              count=tokens, os=os, as_=frame, bs=frame))
        checks.append((r, os, out, product, c))
    L = pkg.library()
    assert jobs.phase(L, table) == 0, L.hq_last_error_message()
    some = range(tokens) if tokens * n < 1 << 20 else sorted({0, 1, 2, 63, 64, tokens - 2, tokens - 1})
    for r, os, out, product, c in checks:
        got = arena.get(out, F, (tokens * os + 64) // 4)
        assert np.all(got[tokens * os // 4:] == -7)
        got = got[:tokens * os // 4].reshape(tokens, -1)
        assert np.all(got[:, r:] == -7)
        for t in some:
            want = product(*ready[t]) if c is None else product(*ready[t], c)
            mine, theirs = plain_nan(got[t, :r]), plain_nan(want)
            assert same_bits(mine, theirs), f"{r} rows, token {t}: {first_difference(mine, theirs)}"
            if special and t > 2:  # (a float16's all-ones exponent is a value like the others: 65536 and more)
                assert np.isfinite(theirs[::4]).all() and (signs or not np.isfinite(theirs[1::4]).any())


PROMPTS = [(k, n, t, s) for k in ("matmul_q8r", "matmul_q6r") for n, t, s in ((32, 129, 0), (416, 193, 0), (512, 129, 0), (512, 200, 4),
                                                                         (1664, 257, 0), (4096, 130, 0))] + \
          [(k, n, t, 0) for k in SIGNS for n, t in ((128, 401), (1152, 401), (2560, 449), (17408, 401))]


@pytest.mark.parametrize("kind,n,tokens,shift", PROMPTS)
def test_prompt_tiles_of_several_jobs(pkg, arena, oracle, kind, n, tokens, shift):
    """rows: more than one tile (of 32, 64, 96 or 128) and a ragged end, jobs with and without corrections in turn"""
    rows = (100, 33) if n > 4096 else (300, 1, 130, 65, 97)
    check(pkg, arena, oracle, kind, n, tokens, rows, shift)


@pytest.mark.parametrize("kind", ["matmul_q8r", "matmul_q6r", "matmul_t2r", "matmul_b1r"])
@pytest.mark.parametrize("n", [384, 640, 1664])
@pytest.mark.parametrize("tokens", [4, 13, 33, 130, 401])
def test_infinite_and_nan_scales(pkg, arena, oracle, kind, n, tokens):
    """rows whose neighbours' scales are infinite or NaN end in the middle of a stage (640: 5 groups of 128)"""
    check(pkg, arena, oracle, kind, n, tokens, (70, 37), special=True)


@pytest.mark.parametrize("kind", ["matmul_q8r", "matmul_q6r"])
@pytest.mark.parametrize("n", [32, 288, 416])
@pytest.mark.parametrize("tokens", [5, 33, 130])
def test_infinite_and_nan_scales_past_the_fours(pkg, arena, oracle, kind, n, tokens):
    check(pkg, arena, oracle, kind, n, tokens, (70, 37), special=True)
