"""A few tokens on the matrix cores (few.hip), as hq_phase runs them: every (row, token) bit for bit the oracle's token
kernel, at the edges of its tiles (16 rows, 32 of ternary and binary; 16 to 64 tokens), of its stages (256 or 512 values
of a row), of its rule (the fewest and most tokens it takes, few long rows), with groups past the fours, with scales that allow no
16-byte loads, jobs of several row counts and both correction forms in one call, and no word outside the outputs
written."""
import numpy as np
import pytest

from gpu_util import Arena, first_difference, same_bits
from models import F
from streams import pack6, pack_ternary

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arena():
    return Arena(1 << 28)


@pytest.fixture(autouse=True)
def fresh(arena):
    arena.reset()
    yield


def matrix(rng, oracle, kind, rows, n):
    """a matrix's packed bytes, scales, corrections, and f(bytes, scales of a token) -> its rows' outputs"""
    ng = n // 32
    if kind in ("matmul_t2r", "matmul_b1r"):
        if kind == "matmul_t2r":
            w = pack_ternary(rng.integers(0, 3, rows * n).astype(np.uint8))
        else:
            w = rng.integers(0, 256, rows * n // 8).astype(np.uint8)
        ws = (rng.standard_normal(rows * (n // 128)) * 0.01).astype(np.float16).view(np.uint16)
        product = oracle.matmul_t2r if kind == "matmul_t2r" else oracle.matmul_b1r
        return w, ws, None, lambda q, s: product(q, s, w, ws, n)
    ws = (rng.standard_normal(rows * ng) * 0.02 / 127).astype(F)
    if kind == "matmul_q6r":
        w = pack6((4 * rng.integers(-32, 32, rows * n)).astype(np.int8))
        wc = oracle.six_sums(w)
    else:
        w = rng.integers(-128, 128, rows * n).astype(np.int8)
        wc = oracle.int8_sums(w)
    product = oracle.matmul_q6r if kind == "matmul_q6r" else oracle.matmul_q8r
    return w, ws, wc, lambda q, s, c=None: product(q, s, w, ws, wc if c is None else c, n)


CASES = [("matmul_q8r", n, t, 0) for n in (32, 96, 288, 512, 1056, 1664) for t in (5, 16, 17, 33, 48, 64, 96)] + \
        [("matmul_q6r", n, t, 0) for n in (32, 288, 512, 1664) for t in (5, 16, 33, 49, 64)] + \
        [(k, n, t, 4) for k in ("matmul_q8r", "matmul_q6r") for n in (32, 512, 1664) for t in (5, 33)] + \
        [(k, n, t, 0) for k in ("matmul_t2r", "matmul_b1r") for n in (128, 384, 512, 1664) for t in (3, 16, 17, 33, 160, 400)] + \
        [("matmul_q8r", 288, 130, 0), ("matmul_q8r", 512, 130, 4), ("matmul_q6r", 288, 130, 0),  # gemm.hip's tiles of several jobs
         ("matmul_t2r", 384, 420, 0), ("matmul_b1r", 384, 420, 0)] + \
        [("matmul_q8r", 512, 128, 0), ("matmul_q6r", 512, 128, 0)] + \
        [(k, 16384, t, 0) for k in ("matmul_q8r", "matmul_q6r", "matmul_t2r", "matmul_b1r") for t in (7, 8)]  # few long rows: 8
#                                       tokens are cheaper in one launch of the token kernel, 7 (two launches) on the tiles


@pytest.mark.parametrize("kind,n,tokens,shift", CASES)
def test_few_tokens(pkg, arena, oracle, kind, n, tokens, shift):
    """shift: the bytes that int8's and int6's scales lie past 16-byte places (the narrow loads; int8's xs too)"""
    signs = kind in ("matmul_t2r", "matmul_b1r")
    from pyodide_llm_amd import jobs
    rng = np.random.default_rng(n * 7 + tokens)
    ng = n // 32
    x = (rng.standard_normal((tokens, n)) * np.exp(rng.uniform(-3, 3, (tokens, 1)))).astype(F)
    frame = (n + 8 * ng + 16 + 15) // 16 * 16
    acts = np.zeros((tokens, frame), np.uint8)
    ready = []
    for t in range(tokens):
        q, s = oracle.quantize_x(x[t], 0 if signs else 64)
        if signs:
            q, s = oracle.interleave(q.view(np.int8), s)
        ready.append((q, s))
        acts[t, :n] = q.view(np.uint8)
        acts[t, n + shift:n + shift + s.nbytes] = np.ascontiguousarray(s).view(np.uint8)
    a = arena.put(acts)
    table, checks = [], []
    for rows, form in ((33, "derived"), (1, "wc"), (16, "wc"), (50, "moved"), (7, "derived")):
        w, ws, wc, product = matrix(rng, oracle, kind, rows, n)
        os = 4 * rows + 8
        out = arena.alloc(tokens * os + 64, fill=np.full((tokens * os + 64) // 4, -7, F))
        wsa = arena.alloc(ws.nbytes + 16) + (0 if signs else shift)
        arena.write(wsa, ws)
        c = None if signs or form == "derived" else wc if form == "wc" else (wc + rng.integers(-9, 9, wc.size)).astype(np.int32)
        table.append(jobs.job(kind, out, a, a + n + shift, arena.put(w), wsa, arena.put(c) if c is not None else 0, n,
                              rows=rows, count=tokens, os=os, as_=frame, bs=frame))
        checks.append((rows, os, out, product, c))
    L = pkg.library()
    assert jobs.phase(L, table) == 0, L.hq_last_error_message()
    for rows, os, out, product, c in checks:
        got = arena.get(out, F, (tokens * os + 64) // 4)
        want = np.full_like(got, -7)
        for t, (q, s) in enumerate(ready):
            want[t * os // 4:t * os // 4 + rows] = product(q, s) if c is None else product(q, s, c)
        assert same_bits(got, want), f"{rows} rows: {first_difference(got, want)}"
