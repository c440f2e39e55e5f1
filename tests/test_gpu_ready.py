"""The activations readied in one launch: quantize_x's bytes and scales with interleave's planes and sums (ternary) or
sums_x's sums (llama.cpp's blocks), as hq_matmuls leaves them in the jobs' a / b, byte for byte against the oracle, at
widths that end inside a block of 1024 values; and quantize_x where its addresses do not take 16-byte loads."""
import numpy as np
import pytest

from gpu_util import Arena, same_bits
from models import F
from streams import pack6

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def arena():
    return Arena(1 << 27)


@pytest.fixture(autouse=True)
def fresh(arena):
    arena.reset()
    yield


def activations(rng, tokens, n):
    """groups of every size, and one each of zeros, -0, an infinity, a NaN in groupMax's lane 0 and in another, and
    subnormals"""
    x = (rng.standard_normal((tokens, n)) * np.exp(rng.uniform(-8, 8, (tokens, n // 32, 1))).repeat(32, 1).reshape(
        tokens, n)).astype(F)
    x[0, :32] = 0.0
    x[0, 5] = -0.0
    x[-1, 32 + 6] = np.inf
    x[-1, 64 + 4] = np.nan
    x[0, 96 + 7] = np.nan
    x[0, 97] = 2.0 ** -140
    return x


@pytest.mark.parametrize("kind,n", [("matmul_t2r", 128), ("matmul_t2r", 1152), ("matmul_t2r", 17408),
                                    ("matmul_sbr", 256), ("matmul_sbr", 1280), ("matmul_q8r", 128),
                                    ("matmul_q8r", 1056)])
@pytest.mark.parametrize("tokens", [1, 3])
def test_readied_in_one_launch(pkg, arena, oracle, kind, n, tokens):
    from pyodide_llm_amd import jobs
    rng = np.random.default_rng(n + tokens)
    x = activations(rng, tokens, n)
    frame = 2 * n + 64
    acts = arena.alloc(tokens * frame, fill=np.full(tokens * frame, 0xAA, np.uint8))
    w = arena.put(np.zeros(4 * n, np.uint8))  # a row of any packing, and its scales or tables
    out = arena.alloc(4 * tokens)
    table = [jobs.job(kind, out, acts, acts + n, w, arena.put(np.zeros(40000, np.uint8)),
                      12 if kind == "matmul_sbr" else 0, n, rows=1, count=tokens, os=4, as_=frame, bs=frame)]
    L = pkg.library()
    assert jobs.matmuls(L, arena.put(x), 4 * n, table) == 0, L.hq_last_error_message()
    got = arena.get(acts, np.uint8, tokens * frame).reshape(tokens, frame)
    for t in range(tokens):
        q, scales = oracle.quantize_x(x[t], 64 if kind == "matmul_q8r" else 0)
        area = scales
        if kind == "matmul_t2r":
            q, area = oracle.interleave(q.view(np.int8), scales)
        elif kind == "matmul_sbr":
            area = oracle.sums_x(q.view(np.int8), scales)
        want = np.full(frame, 0xAA, np.uint8)
        bytes_ = np.ascontiguousarray(area).view(np.uint8)
        want[:n] = q.view(np.uint8)
        want[n:n + bytes_.size] = bytes_
        # (a NaN's own bits are not compared)
        mine, theirs = got[t].copy(), want
        for row in (mine, theirs):
            s = row[n:n + n // 8].view(F)
            s[np.isnan(s)] = np.nan
        assert np.array_equal(mine, theirs), (t, np.nonzero(mine != theirs)[0][:8])


@pytest.mark.parametrize("x_off,xq_off", [(4, 0), (0, 1), (8, 2), (0, 4)])
def test_quantize_x_anywhere(pkg, arena, oracle, x_off, xq_off):
    rng = np.random.default_rng(x_off + 16 * xq_off)
    n = 1056
    x = rng.standard_normal(n).astype(F)
    ax = arena.alloc(4 * n + 16) + x_off
    arena.write(ax, x)
    xq = arena.alloc(n + 16, fill=np.full(n + 16, 0xAA, np.uint8)) + xq_off
    xs = arena.alloc(4 * (n // 32))
    assert pkg.library().hq_quantize_x_ex(xq, xs, ax, n, 64, None) == 0
    want_q, want_s = oracle.quantize_x(x, 64)
    got = arena.get(xq - xq_off, np.uint8, n + 16)
    assert np.array_equal(got[xq_off:xq_off + n], want_q)
    assert np.all(got[:xq_off] == 0xAA) and np.all(got[xq_off + n:] == 0xAA)
    assert same_bits(arena.get(xs, F, n // 32), want_s)


@pytest.mark.parametrize("kind,n", [("matmul_q8r", 512), ("matmul_q6r", 1536), ("matmul_sbr", 1280)])
@pytest.mark.parametrize("place", ["apart", "over x"])
def test_one_token_from_its_float32_input(pkg, arena, oracle, kind, n, place):
    """one token's products with the input readied in their own launch; outputs over the input take the input apart first
    (the launch's blocks would read what others of it write)"""
    from pyodide_llm_amd import jobs
    rng = np.random.default_rng(n)
    ng = n // 32
    x = rng.standard_normal(n).astype(F)
    rows = (70, 33)
    acts = arena.alloc(8 * n, fill=np.zeros(8 * n, np.uint8))
    ax, b = arena.put(x), acts + n
    outs = [ax if place == "over x" else arena.alloc(4 * r, fill=np.full(r, -7, F)) for r in rows]
    if place == "over x":
        outs[1] = ax + 4 * rows[0]
    q, scales = oracle.quantize_x(x, 0 if kind == "matmul_sbr" else 64)
    table, wants = [], []
    if kind == "matmul_sbr":
        import blocks_model as bm
        row = bm.codebooks(rng)
        tab, area = oracle.sb_tables(row), arena.alloc(34992)
        assert pkg.library().hq_sb_tables_ex(area, arena.put(row), None) == 0
        acts_area = oracle.sums_x(q.view(np.int8), scales)
    for r, out in zip(rows, outs):
        if kind == "matmul_sbr":
            w = bm.random_blocks(rng, 12, r * (n // 256))
            args = (arena.put(w), area, 12)
            wants.append(oracle.matmul_sbr(q.view(np.int8), acts_area, w, tab, n, 12))
        else:
            ws = (np.abs(rng.standard_normal(r * ng)) * 0.02).astype(F)
            if kind == "matmul_q6r":
                w = pack6((4 * rng.integers(-32, 32, r * n)).astype(np.int8))
                wc, product = oracle.six_sums(w), oracle.matmul_q6r
            else:
                w = rng.integers(-128, 128, r * n).astype(np.int8)
                wc, product = oracle.int8_sums(w), oracle.matmul_q8r
            args = (arena.put(w), arena.put(ws), arena.put(wc))
            wants.append(product(q, scales, w, ws, wc, n))
        table.append(jobs.job(kind, out, acts, b, *args, n, rows=r))
    L = pkg.library()
    assert jobs.matmuls(L, ax, 4 * n, table) == 0, L.hq_last_error_message()
    for out, r, want in zip(outs, rows, wants):
        assert same_bits(arena.get(out, F, r), want)
    assert np.array_equal(arena.get(acts, np.uint8, n), q.view(np.uint8))
    assert same_bits(arena.get(b, F, ng), scales)


def special(rng, n):
    """a token's input with groups of every size, zeros, a NaN and an infinity (in groups the outputs of which are then NaN)"""
    return activations(rng, 1, max(n, 128))[0, :n] if n >= 128 else rng.standard_normal(n).astype(F)


def alike(got, want):
    """the same bits, any NaN as any other"""
    nan = np.isnan(want)
    return np.array_equal(np.isnan(got), nan) and same_bits(got[~nan], want[~nan])


BLOCK_READY = [(t, n) for t in ("Q2_K", "Q4_K", "IQ2_XXS", "IQ2_XS", "IQ2_S", "IQ3_XXS", "IQ3_S", "IQ1_S", "IQ1_M", "IQ4_XS")
               for n in (256, 4352, 8192, 8448)] + [("Q4_K", 1280), ("Q4_K", 14336), ("Q4_K", 14592)]


@pytest.mark.parametrize("name,n", BLOCK_READY)
@pytest.mark.parametrize("shift,form", [(0, "plain"), (2, "special"), (0, "over x")])
def test_one_token_of_blocks_from_its_float32_input(pkg, arena, oracle, name, n, shift, form):
    """the same for llama.cpp's blocks: rows of 16 and 64 lanes, one round and several of the block's quantization, blocks
    that start on 16 bytes and not, on both sides of the width it is done to; the bytes, scales and sums left in a / b"""
    import blocks_model as bm
    from pyodide_llm_amd import jobs
    t = jobs.BLOCK_TYPES[name][0]
    rng = np.random.default_rng(n + t)
    x = special(rng, n) if form == "special" else rng.standard_normal(n).astype(F)
    rows = (37, 9)
    acts = arena.alloc(2 * n, fill=np.full(2 * n, 0xAA, np.uint8))
    ax = arena.put(np.concatenate([x, np.zeros(64, F)]))
    outs = [arena.alloc(4 * r, fill=np.full(r, -7, F)) for r in rows]
    if form == "over x":
        outs = [ax, ax + 4 * rows[0]]
    q, scales = oracle.quantize_x(x, 0)
    area = oracle.sums_x(q.view(np.int8), scales)
    row = bm.codebooks(rng)
    tab, tables = oracle.sb_tables(row), arena.alloc(34992)
    L = pkg.library()
    assert L.hq_sb_tables_ex(tables, arena.put(row), None) == 0
    table, wants = [], []
    for r, out in zip(rows, outs):
        w = bm.random_blocks(rng, t, r * (n // 256))
        at = arena.alloc(w.size + 16) + shift
        arena.write(at, w)
        wants.append(oracle.matmul_sbr(q.view(np.int8), area, w, tab, n, t))
        table.append(jobs.job("matmul_sbr", out, acts, acts + n, at, tables, t, n, rows=r))
    assert jobs.matmuls(L, ax, 4 * n, table) == 0, L.hq_last_error_message()
    for out, r, want in zip(outs, rows, wants):
        assert alike(arena.get(out, F, r), want)
    got = arena.get(acts, np.uint8, 2 * n)
    left = np.ascontiguousarray(area).view(np.uint8)
    assert np.array_equal(got[:n], q.view(np.uint8))
    assert alike(got[n:n + n // 8].view(F), left[:n // 8].view(F))
    assert np.array_equal(got[n + n // 8:n + left.size], left[n // 8:])
    assert np.all(got[n + left.size:] == 0xAA)


@pytest.mark.parametrize("kind", ["matmul_q8r", "matmul_q6r"])
@pytest.mark.parametrize("n", [32, 96, 288, 512, 1536])
@pytest.mark.parametrize("form", ["wc", "derived"])
@pytest.mark.parametrize("values", ["plain", "special"])
@pytest.mark.parametrize("pairs", ["one a and b", "one a, two b"])
def test_one_token_of_int8_and_int6_from_its_float32_input(pkg, arena, oracle, kind, n, form, values, pairs):
    """the same for int8 and int6, corrections given and derived, with groups past the fours, of rows whose input's groups
    hold a NaN and an infinity; every job's a / b hold the readied activations after the call, also where two jobs of one a
    have a b each (which takes the input apart)"""
    from pyodide_llm_amd import jobs
    rng = np.random.default_rng(n)
    ng = n // 32
    x = special(rng, n) if values == "special" else rng.standard_normal(n).astype(F)
    q, scales = oracle.quantize_x(x, 64)
    a = arena.alloc(n + 16, fill=np.full(n + 16, 0xAA, np.uint8))
    bs = [arena.alloc(n // 8 + 16, fill=np.full(n // 8 + 16, 0xAA, np.uint8)) for _ in range(2)]
    table, wants = [], []
    for i, r in enumerate((37, 9)):
        ws = (rng.standard_normal(r * ng) * 0.02).astype(F)
        if kind == "matmul_q6r":
            w = pack6((4 * rng.integers(-32, 32, r * n)).astype(np.int8))
            wc, product = oracle.six_sums(w), oracle.matmul_q6r
        else:
            w = rng.integers(-128, 128, r * n).astype(np.int8)
            wc, product = oracle.int8_sums(w), oracle.matmul_q8r
        out = arena.alloc(4 * r, fill=np.full(r, -7, F))
        b = bs[i] if pairs == "one a, two b" else bs[0]
        table.append(jobs.job(kind, out, a, b, arena.put(w), arena.put(ws), arena.put(wc) if form == "wc" else 0, n, rows=r))
        wants.append((out, r, product(q, scales, w, ws, wc, n)))
    L = pkg.library()
    assert jobs.matmuls(L, arena.put(np.concatenate([x, np.zeros(64, F)])), 4 * n, table) == 0, L.hq_last_error_message()
    for out, r, want in wants:
        assert alike(arena.get(out, F, r), want)
    got = arena.get(a, np.uint8, n + 16)
    assert np.array_equal(got[:n], q.view(np.uint8)) and np.all(got[n:] == 0xAA)
    for b in bs[:2 if pairs == "one a, two b" else 1]:
        got = arena.get(b, np.uint8, n // 8 + 16)
        assert alike(got[:n // 8].view(F), scales) and np.all(got[n // 8:] == 0xAA)
