"""Kernels at the sizes where their tiling turns: one token more or less than a block or a
stage, head sizes around the padded ones, the first and last sizes of a dispatch's ranges.
References are the oracle or float64; every multi-token result is also compared bit for bit
with the same tokens taken one at a time or a few at a time.
"""

import ctypes as C

import numpy as np
import pytest

import oracle as O
from helpers import attend64, rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip(pkg):
    h = pkg.Hip(0)
    yield h
    h.close()


# blocks of 16 tokens in stages of 32 (head sizes to 64) or 16 (above), a ring of four stages;
# heads padded to 16, 32, 64, 128 or 256 rows
@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("m,heads,dh", [(15, 2, 64), (16, 2, 64), (17, 3, 64), (31, 1, 64), (33, 2, 64),
                                        (128, 2, 64), (161, 2, 64), (49, 2, 60), (47, 2, 33), (63, 3, 17),
                                        (16, 2, 16), (95, 1, 1), (34, 2, 65), (97, 1, 100), (15, 1, 129),
                                        (81, 1, 200), (65, 1, 256)])
def test_gla_blocks(hip, m, heads, dh, fp16):
    """Against the oracle (2e-6, the bound of test_gpu_ops.py; fp16 mode rounds every element
    and is compared with itself only), and the same bits one token at a time and in two calls."""
    rng = np.random.default_rng(m * 1000 + dh)

    def rnd(*shape, scale=1.0):
        return (rng.standard_normal(shape) * scale).astype(np.float32)

    q, k, v = rnd(m, heads, dh), rnd(m, heads, dh), rnd(m, heads, dh)
    q /= np.linalg.norm(q, axis=-1, keepdims=True)
    k /= np.linalg.norm(k, axis=-1, keepdims=True)
    dec, bias, s0 = rnd(m, heads), rnd(heads) - 3, rnd(heads, dh, dh, scale=0.1)
    hip.set_fp16(fp16)
    try:
        dq, dk, dv, dd, db = [hip.upload(t) for t in (q, k, v, dec, bias)]

        def run(cuts):
            ds, out = hip.upload(s0), []
            for a, b in zip(cuts, cuts[1:]):
                dy = hip.alloc((b - a) * heads * dh)
                hip.gla(dy.ptr, ds.ptr, dq.at(a * heads * dh), dk.at(a * heads * dh), dv.at(a * heads * dh),
                        dd.at(a * heads), db.ptr, b - a, heads, dh)
                out.append(dy.read())
            return np.concatenate(out), ds.read()

        y, s = run([0, m])
        for cuts in (list(range(m + 1)), [0, m // 3, m]):
            y2, s2 = run([c for i, c in enumerate(cuts) if i == 0 or c > cuts[i - 1]])
            assert np.array_equal(y, y2) and np.array_equal(s, s2)
        if not fp16:
            wy, ws = O.gla(s0, q, k, v, dec, bias, m, heads, dh)
            assert rel(y, wy) < 2e-6 and rel(s, ws) < 2e-6
    finally:
        hip.set_fp16(False)


# a query tile of 16 / group queries a workgroup, its segments on four waves (calls this short: longer
# ones are in test_attend_shared_tiles); 16-key tiles, 64-key segments, 256-key superblocks; rings
# shorter than a superblock, spans that start or end inside a tile
@pytest.mark.parametrize("pos,m,reach,gap,cap,heads,kh,dh", [
    (0, 2, O.USIZE_MAX, 0, 300, 2, 2, 64), (0, 64, O.USIZE_MAX, 0, 64, 1, 1, 64), (1000, 65, 100, 0, 165, 2, 2, 64),
    (255, 17, 256, 0, 512, 1, 1, 64), (513, 63, 49, 0, 112, 2, 1, 60), (300, 33, O.USIZE_MAX, 64, 400, 8, 1, 64),
    (77, 129, 15, 0, 144, 4, 2, 32), (2000, 16, 1024, 0, 1040, 3, 3, 16), (40, 100, 8, 0, 24 + 100, 2, 1, 4)])
def test_attend_tiles(hip, pos, m, reach, gap, cap, heads, kh, dh):
    """Against float64 (no further than twice the oracle's fp32 sums, as test_gpu_ops.py), and
    every query alone gives the same bits; slots no query sees hold NaN."""
    rng = np.random.default_rng(pos * 1000 + m)
    a = dict(pos=pos, m=m, reach=reach, gap=gap, cap=cap, heads=heads, key_heads=kh, dh=dh,
             scale=float(1 / np.sqrt(dh)))
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((m, heads, dh), (kh, cap, dh), (kh, cap, dh)))
    first, last = max(0, pos - reach + 1), max(0, pos + m - gap)
    unseen = sorted(set(range(cap)) - {p % cap for p in range(first // 16 * 16, (last + 15) // 16 * 16)})
    k[:, unseen] = v[:, unseen] = np.nan
    dq, dk, dv, dy, d1 = hip.upload(q), hip.upload(k), hip.upload(v), hip.alloc(q.size), hip.alloc(heads * dh)
    hip.attend(dy.ptr, dq.ptr, dk.ptr, dv.ptr, **a)
    got = dy.read().reshape(m, -1)
    for i in range(m):
        hip.attend(d1.ptr, dq.at(i * heads * dh), dk.ptr, dv.ptr, **dict(a, pos=pos + i, m=1))
        assert np.array_equal(d1.read(), got[i]), i
    want, exact = O.attend(q, k, v, **a), attend64(q, k, v, **a)
    assert rel(got.ravel(), exact) <= 2 * rel(want, exact) + 1e-7


# calls past the 1024 (query tiles x key heads x visible superblocks) from which query tiles share
# copied key tiles: head sizes in 1, 2 and 4 blocks of 16 and between them, 1 to 4 heads a key head, a
# gap, a ragged last group of tiles, rings shorter than a superblock
SHARED = [
    (5000, 300, 4096, 0, 4400, 12, 12, 64), (3000, 403, O.USIZE_MAX, 64, 3500, 3, 1, 60), (0, 3001, 150, 0, 200, 2, 2, 48),
    (700, 1030, 512, 100, 1600, 8, 2, 32), (30, 2500, 5, 0, 5, 1, 1, 24), (2000, 777, 1000, 0, 1777, 4, 4, 16),
    (2000, 777, 1000, 0, 900, 4, 4, 8)]


# (fp16 mode: the rings that it keeps in fp16)
@pytest.mark.parametrize("pos,m,reach,gap,cap,heads,kh,dh,fp16", [
    (*c, f) for c in SHARED for f in (False, True) if not f or (c[7] % 8 == 0 and c[4] >= 64)])
def test_attend_shared_tiles(hip, pos, m, reach, gap, cap, heads, kh, dh, fp16):
    """Against float64 (fp32: no further than twice the oracle's sums; fp16 mode: half a step of its
    rounding), and the bits of queries taken alone: the first, the last and some between."""
    rng = np.random.default_rng(pos + m + dh)
    a = dict(pos=pos, m=m, reach=reach, gap=gap, cap=cap, heads=heads, key_heads=kh, dh=dh, scale=0.25)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((m, heads, dh), (kh, cap, dh), (kh, cap, dh)))
    dt = 1 if dh <= 16 else 2 if dh <= 32 else 4
    hip.set_fp16(fp16)
    try:
        if fp16:
            q, k, v = (t.astype(np.float16).astype(np.float32) for t in (q, k, v))
        dk, dv = hip.alloc_cache(kh, cap, dh), hip.alloc_cache(kh, cap, dh)
        hip.upload_into(dk, k), hip.upload_into(dv, v)
        dq, dy, d1 = hip.upload(q), hip.alloc(q.size), hip.alloc(heads * dh)
        hip.set_timing(True)
        hip.attend(dy.ptr, dq.ptr, dk.ptr, dv.ptr, **a)
        got = dy.read().reshape(m, -1)
        assert hip.kernel_stat(f"slm_attn_pq{'16' if fp16 else ''}_{dt}")["launches"] == 1
        hip.set_timing(False)
        for i in sorted({0, 1, m - 2, m - 1, *range(15, m, max(1, m // 40))}):
            hip.attend(d1.ptr, dq.at(i * heads * dh), dk.ptr, dv.ptr, **dict(a, pos=pos + i, m=1))
            assert np.array_equal(d1.read(), got[i]), i
    finally:
        hip.set_timing(False)
        hip.set_fp16(False)
    exact = attend64(q, k, v, **a)
    err = rel(got.ravel(), exact)
    assert err <= (2.0 ** -11 + 2e-6 if fp16 else 2 * rel(O.attend(q, k, v, **a), exact) + 1e-7)


# a visible key or value that is infinite or NaN, in every attention kernel (one superblock)
@pytest.mark.parametrize("m,heads,dh,n", [(1, 2, 64, 250), (3, 2, 64, 250), (100, 160, 64, 250), (5, 2, 128, 250), (1, 2, 128, 250)])
@pytest.mark.parametrize("what", ["k nan", "k inf", "k -inf", "v inf", "v nan"])
def test_attend_visible_infinities(hip, m, heads, dh, n, what):
    """A score of -inf weighs nothing; a value's infinity or NaN reaches its own dim only; a score of
    +inf or NaN leaves its superblock out. The other heads are untouched."""
    rng = np.random.default_rng(n + m)
    q, k, v = (rng.standard_normal(s).astype(np.float32) for s in ((m, heads, dh), (heads, n, dh), (heads, n, dh)))
    q[:, :, 0] = np.abs(q[:, :, 0]) + 0.5  # (an infinite key coordinate gives an infinite score of its sign)
    a = dict(pos=n - m, m=m, reach=O.USIZE_MAX, gap=0, cap=n, heads=heads, key_heads=heads, dh=dh, scale=0.125)
    dq, dk, dv, dy = hip.upload(q), hip.upload(k), hip.upload(v), hip.alloc(q.size)
    hip.attend(dy.ptr, dq.ptr, dk.ptr, dv.ptr, **a)
    plain = dy.read().reshape(m, heads, dh)
    at, val = 70, {"nan": np.nan, "inf": np.inf, "-inf": -np.inf}[what[2:]]
    (k if what[0] == "k" else v)[0, at, 0 if what[0] == "k" else 3] = val
    hip.upload_into(dk, k), hip.upload_into(dv, v)
    hip.attend(dy.ptr, dq.ptr, dk.ptr, dv.ptr, **a)
    got = dy.read().reshape(m, heads, dh)
    same = np.array_equal(got[:, 1:], plain[:, 1:])
    assert same
    if what == "k -inf":
        k[0, at, 0], q64 = 0.0, q.astype(np.float64)
        s = np.where(np.arange(n) == at, -np.inf, q64[:, 0] @ k[0].T.astype(np.float64) * 0.125)
        s[np.arange(n)[None] > np.arange(n - m, n)[:, None]] = -np.inf
        p = np.exp(s - s.max(1, keepdims=True))
        err = rel(got[:, 0], p / p.sum(1, keepdims=True) @ v[0].astype(np.float64))
        assert err < 2e-6
    elif what[0] == "k":
        none = (got[:, 0] == 0).all()
        assert none
    else:
        bad = np.isnan(got[:, 0, 3]) if what == "v nan" else got[:, 0, 3] == np.inf
        rest = [d for d in range(dh) if d != 3]
        same = np.array_equal(got[:, 0, rest], plain[:, 0, rest])
        assert bad.all() and same


# one token, a query tile's segments on waves of their own, query tiles sharing key tiles, the general kernel
@pytest.mark.parametrize("m,heads,dh", [(1, 2, 64), (3, 2, 64), (256, 12, 64), (40, 1, 32), (5, 1, 128), (1, 1, 128)])
def test_attend_weights_of_large_scores(hip, m, heads, dh):
    """Scores near +-100, exact in 32 bits, 0 to 4 under their maximum: a weight's exponent is at most 5.8
    in powers of two, off by half its last step (1.7e-7 of the weight) and the exponential's ulp
    (1.2e-7), whatever the scores' own size; with sums and values 5e-7 of the largest result."""
    rng = np.random.default_rng(dh + m)
    n = 4096
    q, k = np.zeros((m, heads, dh), np.float32), np.zeros((heads, n, dh), np.float32)
    q[:, :, 0] = 1.0
    k[:, :, 0] = rng.choice([-800.0, 800.0], (heads, 1)) - np.round(rng.random((heads, n)) * 32 * 512) / 512
    v = rng.standard_normal((heads, n, dh)).astype(np.float32)
    a = dict(pos=n - m, m=m, reach=O.USIZE_MAX, gap=0, cap=n, heads=heads, key_heads=heads, dh=dh, scale=0.125)
    dq, dk, dv, dy = hip.upload(q), hip.upload(k), hip.upload(v), hip.alloc(q.size)
    hip.attend(dy.ptr, dq.ptr, dk.ptr, dv.ptr, **a)
    err = rel(dy.read(), attend64(q, k, v, **a))
    assert err < 5e-7


@pytest.mark.parametrize("m,dh", [(1, 64), (40, 64), (40, 60), (5, 33), (3, 129)])
@pytest.mark.parametrize("what", ["q", "k", "v", "s"])
def test_gla_infinities(hip, m, dh, what):
    """NaN and infinities come out where the oracle has them, the other elements within 2e-6."""
    rng, heads = np.random.default_rng(m + dh), 2
    q, k, v = (rng.standard_normal((m, heads, dh)).astype(np.float32) for _ in range(3))
    s, dec, bias = (rng.standard_normal(n).astype(np.float32) for n in ((heads, dh, dh), (m, heads), heads))
    if what == "s":
        s[0, 3, 5] = np.inf
    else:
        dict(q=q, k=k, v=v)[what][m // 2, 0, 5] = np.nan
    b = [hip.upload(t) for t in (s, q, k, v, dec, bias)]
    dy = hip.alloc(q.size)
    hip.gla(dy.ptr, *(t.ptr for t in b), m, heads, dh)
    for got, want in zip((dy.read(), b[0].read()), O.gla(s, q, k, v, dec, bias, m, heads, dh)):
        want = want.ravel()
        fin = np.isfinite(want)
        same = np.array_equal(got[~fin], want[~fin], equal_nan=True)
        err = rel(got[fin], want[fin])
        assert same and err < 2e-6


@pytest.mark.parametrize("rows,cols,m", [(100, 768, 5), (100, 768, 20), (100, 768, 40), (100, 770, 5), (100, 770, 20),
                                         (100, 770, 40), (100, 3072, 5), (9, 100, 33)])
def test_linear_infinities(hip, rows, cols, m):
    """An infinite weight reaches its row, an infinite input its token, NaN where both meet."""
    rng = np.random.default_rng(rows + m)
    w, x = (rng.standard_normal(s).astype(np.float32) for s in ((rows, cols), (m, cols)))
    w[2, 37], w[4, 1], x[3, cols - 1] = np.inf, np.nan, -np.inf
    dw, dx, dy = hip.upload(w), hip.upload(x), hip.alloc(rows * m)
    hip.linear(dy.ptr, dw.ptr, rows, cols, dx.ptr, m)
    with np.errstate(invalid="ignore"):
        want = (x.astype(np.float64) @ w.T.astype(np.float64)).ravel()
    got, fin = dy.read(), np.isfinite(want)
    same = np.array_equal(got[~fin], want[~fin], equal_nan=True)
    err = rel(got[fin], want[fin])
    assert same and err < 2e-6


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("d,kh,dh,cap,shift,logn", [(768, 4, 64, 300, True, True), (768, 4, 64, 128, False, True),
                                                    (64, 1, 16, 64, True, False), (128, 2, 48, 65, False, False)])
def test_global_layer_input(hip, d, kh, dh, cap, shift, logn, fp16):
    """A global layer's one-token input (two matrices on one input, a scaled output, stores out
    of parts of an output, the kept row's matrix moved ahead) leaves the bits of one launch per
    operation in every buffer, in fewer kernels, step after step."""
    rng = np.random.default_rng(d + cap)
    hip.set_fp16(fp16)
    try:
        kd = kh * dh
        up = lambda *s, scale=1.0: hip.upload((rng.standard_normal(s) * scale).astype(np.float32))  # noqa: E731
        inv = hip.upload(np.ones(8, np.float32))
        cs, sn = hip.alloc(8), hip.alloc(8)
        wq, wkv, wm, g = up(d, d, scale=0.05), up(2 * kd, d, scale=0.05), up(d, 2 * d, scale=0.05), up(d)
        x, prev, up2 = up(d), up(d), up(4 * d)
        bufs = dict(n=hip.alloc(d), q=hip.alloc(d), q2=hip.alloc(d), kv=hip.alloc(2 * kd), kv2=hip.alloc(2 * kd),
                    sh=hip.alloc(d), t=hip.alloc(d), mid=hip.alloc(2 * d), h=hip.alloc(d), prev=prev,
                    k=hip.alloc_cache(kh, cap, dh), v=hip.alloc_cache(kh, cap, dh))
        b = {n: t.ptr for n, t in bufs.items()}
        first = prev.read()

        def step(pos, fuse):
            hip.set_fusion(fuse)
            hip.rope_table(cs.ptr, sn.ptr, inv.ptr, pos, 1, 8)
            hip.silu_mul(b["mid"], up2.at(0), up2.at(2 * d), 2 * d)
            hip.linear(b["h"], wm.ptr, d, 2 * d, b["mid"], 1)
            hip.add(b["t"], x.ptr, b["h"], d)
            hip.rms(b["n"], b["t"], g.ptr, 1, d, 1e-6)
            hip.linear(b["q"], wq.ptr, d, d, b["n"], 1)
            hip.linear(b["kv"], wkv.ptr, 2 * kd, d, b["n"], 1)
            if logn:
                hip.scale_rows(b["q2"], b["q"], np.array([0.37 + pos], np.float32), d)
            if shift:
                hip.shift(b["sh"], b["prev"], b["n"], 1, d)
                hip.linear(b["kv2"], wkv.ptr, 2 * kd, d, b["sh"], 1)
                hip.copy(b["prev"], b["n"], d)
            hip.store(b["k"], b["kv2" if shift else "kv"], pos, 1, cap, kh, dh)
            hip.store(b["v"], bufs["kv"].at(kd), pos, 1, cap, kh, dh)
            hip.flush([t.ptr for t in bufs.values()])
            return hip.last_plan()["kernels"]

        got, kernels = {}, {}
        for fuse in (False, True):
            hip.upload_into(prev, first)
            for t in ("k", "v"):
                hip.upload_into(bufs[t], np.zeros(kh * cap * dh, np.float32))
            kernels[fuse] = [step(pos, fuse) for pos in (3, 4, cap - 1, cap, 2 * cap + 7)]
            got[fuse] = {n: t.read() for n, t in bufs.items()}
        for n in got[False]:
            assert np.array_equal(got[False][n], got[True][n]), n
        assert max(kernels[True]) <= 5 < min(kernels[False])
    finally:
        hip.set_fusion(True)
        hip.set_fp16(False)


# few-token kernels: to 16 and to 32 tokens, tiles of 16, 8 or 4 rows, one launch over the
# column splits or one a split; past them the GEMMs. Slices of 64 columns, splits of 768;
# columns that are no multiple of 64 or of 4 (fp32).
@pytest.mark.parametrize("rows,cols", [(16, 64), (5, 4), (33, 767), (12, 768), (700, 772), (40, 769), (768, 3072),
                                       (2050, 1536), (31, 2306), (9, 12300)])
def test_linear_token_ranges(hip, rows, cols):
    """The same bits for a token whatever the call's other tokens (1, 2, 15 to 18, 31 to 34 and 70
    of them), from float64 no further than 2e-6 of the largest result (test_gpu_ops.py's bound)."""
    rng = np.random.default_rng(rows * 10000 + cols)
    w, x = (rng.standard_normal(s).astype(np.float32) for s in ((rows, cols), (70, cols)))
    dw, dx, dy = hip.upload(w), hip.upload(x), hip.alloc(70 * rows)
    hip.linear(dy.ptr, dw.ptr, rows, cols, dx.ptr, 70)
    want = dy.read().reshape(70, rows)
    assert rel(want, x.astype(np.float64) @ w.T.astype(np.float64)) < 2e-6
    for m in (1, 2, 15, 16, 17, 18, 31, 32, 33, 34):
        hip.upload_into(dy, np.full(70 * rows, np.nan, np.float32))
        hip.linear(dy.ptr, dw.ptr, rows, cols, dx.at((70 - m) * cols), m)
        got = dy.read()
        assert np.array_equal(got[:m * rows].reshape(m, rows), want[70 - m:]), m
        assert np.isnan(got[m * rows:]).all()


# either side of the rule for 17 to 32 tokens (few-token kernels or GEMMs): plain linears
@pytest.mark.parametrize("rows,cols,m,fp16,few", [
    (2304, 768, 17, False, True), (2304, 768, 32, False, True), (32000, 768, 17, False, False),
    (4096, 1536, 24, False, True), (3072, 3072, 32, False, False), (768, 3072, 32, False, True),
    (512, 768, 17, True, True), (6144, 768, 32, True, False), (32000, 768, 20, True, False),
    (4096, 1024, 32, True, True), (3072, 3072, 17, True, False), (96, 770, 32, False, True),
    (12288, 770, 32, False, False), (32000, 772, 32, False, False), (32000, 768, 16, True, True)])
def test_linear_17_to_32_tokens(hip, rows, cols, m, fp16, few):
    """The kernels the rule names run, and leave the bits of 1 and m - 1 tokens in calls of their own
    and of a 40-token call."""
    rng = np.random.default_rng(rows + m)
    hip.set_fp16(fp16)
    try:
        w = hip.upload((rng.standard_normal((rows, cols)) * 0.02).astype(np.float32))
        x, y = hip.upload(rng.standard_normal((40, cols)).astype(np.float32)), hip.alloc(40 * rows)
        hip.linear(y.ptr, w.ptr, rows, cols, x.ptr, 40)
        want = y.read()[:m * rows]
        hip.linear(y.ptr, w.ptr, rows, cols, x.ptr, 1)
        hip.linear(y.at(rows), w.ptr, rows, cols, x.at(cols), m - 1)
        assert np.array_equal(y.read()[:m * rows], want)
        hip.upload_into(y, np.full(40 * rows, np.nan, np.float32))
        hip.set_timing(True)
        hip.linear(y.ptr, w.ptr, rows, cols, x.ptr, m)
        got = y.read()
        assert np.array_equal(got[:m * rows], want) and np.isnan(got[m * rows:]).all()
        kind = "s" if cols % 4 else "v" + ("hw" if fp16 else "")
        ran = hip.kernel_stat(f"slm_linear_small_{kind}_{(m + 15) // 16}")["launches"]
        assert ran == int(few)
    finally:
        hip.set_timing(False)
        hip.set_fp16(False)
        for b in (w, x, y):
            b.free()


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("m", [2, 16, 17, 32])
@pytest.mark.parametrize("kind", ["attention", "linear_attention", "mlp"])
def test_few_token_epilogues(hip, kind, m, fp16):
    """The few-token kernels' epilogues (rope and ring stores, per-head L2 norm, the SiLU pair)
    leave the bits of one launch per operation, ring slots wrapping inside the call."""
    d, heads, dh, cap, pos = 128, 2, 64, 70, 60
    rng = np.random.default_rng(m)
    hip.set_fp16(fp16)
    try:
        up = lambda *s: hip.upload(rng.standard_normal(s).astype(np.float32) * np.float32(0.1))  # noqa: E731
        parts = {"attention": 3, "linear_attention": 4, "mlp": 6}[kind]
        w, x = up(parts * d, d), up(m, d)
        inv = hip.upload((1.0 / 10000.0 ** (np.arange(32) / 32)).astype(np.float32))
        cs, sn = hip.alloc(m * 32), hip.alloc(m * 32)
        got = []
        for fuse in (False, True):
            hip.set_fusion(fuse)
            o = {n: hip.alloc(m * d * parts) for n in ("y", "col", "q", "k", "v", "g", "out")}
            ring = [hip.alloc_cache(heads, cap, dh) for _ in range(2)]
            hip.rope_table(cs.ptr, sn.ptr, inv.ptr, pos, m, 32)
            hip.linear(o["y"].ptr, w.ptr, parts * d, d, x.ptr, m)

            def col(y, j, n=d):
                hip.columns(o[y].ptr, o["y"].ptr, m, parts * d, j * n, n)

            if kind == "attention":
                for j, n in enumerate("qk"):
                    col("col", j)
                    hip.rope(o[n].ptr, o["col"].ptr, cs.ptr, sn.ptr, m, heads, dh)
                col("v", 2)
                for r, n in zip(ring, "kv"):
                    hip.store(r.ptr, o[n].ptr, pos, m, cap, heads, dh)
            elif kind == "linear_attention":
                for j, n in enumerate("qk"):
                    col("col", j)
                    hip.l2norm(o[n].ptr, o["col"].ptr, m * heads, dh)
                col("v", 2)
                col("g", 3)
            else:
                col("q", 0, 3 * d)
                col("k", 1, 3 * d)
                hip.silu_mul(o["out"].ptr, o["q"].ptr, o["k"].ptr, m * 3 * d)
                for n in "qky":  # (dead after: overwritten)
                    hip.copy(o[n].ptr, o["v"].ptr, m * d * parts)
            hip.copy(o["col"].ptr, o["out"].ptr, m * d * parts)
            hip.flush([t.ptr for t in o.values()] + [r.ptr for r in ring])
            got.append(([t.read() for t in o.values()] + [r.read() for r in ring], hip.last_plan()["kernels"]))
        for a, b in zip(got[0][0], got[1][0]):
            assert np.array_equal(a, b)
        assert got[1][1] < got[0][1]
    finally:
        hip.set_fusion(True)
        hip.set_fp16(False)


# the first linear of a context under a caller's capture: split partials that fit in LDS, some that
# would take more than a pooled block, and columns that are no whole float4s past what LDS holds
@pytest.mark.parametrize("rows,cols,m", [(96, 3072, 5), (88000, 4096, 16), (40, 12301, 16)])
def test_linear_under_a_callers_capture(pkg, rows, cols, m):
    """No allocation: the capture ends with a graph, whose replays give the eager call's bits."""
    rng = np.random.default_rng(rows)
    hip, rt = pkg.Hip(0), pkg.lib
    try:
        w, some = hip.alloc(rows * cols), min(rows, 64)
        for r in (0, rows - some):
            hip.upload_into(w, rng.standard_normal(some * cols).astype(np.float32), r * cols)
        x, y, nan = hip.upload(rng.standard_normal(m * cols).astype(np.float32)), hip.alloc(m * rows), np.full(m * rows, np.nan, np.float32)
        stream, graph, run = C.c_void_p(hip.stream()), C.c_void_p(), C.c_void_p()
        y.read()
        assert rt.hipStreamBeginCapture(stream, 1) == 0
        hip.linear(y.ptr, w.ptr, rows, cols, x.ptr, m)
        assert rt.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert rt.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
        got = []
        for _ in range(3):
            hip.upload_into(y, nan)
            assert rt.hipGraphLaunch(run, stream) == 0
            got.append(y.read())
        rt.hipGraphExecDestroy(run), rt.hipGraphDestroy(graph)
        hip.upload_into(y, nan)
        hip.linear(y.ptr, w.ptr, rows, cols, x.ptr, m)
        want = y.read()
        assert np.isfinite(want).all() and np.abs(want).max() > 1
        for g in got:
            assert np.array_equal(g, want)
    finally:
        hip.close()
