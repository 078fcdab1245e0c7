"""One-token op lists whose buffers meet: outputs inside a cache that a later op stores into, in
place factors, second matrices over what the prologue read. With fusion every buffer holds the bits
of one launch per operation, and a list takes no more kernels than its parts would.
"""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

D = 64


@pytest.fixture(scope="module")
def hip(pkg):
    h = pkg.Hip(0)
    yield h
    h.close()


class Lists:
    """Buffers of random values, refilled before each run of a list."""

    def __init__(self, hip):
        self.hip, self.bufs, self.first = hip, {}, {}
        self.rng = np.random.default_rng(5)
        self.inv, self.cs, self.sn = hip.upload(np.ones(D // 2, np.float32)), hip.alloc(D // 2), hip.alloc(D // 2)

    def buf(self, name, n, cache=None):
        self.bufs[name] = self.hip.alloc_cache(*cache) if cache else self.hip.alloc(n)
        self.first[name] = self.rng.standard_normal(n).astype(np.float32) * np.float32(0.3)

    def __getitem__(self, name):
        return self.bufs[name].ptr

    def at(self, name, off):
        return self.bufs[name].at(off)

    def run(self, ops, fuse, times=1):
        """Every buffer's bits after `times` runs of the list, and its kernels."""
        for n, b in self.bufs.items():
            self.hip.upload_into(b, self.first[n])
        self.hip.set_fusion(fuse)
        try:
            for _ in range(times):
                self.hip.rope_table(self.cs.ptr, self.sn.ptr, self.inv.ptr, 3, 1, D // 2)
                ops()
                self.hip.flush([b.ptr for b in self.bufs.values()])
            kernels = self.hip.last_plan()["kernels"]
        finally:
            self.hip.set_fusion(True)
        return {n: b.read().view(np.uint32).copy() for n, b in self.bufs.items()}, kernels

    def same(self, ops, most):
        plain, _ = self.run(ops, False)
        fused, kernels = self.run(ops, True)
        for n in plain:
            assert np.array_equal(plain[n], fused[n]), n
        assert kernels <= most, kernels


@pytest.mark.parametrize("kind", ["store", "rope", "pick"])
def test_output_inside_a_range_written_in_part(hip, kind):
    """A copy into another slot of a cache (or another place of an id history) survives the fused
    store (or pick) that writes one slot (or id) of it."""
    s = Lists(hip)
    cap = 8
    s.buf("x", D), s.buf("n", D), s.buf("g", D), s.buf("row", D), s.buf("w", 3 * D * D), s.buf("y", 3 * D)
    s.buf("k", cap * D, (1, cap, D)), s.buf("v", cap * D, (1, cap, D))
    s.buf("q", D), s.buf("kr", D), s.buf("ids", 16), s.buf("tok", 4)

    def ops():
        h = hip
        if kind == "pick":
            h.copy(s.at("ids", 8), s["row"], 4)
        else:
            h.copy(s.at("k", 5 * D), s["row"], D)
        h.rms(s["n"], s["x"], s["g"], 1, D, 1e-6)
        if kind == "store":
            h.linear(s["y"], s["w"], 2 * D, D, s["n"], 1)
            h.store(s["k"], s["y"], 6, 1, cap, 1, D)
            h.store(s["v"], s.at("y", D), 6, 1, cap, 1, D)
        elif kind == "rope":
            h.linear(s["y"], s["w"], 3 * D, D, s["n"], 1)
            h.rope(s["q"], s["y"], s.cs.ptr, s.sn.ptr, 1, 1, D)
            h.rope(s["kr"], s.at("y", D), s.cs.ptr, s.sn.ptr, 1, 1, D)
            h.store(s["k"], s["kr"], 6, 1, cap, 1, D)
            h.store(s["v"], s.at("y", 2 * D), 6, 1, cap, 1, D)
        else:
            h.linear(s["y"], s["w"], 3 * D, D, s["n"], 1)
            h.argmax(s["tok"], s["ids"], 16, 3, s["y"], 3 * D)

    s.same(ops, 8)
    got, _ = s.run(ops, True)
    where = ("ids", 8, 4) if kind == "pick" else ("k", 5 * D, D)
    assert np.array_equal(got[where[0]][where[1]:where[1] + where[2]],
                          s.first["row"][:where[2]].view(np.uint32))


@pytest.mark.parametrize("kind", ["pick", "grow"])
def test_output_inside_a_range_a_later_op_writes_in_part(hip, kind):
    """A pick writes one id of its history and a doubling half of each head's slots: what an earlier
    op put elsewhere in them stays, with other ops between."""
    s = Lists(hip)
    s.buf("x", D), s.buf("n", D), s.buf("g", D), s.buf("row", D), s.buf("w", 3 * D * D), s.buf("y", 3 * D)
    s.buf("y2", D), s.buf("w2", 3 * D * D), s.buf("ids", 16), s.buf("tok", 4)
    s.buf("k", 4 * D, (1, 4, D)), s.buf("k2", 8 * D, (1, 8, D))

    def ops():
        if kind == "pick":
            hip.copy(s.at("ids", 8), s["row"], 4)
        else:
            hip.copy(s.at("k2", 6 * D), s["row"], D)
        hip.rms(s["n"], s["x"], s["g"], 1, D, 1e-6)
        hip.linear(s["y2"], s["w2"], D, D, s["n"], 1)
        hip.rms(s["n"], s["y2"], s["g"], 1, D, 1e-6)
        hip.linear(s["y"], s["w"], 3 * D, D, s["n"], 1)
        if kind == "pick":
            hip.argmax(s["tok"], s["ids"], 16, 3, s["y"], 3 * D)
        else:
            hip.grow_cache(s.bufs["k2"], s.bufs["k"], 1, 4, D)

    s.same(ops, 6)


# kernels: what each list took before matrices were taken in pairs and factors and stores with them
@pytest.mark.parametrize("kind,most", [("scale in place", 3), ("second over the prologue's input", 2),
                                       ("two stores into one cache", 3), ("pair and scale in place", 3)])
def test_lists_with_an_extra_that_cannot_join(hip, kind, most):
    """An op that cannot join a matrix's launch leaves the matrix fused with what can."""
    s = Lists(hip)
    s.buf("x", D), s.buf("n", D), s.buf("g", D), s.buf("y", 2 * D), s.buf("z", D), s.buf("o", D)
    s.buf("w", 2 * D * D), s.buf("w2", D * D), s.buf("k", 8 * D, (1, 8, D))

    def ops():
        h = hip
        h.rms(s["n"], s["x"], s["g"], 1, D, 1e-6)
        if kind == "scale in place":
            h.linear(s["z"], s["w2"], D, D, s["n"], 1)
            h.scale_rows(s["z"], s["z"], np.array([0.37], np.float32), D)
            h.linear(s["o"], s["w"], D, D, s["z"], 1)
        elif kind == "second over the prologue's input":
            h.linear(s["z"], s["w2"], D, D, s["n"], 1)
            h.linear(s["x"], s["w"], D, D, s["n"], 1)
        elif kind == "two stores into one cache":
            h.linear(s["y"], s["w"], 2 * D, D, s["n"], 1)
            h.store(s["k"], s["y"], 2, 1, 8, 1, D)
            h.store(s["k"], s.at("y", D), 3, 1, 8, 1, D)
        else:
            h.linear(s["z"], s["w2"], D, D, s["n"], 1)
            h.linear(s["o"], s["w"], D, D, s["n"], 1)
            h.scale_rows(s["z"], s["z"], np.array([0.37], np.float32), D)

    s.same(ops, most)


@pytest.mark.parametrize("kind,most", [("rope", 2), ("l2norm", 3), ("pick", 2), ("rope of another", 5)])
def test_second_matrix_with_an_epilogue_of_its_own(hip, kind, most):
    """A matrix whose own launch takes the ops after it (rope and ring stores, the l2norms of a
    linear-attention input, a pick) is not paired with the matrix before it."""
    s = Lists(hip)
    s.buf("x", D), s.buf("n", D), s.buf("g", D), s.buf("a", D), s.buf("wa", D * D), s.buf("w", 4 * D * D)
    s.buf("y", 4 * D), s.buf("q", D), s.buf("kr", D), s.buf("dec", 4), s.buf("wd", D), s.buf("b", 4)
    s.buf("k", 8 * D, (1, 8, D)), s.buf("v", 8 * D, (1, 8, D)), s.buf("s", D * D), s.buf("o", D)
    s.buf("tok", 4), s.buf("ids", 8)

    def ops():
        h = hip
        h.rms(s["n"], s["x"], s["g"], 1, D, 1e-6)
        h.linear(s["a"], s["wa"], D, D, s["n"], 1)
        if kind == "rope":
            h.linear(s["y"], s["w"], 3 * D, D, s["n"], 1)
            h.rope(s["q"], s["y"], s.cs.ptr, s.sn.ptr, 1, 1, D)
            h.rope(s["kr"], s.at("y", D), s.cs.ptr, s.sn.ptr, 1, 1, D)
            h.store(s["k"], s["kr"], 6, 1, 8, 1, D)
            h.store(s["v"], s.at("y", 2 * D), 6, 1, 8, 1, D)
        elif kind == "rope of another":  # (these two are a pair)
            h.linear(s["y"], s["w"], 3 * D, D, s["n"], 1)
            h.rope(s["q"], s["s"], s.cs.ptr, s.sn.ptr, 1, 1, D)
            h.rope(s["kr"], s.at("s", D), s.cs.ptr, s.sn.ptr, 1, 1, D)
            h.store(s["k"], s["kr"], 6, 1, 8, 1, D)
            h.store(s["v"], s.at("s", 2 * D), 6, 1, 8, 1, D)
        elif kind == "l2norm":
            h.linear(s["y"], s["w"], 4 * D, D, s["n"], 1)
            h.l2norm(s["q"], s["y"], 1, D)
            h.l2norm(s["kr"], s.at("y", D), 1, D)
            h.linear(s["dec"], s["wd"], 1, D, s["n"], 1)
            h.gla(s["o"], s["s"], s["q"], s["kr"], s.at("y", 2 * D), s["dec"], s["b"], 1, 1, D)
        else:
            h.linear(s["y"], s["w"], 3 * D, D, s["n"], 1)
            h.argmax(s["tok"], s["ids"], 8, 3, s["y"], 3 * D)

    s.same(ops, most)


def test_pending_op_in_a_matrix_launchs_way(hip):
    """A pending op that reads what a matrix's epilogue writes runs first; the matrix keeps its
    fusion (here a QKV input whose rotated q replaces the row a shift read)."""
    s = Lists(hip)
    s.buf("x", D), s.buf("prev", D), s.buf("sh", D), s.buf("w", 3 * D * D), s.buf("y", 3 * D), s.buf("kr", D)
    s.buf("k", 8 * D, (1, 8, D)), s.buf("v", 8 * D, (1, 8, D))

    def ops():
        h = hip
        h.shift(s["sh"], s["prev"], s["x"], 1, D)
        h.linear(s["y"], s["w"], 3 * D, D, s["x"], 1)
        h.rope(s["prev"], s["y"], s.cs.ptr, s.sn.ptr, 1, 1, D)
        h.rope(s["kr"], s.at("y", D), s.cs.ptr, s.sn.ptr, 1, 1, D)
        h.store(s["k"], s["kr"], 6, 1, 8, 1, D)
        h.store(s["v"], s.at("y", 2 * D), 6, 1, 8, 1, D)

    s.same(ops, 3)


def test_step_whose_capture_fails(hip):
    """A list whose graph cannot be made has run all the same: no error, its state advanced once a
    run (a running sum, a ring), over replays of another list and after captures work again."""
    s = Lists(hip)
    s.buf("x", D), s.buf("n", D), s.buf("g", D), s.buf("w", D * D), s.buf("y", D), s.buf("sum", D)
    s.buf("k", 8 * D, (1, 8, D))

    def ops():
        hip.rms(s["n"], s["x"], s["g"], 1, D, 1e-6)
        hip.linear(s["y"], s["w"], D, D, s["n"], 1)
        hip.add(s["sum"], s["sum"], s["y"], D)
        hip.store(s["k"], s["sum"], 3, 1, 8, 1, D)

    want, _ = s.run(ops, True, times=6)
    hip.set_capture(False)
    try:
        before = hip.graph_stats()
        got, _ = s.run(ops, True, times=6)
        after = hip.graph_stats()
    finally:
        hip.set_capture(True)
    for n in want:
        assert np.array_equal(want[n], got[n]), n
    assert after["captured"] == before["captured"] and after["launched"] == before["launched"] + 6
    got, _ = s.run(ops, True, times=6)
    for n in want:
        assert np.array_equal(want[n], got[n]), n
    assert hip.graph_stats()["captured"] == after["captured"] + 1


def test_more_lists_than_are_kept(hip):
    """Forty lists in turn, four times over (32 are kept): each run's bits are its first run's."""
    s = Lists(hip)
    n = 40
    s.buf("x", D), s.buf("w", D * D)
    for i in range(n):
        s.buf(f"y{i}", D)

    def step(i):
        hip.rope_table(s.cs.ptr, s.sn.ptr, s.inv.ptr, 3, 1, D // 2)
        hip.linear(s[f"y{i}"], s["w"], D, D, s["x"], 1)
        hip.add(s[f"y{i}"], s[f"y{i}"], s["x"], D - 4 * (i % 8))
        hip.flush([b.ptr for b in s.bufs.values()])

    want = {}
    for b, v in s.first.items():
        hip.upload_into(s.bufs[b], v)
    for turn in range(4):
        for i in range(n):
            hip.upload_into(s.bufs[f"y{i}"], s.first[f"y{i}"])
            step(i)
            got = s.bufs[f"y{i}"].read()
            assert np.array_equal(got, want.setdefault(i, got)), (turn, i)
