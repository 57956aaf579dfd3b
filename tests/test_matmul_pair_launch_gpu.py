"""A Q4_0 matmul with its residual add, the RMSNorm behind it and the matmul that reads it, in one launch for up to four
requests: every buffer holds the bits that the separate launches leave."""
import numpy as np
import pytest

from oracle import paged_oracle as po
from test_matmul_norm_fusion_gpu import EPS, _read

pytestmark = pytest.mark.gpu


def _weights(rng, rows, cols):
    return po.quantize_q4_0((rng.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32))


class Pair:
    """h = r + W0 mix, where mix = silu(gate) * up of Wg x0; n = norm(h); then W1 n and its split + SiLU ("silu"), its split + RoPE +
    cast ("rope"), that and the scatters of K and V ("scatters") or the call that does all of it ("pages")"""
    PAGE, PAGES = 16, 9

    def __init__(self, exe, reader, batch, mid, hid, heads, same=()):
        rng = np.random.default_rng(batch * 1000 + hid)
        self.exe, self.reader, self.batch, self.mid, self.hid, self.same = exe, reader, batch, mid, hid, dict(same)
        self.heads, self.kv, self.d = heads, max(1, heads // 4), 64
        self.rows = 2 * heads * self.d if reader == "silu" else (heads + 2 * self.kv) * self.d
        self.name = f"pair.{reader}.{batch}.{mid}.{hid}.{heads}"
        self.wg, self.w0, self.w1 = _weights(rng, 2 * mid, 64), _weights(rng, hid, mid), _weights(rng, self.rows, hid)
        self.gamma = rng.uniform(0.5, 1.5, hid - 8).astype(np.float32)      # (1 beyond)
        half, kvd = self.rows // 2, self.kv * self.d
        shapes = {"x0": 64, "gu": 2 * mid, "g0": mid, "u0": mid, "mix": mid, "p": hid, "r": hid, "h": hid, "n": hid, "y": self.rows}
        shapes |= {"g": half, "u": half, "m": half} if reader == "silu" else {"q": heads * self.d, "k": kvd, "v": kvd}
        self.init = {m: rng.standard_normal((batch, n)).astype(np.float32) for m, n in shapes.items()}
        if reader != "silu":
            self.init |= {m: rng.uniform(-1, 1, (batch, self.d // 2)).astype(np.float32) for m in ("cos", "sin")}
            self.init |= {m: np.zeros((batch, kvd), np.uint16) for m in ("k16", "v16")}
        if reader in ("scatters", "pages"):
            self.init |= {m: np.zeros((self.PAGES, self.PAGE, kvd), np.uint16) for m in ("kp", "vp")}
            self.ids, self.slots = rng.permutation(self.PAGES)[:batch].astype(np.uint32), rng.integers(0, self.PAGE, batch).astype(np.uint32)
        most = max(a.nbytes for a in self.init.values())       # (any of them can be another)
        self.dev = {m: exe.allocateScratchBuffer(most) for m in self.init}
        self.reset()

    def at(self, m):
        return self.dev[self.same.get(m, m)]

    def reset(self):
        for m, a in self.init.items():
            assert self.exe.uploadToBuffer(self.dev[m], a)

    def read(self):
        return {m: _read(self.exe, b, self.init[m]) for m, b in self.dev.items()}

    def encode(self):
        exe, at, b = self.exe, self.at, self.batch

        def matmul(i, w, src, rows, cols, dst):
            return exe.encodeMatMulQ4_0Batched(f"{self.name}.{i}", w, at(src), b, rows, cols, w.shape[1], 1, at(dst))
        # (the gate/up launch in front hands the first matmul its activations with block scales)
        ok = matmul("g", self.wg, "x0", 2 * self.mid, 64, "gu")
        ok = ok and exe.encodeGateUpSplitSiluMul(at("gu"), at("g0"), at("u0"), at("mix"), b, self.mid, 2 * self.mid)
        ok = ok and matmul(0, self.w0, "mix", self.hid, self.mid, "p")
        ok = ok and exe.encodeAddBatched(at("p"), at("r"), at("h"), b * self.hid)
        ok = ok and exe.encodeRmsNormBatched(at("h"), self.gamma, EPS, b, self.hid, at("n"))
        ok = ok and matmul(1, self.w1, "n", self.rows, self.hid, "y")
        if self.reader == "silu":
            return ok and exe.encodeGateUpSplitSiluMul(at("y"), at("g"), at("u"), at("m"), b, self.rows // 2, self.rows)
        kvd = self.kv * self.d
        sizes = b, self.heads, self.kv, self.d, self.rows, self.heads * self.d, kvd, kvd, self.d
        if self.reader == "pages":
            return ok and exe.encodeQkvSplitRopeScatter(at("y"), at("q"), at("kp"), at("vp"), at("cos"), at("sin"), self.ids, self.slots,
                                                        self.PAGE, *sizes, at("k"), at("v"))
        ok = ok and exe.encodeQkvSplitRopeCast(at("y"), at("q"), at("k"), at("v"), at("k16"), at("v16"), at("cos"), at("sin"), *sizes)
        for pages, src in (("kp", "k16"), ("vp", "v16")) if self.reader == "scatters" else ():
            ok = ok and exe.encodeScatterKVPagedBatched(at(pages), self.ids, self.slots, self.PAGE, self.kv, self.d, b, at(src))
        return ok

    def once(self):
        return self.exe.beginForwardPassCB() and self.encode() and self.exe.flushForwardPassCB()

    def captured(self, replays, places=()):
        """(launches of the pass, the buffers after every replay); places: pages and slots for each replay"""
        exe = self.exe
        assert exe.beginForwardPassCB() and exe.captureBegin() and self.encode()
        handle = exe.captureEnd()
        assert handle > 0 and exe.flushForwardPassCB(), exe.lastError()
        out = []
        none = np.zeros(0, np.uint32)
        for i in range(replays):
            self.reset()
            if places:
                assert exe.replayUpdate(handle, none, np.zeros(1, np.uint32), np.zeros(self.batch, np.uint32), none, *places[i]), exe.lastError()
            assert exe.beginForwardPassCB() and exe.replay(handle) and exe.flushForwardPassCB(), exe.lastError()
            out.append(self.read())
        n = exe.capturedLaunches(handle)
        exe.captureRelease(handle)
        return n, out

    def free(self):
        for b in self.dev.values():
            self.exe.releaseScratchBuffer(b)


def _same_bits(got, want):
    for m in want:
        assert np.array_equal(got[m].view(np.uint8), want[m].view(np.uint8)), m


@pytest.mark.parametrize("reader,batch,mid,hid,heads,pair", [
    ("silu", 1, 4224, 2048, 88, True),      # a whole quad of K per wave
    ("silu", 4, 4160, 64, 66, True),        # half a quad in all
    ("silu", 3, 5632, 192, 72, True),       # a quad and a half; the first matmul's K in slices
    ("silu", 1, 4224, 2112, 88, False),     # more than a quad per wave
    ("silu", 5, 4224, 1024, 88, False),     # more requests
    ("silu", 1, 4224, 1024, 124, True),     # 31 of an XCD's 32 CUs
    ("silu", 1, 4224, 1024, 125, False),    # all of them: none is left for what they wait for, if that is another process's turn
    ("silu", 2, 4224, 1024, 128, False),
    ("rope", 1, 5632, 2048, 32, True),      # three slices, one row tile to a workgroup
    ("rope", 4, 4160, 2112, 8, True),       # a wave with a second quad, and that a part of one
    ("rope", 2, 4224, 4096, 72, True),      # two quads per wave, two row tiles
    ("rope", 4, 4224, 1984, 4, True),
])
def test_two_matmuls_in_a_launch(exe, reader, batch, mid, hid, heads, pair):
    c = Pair(exe, reader, batch, mid, hid, heads)
    try:
        got = {}
        for on in (0, 1):
            assert exe.setOption("q4_chain", on)
            c.reset()
            assert c.once(), exe.lastError()
            got[on] = c.read(), *c.captured(3)
        assert np.isfinite(got[0][0]["y"]).all()
        _same_bits(got[1][0], got[0][0])
        for on in (0, 1):
            for after in got[on][2]:
                _same_bits(after, got[0][0])
        assert got[0][1] - got[1][1] == (1 if pair else 0)
    finally:
        exe.setOption("q4_chain", 1)
        c.free()


@pytest.mark.parametrize("reader,batch,mid,hid,heads", [
    ("pages", 1, 5632, 2048, 32), ("pages", 4, 4224, 1984, 4), ("pages", 3, 4224, 4096, 72), ("scatters", 2, 5632, 2048, 32), ("scatters", 4, 4224, 4096, 72)])
def test_rows_of_keys_and_values_in_pages(exe, reader, batch, mid, hid, heads):
    """Page rows inside the arguments and, in a captured pass, on the device, where they change from replay to replay."""
    c = Pair(exe, reader, batch, mid, hid, heads)
    rng = np.random.default_rng(batch)
    places = [(rng.permutation(c.PAGES)[:batch].astype(np.uint32), rng.integers(0, c.PAGE, batch).astype(np.uint32)) for _ in range(2)]
    places = [(c.ids, c.slots), *places, (c.ids, c.slots)]
    try:
        got = {}
        for on in (0, 1):
            assert exe.setOption("q4_chain", on)
            c.reset()
            assert c.once(), exe.lastError()
            got[on] = c.read(), *c.captured(4, places)
        _same_bits(got[1][0], got[0][0])
        _same_bits(got[1][2][0], got[0][0])
        for i, (ids, slots) in enumerate(places):
            _same_bits(got[1][2][i], got[0][2][i])
            for pages, rows in (("kp", "k"), ("vp", "v")):
                want = np.zeros_like(c.init[pages])
                want[ids, slots] = got[1][2][i][rows].astype(np.float16).view(np.uint16)
                assert np.array_equal(got[1][2][i][pages], want), (pages, i)
        assert got[0][1] - got[1][1] == 1
    finally:
        exe.setOption("q4_chain", 1)
        c.free()


@pytest.mark.parametrize("reader,same,pair", [
    ("silu", {"h": "r"}, True), ("silu", {"h": "p"}, True),           # the first matmul's own buffers
    ("silu", {"n": "h"}, False), ("silu", {"y": "r"}, False), ("silu", {"m": "p"}, False), ("silu", {"u": "r", "g": "p"}, False),
    ("silu", {"m": "mix"}, True), ("silu", {"m": "x0"}, True),        # what the launch in front has read
    ("rope", {"q": "r"}, False), ("rope", {"k": "p"}, False), ("rope", {"v": "r"}, False), ("rope", {"k16": "p"}, False),
    ("rope", {"v16": "r"}, False), ("rope", {"q": "h"}, False), ("rope", {"cos": "h"}, False), ("rope", {"sin": "p"}, False),
    ("rope", {"cos": "r"}, True),                                     # both read it
    ("rope", {"q": "mix", "k16": "x0"}, True),
    ("pages", {"kp": "r"}, False), ("pages", {"vp": "p"}, False), ("pages", {"kp": "mix"}, True), ("scatters", {"vp": "r"}, False),
])
def test_buffers_that_meet(exe, reader, same, pair):
    """Where the second matmul writes what the first one reads or writes, or reads what it writes, the two are launched one after the
    other."""
    c = Pair(exe, reader, 2, 5632, 512, 88 if reader == "silu" else 32, same)
    try:
        got = {}
        for on in (0, 1):
            assert exe.setOption("q4_chain", on)
            c.reset()
            assert c.once(), exe.lastError()
            got[on] = c.read(), *c.captured(2)
        _same_bits(got[1][0], got[0][0])
        for after in got[1][2]:
            _same_bits(after, got[0][0])
        assert got[0][1] - got[1][1] == (1 if pair else 0)
    finally:
        exe.setOption("q4_chain", 1)
        c.free()


def test_the_first_of_two_keeps_what_it_reads(exe):
    """Behind the held-back pair a gate/up projection with longer rows: its products go where the pair's first matmul
    still finds its input, and that buffer grows."""
    first = Pair(exe, "silu", 4, 4224, 512, 72)
    rng = np.random.default_rng(9)
    try:
        assert exe.setOption("q4_chain", 0) and first.once(), exe.lastError()
        want = first.read()
        assert exe.setOption("q4_chain", 1)
        first.reset()
        wide = first.rows // 2
        w = _weights(rng, 128, wide)
        out = exe.allocateScratchBuffer(4 * 128 * 4)
        assert exe.beginForwardPassCB() and first.encode()
        assert exe.encodeMatMulQ4_0Batched("pair.behind", w, first.at("m"), 4, 128, wide, w.shape[1], 1, out)
        assert exe.flushForwardPassCB(), exe.lastError()
        _same_bits(first.read(), want)
        exe.releaseScratchBuffer(out)
    finally:
        exe.setOption("q4_chain", 1)
        first.free()


def test_words_that_never_come(exe):
    """The second matmul gives up, the pass fails, and the next one is as if nothing had been."""
    c = Pair(exe, "rope", 1, 4224, 512, 8)
    try:
        assert c.once(), exe.lastError()
        want = c.read()
        assert exe.setOption("decode_spin_limit", 3) and exe.setOption("decode_test_flags", 1)
        assert not c.once() and "gave up" in exe.lastError()
        assert exe.setOption("decode_spin_limit", 200000) and exe.setOption("decode_test_flags", 0)
        c.reset()
        assert c.once(), exe.lastError()
        _same_bits(c.read(), want)
    finally:
        exe.setOption("decode_spin_limit", 200000)
        exe.setOption("decode_test_flags", 0)
        c.free()


MEMORY = """
import ctypes as C, sys
sys.path[:0] = ["tests", "."]
from mlcompiler_amd import HipExecutor
from test_matmul_pair_launch_gpu import Pair
exe, hip = HipExecutor.Instance(), C.CDLL("libamdhip64.so")
exe.requireAvailable()
free, total = C.c_size_t(), C.c_size_t()
def used():
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return total.value - free.value
c = Pair(exe, "silu", 4, 4224, 4096 // 2, 88)
assert exe.beginForwardPassCB() and c.encode()
before = used()
assert exe.flushForwardPassCB(), exe.lastError()
print("used", before, used())
"""


def test_the_launch_of_a_held_back_pair_allocates_nothing():
    """(A process of its own: the library's buffers are for good.)"""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    out = subprocess.run([sys.executable, "-c", MEMORY], cwd=root, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    before, after = (int(v) for v in out.stdout.split("used")[1].split())
    assert before == after
