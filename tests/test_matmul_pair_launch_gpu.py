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
    """h = r + W0 mix, where mix = silu(gate) * up of Wg x0; n = norm(h); then W1 n and its split + SiLU or its split + RoPE + cast"""

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
        if reader == "rope":
            self.init |= {m: rng.uniform(-1, 1, (batch, self.d // 2)).astype(np.float32) for m in ("cos", "sin")}
            self.init |= {m: np.zeros((batch, kvd), np.uint16) for m in ("k16", "v16")}
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
        return ok and exe.encodeQkvSplitRopeCast(at("y"), at("q"), at("k"), at("v"), at("k16"), at("v16"), at("cos"), at("sin"), b,
                                                 self.heads, self.kv, self.d, self.rows, self.heads * self.d, kvd, kvd, self.d)

    def once(self):
        return self.exe.beginForwardPassCB() and self.encode() and self.exe.flushForwardPassCB()

    def captured(self, replays):
        """(launches of the pass, the buffers after every replay)"""
        exe = self.exe
        assert exe.beginForwardPassCB() and exe.captureBegin() and self.encode()
        handle = exe.captureEnd()
        assert handle > 0 and exe.flushForwardPassCB(), exe.lastError()
        out = []
        for _ in range(replays):
            self.reset()
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


@pytest.mark.parametrize("same,pair", [
    ({"h": "r"}, True), ({"h": "p"}, True),           # the first matmul's own buffers
    ({"n": "h"}, False), ({"y": "r"}, False), ({"m": "p"}, False), ({"u": "r", "g": "p"}, False),
    ({"m": "mix"}, True), ({"m": "x0"}, True),        # what the launch in front has read
])
def test_buffers_that_meet(exe, same, pair):
    """Where the second matmul writes what the first one reads or writes the two are launched one after the other."""
    c = Pair(exe, "silu", 2, 5632, 512, 88, same)
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
