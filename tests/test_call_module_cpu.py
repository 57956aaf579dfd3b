"""The module of HipExecutor's inner-loop calls (csrc/py_call.cpp) without a GPU: built against a stand-in for the
library whose every call waits until another Python thread has run."""
import os
import subprocess
import sys
import sysconfig

import numpy
import pytest

from mlcompiler_amd import build

STAND_IN = r"""
#include <unistd.h>
static volatile int inside, go;
int stand_in_inside(void) { return inside; }
void stand_in_go(void) { go = 1; }
static int call(void) {
    inside = 1;
    for (int i = 0; i < 500 && !go; ++i) usleep(1000);
    const int seen = go;
    inside = go = 0;
    return seen;
}
#define CALL(name) int mlc_hip_##name() { return call(); }
CALL(begin) CALL(flush) CALL(paged_attn_decode) CALL(paged_attn_prefill) CALL(scatter_kv_paged_batched_f16)
CALL(scatter_kv_paged) CALL(gather_kv_pages) CALL(qkv_split_rope_cast) CALL(rms_norm_batched) CALL(add_batched)
CALL(gate_up_split_silu_mul) CALL(matmul_q4_0_batched) CALL(matmul_q6_k_batched) CALL(replay_update) CALL(replay)
"""

PROGRAM = r"""
import ctypes, sys, threading, time
import numpy as np
sys.path.insert(0, sys.argv[1])
import _call
lib = ctypes.CDLL(sys.argv[1] + "/libmlc_hip.so")
one, two, w = np.zeros(1, np.uint32), np.zeros(2, np.uint32), np.zeros(18, np.uint8)
cases = dict(
    begin=(), flush=(), replay=(1,), replay_update=(1, one, two, one, one, None, None),
    scatter=(1, one, 64, 1, 64, 1, 0, 1, 2), gather=(1, one, 64, 1, 64, 1, 1, 2))
for sync in (False, True):
    cases.update({
        ("attention", sync): (1, 1, 1, 1, one, two, one, one, 1, 1, 1, 64, 64, True, sync),
        ("prefill", sync): (1, 1, 1, 1, one, two, one, one, 1, 1, 1, 1, 64, 64, sync),
        ("scatter_batched", sync): (1, one, one, 64, 1, 64, 1, 1, sync),
        ("rope_cast", sync): (1,) * 8 + (1,) * 9 + (sync,),
        ("rms_norm", sync): (1, np.ones(4, np.float32), 1e-5, 1, 4, 1, sync),
        ("add", sync): (1, 1, 1, 4, sync), ("gate_up", sync): (1, 1, 1, 1, 1, 4, 8, sync),
        ("matmul_q4_0", sync): ("w", w, 1, 1, 1, 32, 18, 2, 1, sync), ("matmul_q6_k", sync): ("w", w, 1, 1, 1, 32, 18, 1, sync)})
names = {n if isinstance(n, str) else n[0] for n in cases}
assert names == {n for n in dir(_call) if not n.startswith("__")}, names
end = threading.Event()
def other():
    while not end.is_set():
        if lib.stand_in_inside():
            lib.stand_in_go()
        time.sleep(0.0005)
t = threading.Thread(target=other); t.start()
held = [n for n, args in cases.items() if getattr(_call, n if isinstance(n, str) else n[0])(*args) is not True]
end.set(); t.join()
print("held the interpreter:", held)
sys.exit(1 if held else 0)
"""


def test_other_threads_run_during_every_call(tmp_path):
    (tmp_path / "stand_in.c").write_text(STAND_IN)
    (tmp_path / "program.py").write_text(PROGRAM)
    subprocess.check_call(["gcc", "-w", "-shared", "-fPIC", str(tmp_path / "stand_in.c"), "-o", str(tmp_path / "libmlc_hip.so")])
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I" + sysconfig.get_paths()["include"],
                           "-I" + numpy.get_include(), os.path.join(build.CSRC, "py_call.cpp"),
                           "-o", str(tmp_path / ("_call" + sysconfig.get_config_var("EXT_SUFFIX"))),
                           "-L" + str(tmp_path), "-lmlc_hip", "-Wl,-rpath," + str(tmp_path)])
    done = subprocess.run([sys.executable, str(tmp_path / "program.py"), str(tmp_path)], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout + done.stderr


def test_the_built_module_names_its_interpreter_and_is_current():
    assert build.CALL_MODULE_PATH.endswith("_call" + sysconfig.get_config_var("EXT_SUFFIX"))
    assert sysconfig.get_config_var("SOABI") in os.path.basename(build.CALL_MODULE_PATH)
    assert build.call_module_is_current()


def test_another_numpy_or_other_sources_make_it_stale(tmp_path, monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(numpy, "__version__", "1.0.0")
        assert not build.call_module_is_current()
    (tmp_path / "py_call.cpp").write_text("// other\n")
    with monkeypatch.context() as m:
        m.setattr(build, "CSRC", str(tmp_path))
        assert not build.call_module_is_current()
    with monkeypatch.context() as m:      # an interpreter that nothing was built for yet
        m.setattr(build, "CALL_MODULE_PATH", str(tmp_path / "_call.other.so"))
        assert not build.call_module_is_current()
    assert build.call_module_is_current()


def test_a_stale_module_alone_does_not_rebuild_the_libraries(monkeypatch):
    from mlcompiler_amd import _lib
    asked = []
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "call_module_is_current", lambda: False)
    monkeypatch.setattr(_lib, "build_call_module", lambda: asked.append("module"))
    monkeypatch.setattr(_lib, "build_all", lambda: asked.append("all"))
    with pytest.raises(_lib.NativeLibraryError):
        _lib.load(build_if_missing=False)
    _lib.load()
    assert asked == ["module"]
