"""CPU: who owns a Qwen model's embedding table on the device. The host layer (libtl_qwen.so) runs over a stand-in for the HIP library
that keeps "device" memory in host memory and counts its blocks by size; every launch succeeds and does nothing."""
import os
import re
import subprocess
import sys
import textwrap

import pytest

import ggufwriter as W
from test_gpu_gguf import synth_weights

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HERE = os.path.join(ROOT, "tests")

OWN = {
    "tlhip_abi_version": "int tlhip_abi_version(void) { return 1; }",
    "tlhip_last_error": 'const char* tlhip_last_error(void) { return ""; }',
    "tlhip_malloc": "int tlhip_malloc(void** p, size_t n) { *p = block(n); return *p ? 0 : -1; }",
    "tlhip_free": "int tlhip_free(void* p) { return drop(p); }",
    "tlhip_host_alloc": "int tlhip_host_alloc(void** p, size_t n) { *p = aligned_alloc(64, (n + 63) / 64 * 64); return *p ? 0 : -1; }",
    "tlhip_host_free": "int tlhip_host_free(void* p) { free(p); return 0; }",
}
COPIES = ("tlhip_memcpy_h2d", "tlhip_memcpy_d2h", "tlhip_memcpy_h2d_async", "tlhip_memcpy_d2d_async")


@pytest.fixture(scope="module")
def stand_in(tmp_path_factory):
    d = tmp_path_factory.mktemp("standin")
    hip_h = open(os.path.join(ROOT, "cpp-tensorlib_amd", "include", "tl", "hip.h")).read()
    names = sorted(set(re.findall(r'"(tlhip_\w+)"', hip_h)))
    src = textwrap.dedent("""
        #include <stdlib.h>
        #include <string.h>
        static struct { void* p; size_t n; } held[1 << 16];
        static int count, freed;
        static size_t watched;
        static void* block(size_t n) { void* p = calloc(1, n + 64); held[count].p = p; held[count++].n = n; return p; }
        static int drop(void* p) {
          for (int i = 0; i < count; i++) if (held[i].p == p) { freed += held[i].n == watched; held[i] = held[--count]; free(p); return 0; }
          return -1;
        }
        int standin_freed(size_t n) { int k = freed; watched = n; freed = 0; return k; }   /* blocks of n bytes, since it was asked last */
        int standin_holds(size_t n, const void* bytes) {
          for (int i = 0; i < count; i++) if (held[i].n == n && !memcmp(held[i].p, bytes, n)) return 1;
          return 0;
        }
        int standin_live(size_t n) { int k = 0; for (int i = 0; i < count; i++) k += held[i].n == n; return k; }
    """)
    for n in names:
        if n in OWN:
            src += OWN[n] + "\n"
        elif n in COPIES:
            src += "int %s(void* d, const void* s, size_t n) { memcpy(d, s, n); return 0; }\n" % n
        else:
            src += "long %s() { return 0; }\n" % n
    c, so = str(d / "standin.c"), str(d / "libstandin.so")
    open(c, "w").write(src)
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-o", so, c], check=True)
    return so


def _program(stand_in, body):
    """In a process of its own: the backend is chosen once per process."""
    head = "import sys, ctypes as C, importlib, numpy as np\nsys.path[:0] = [%r, %r]\n" % (ROOT, HERE)
    head += "q, models = (importlib.import_module('cpp-tensorlib_amd.' + m) for m in ('qwen', 'model'))\n"
    head += "s = C.CDLL(%r)\ns.standin_live.argtypes = s.standin_freed.argtypes = [C.c_size_t]\n" % stand_in
    r = subprocess.run([sys.executable, "-c", head + textwrap.dedent(body)], env=dict(os.environ, TENSORLIB_HIP_LIB=stand_in),
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=110)
    assert r.returncode == 0, r.stdout.decode(errors="replace")[-2000:]


DIMS = dict(n_layers=1, hidden=128, n_q_heads=2, n_kv_heads=1, head_dim=64, ff=160, vocab=777, max_ctx=16, eps=1e-6, rope_base=1e6)
TABLE = DIMS["vocab"] * DIMS["hidden"] * 2


@pytest.mark.parametrize("api", ["models", "harness"])
def test_closing_a_model_lets_its_table_go(stand_in, tmp_path, api):
    path = str(tmp_path / "m.gguf")
    W.qwen2_file(path, DIMS, synth_weights(DIMS, 3))
    opener = "models.Model.open(path, max_ctx=16, q4=True)" if api == "models" else "q.QwenGPU.from_gguf(path, max_ctx=16)"
    _program(stand_in, """
        path, live = %r, []
        for _ in range(4):
            %s.close()
            live.append(s.standin_live(%d))
        assert live[1:] == live[:-1], live       # (a staging block of the same size stays for the next one)
    """ % (path, opener, TABLE))


def test_another_table_takes_the_place_of_the_first(stand_in):
    """A token loop recorded before reads the table where it was: the block must not be given back."""
    _program(stand_in, """
        d, table = %r, %d
        g = q.QwenGPU(d)
        onorm, head = np.ones(d["hidden"], np.float32), np.zeros(d["vocab"] * d["hidden"], np.uint8)
        s.standin_freed(table)
        for seed in (1, 2):
            rows = np.random.default_rng(seed).integers(0, 1 << 16, (d["vocab"], d["hidden"]), np.uint16)
            assert g.L.tlq_set_head_q4(g.h, q._p(rows), q._p(onorm), q._p(head)) == 0
            assert s.standin_holds(C.c_size_t(table), q._p(rows))
        assert s.standin_freed(table) == 0
        g.close()
        assert s.standin_freed(table) == 1
    """ % (DIMS, TABLE))
