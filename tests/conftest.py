import importlib
import os
import shutil
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def pkg():
    return importlib.import_module("cpp-tensorlib_amd")


@pytest.fixture(scope="session")
def orc():
    from oraclelib import oracle
    return oracle()


@pytest.fixture(scope="session")
def refimpl():
    """The compiled reference (oracle/_ref), or skip where it was not built."""
    from oraclelib import ref
    r = ref()
    if r is None:
        pytest.skip("oracle/_ref/libtlref.so not built (needs /root/reference at build time)")
    return r


@pytest.fixture(scope="session")
def lib(pkg):
    """The HIP library on a real GPU. No fallback: a GPU test without the
    library or the device is an error, not a skip."""
    return pkg.load()


@pytest.fixture
def fresh_lib(pkg, tmp_path):
    """A second copy of the library with a state of its own: nothing has grown its scratch yet."""
    return pkg.TlHip(shutil.copy(pkg.LIB_PATH, str(tmp_path)))


@pytest.fixture
def recorded(fresh_lib):
    """recorded(call, out): `call` recorded while the library has no scratch, which a recording may not grow; the results of three
    replays with eager work between them. Nothing is allocated on the way."""
    def run(call, out):
        before = fresh_lib.alloc_calls()
        fresh_lib.graph_begin()
        call()
        g = fresh_lib.graph_end()
        assert fresh_lib.alloc_calls() == before
        results = []
        for _ in range(3):
            fresh_lib._chk(fresh_lib.c.tlhip_fill_u32(out.ptr, 0x7fc00000, out.nbytes // 4))
            fresh_lib.graph_launch(g)
            fresh_lib.sync()
            results.append(out.numpy())
        fresh_lib.graph_destroy(g)
        return results
    return run
