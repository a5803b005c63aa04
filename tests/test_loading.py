"""When the native libraries are loaded, and what is said where they are missing or of another ABI (no GPU: a call on
CPU tensors gets as far as the operator, which refuses them)."""
import shutil
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

from monarch_muon_amd import _abi, butterfly

PACKAGE = Path(_abi.__file__).resolve().parent
BUILT = [PACKAGE / "libmmuon.so", _abi.TORCH_LIB_PATH]

CALL = """
import torch
import monarch_muon_amd as m
from monarch_muon_amd import _abi, butterfly
x, w1, w2 = torch.ones(4, 64).bfloat16(), torch.ones(2, 32, 32).bfloat16(), torch.ones(2, 40, 32).bfloat16()

def refused(fn, *args):
    try:
        fn(*args)
    except RuntimeError as e:
        return str(e)
    raise AssertionError("accepted")
"""


@pytest.fixture
def copy(tmp_path):
    """The package without its built libraries, and a way to run a program on it."""
    shutil.copytree(PACKAGE, tmp_path / "monarch_muon_amd",
                    ignore=shutil.ignore_patterns("*.so", "*.o", "_build", "__pycache__"))

    def run(body):
        r = subprocess.run([sys.executable, "-c", CALL + textwrap.dedent(body)], cwd=tmp_path, capture_output=True,
                           text=True, timeout=300)
        assert r.returncode == 0, r.stdout + r.stderr
    return tmp_path / "monarch_muon_amd", run


def stub(path, version, tmp_path):
    """A libmmuon.so that has no function but the two every version has had."""
    src = tmp_path / "stub.c"
    src.write_text(f'int mmuon_abi_version(void) {{ return {version}; }}\nconst char* mmuon_last_error(void) '
                   '{ return ""; }\n')
    subprocess.run(["gcc", "-shared", "-fPIC", str(src), "-o", str(path)], check=True)


def test_libraries_built_after_the_import_are_used(copy):
    """Importing without a built library, building, and calling, in one process."""
    where, run = copy
    run(f"""
        import shutil
        assert "is missing" in refused(m.butterfly_blk, x, w1, w2)
        assert "is missing" in refused(_abi.lib)
        for f in {[str(p) for p in BUILT]}:
            shutil.copy(f, r"{where}")
        assert "ROCm GPU" in refused(m.butterfly_blk, x, w1, w2)
        assert m.butterfly_blk(*(t.to("meta") for t in (x, w1, w2))).shape == (4, 80)
        assert _abi._lib is None and butterfly._bind() == 0 and _abi._lib is not None
    """)


@pytest.mark.parametrize("version", [_abi.ABI_VERSION - 1, _abi.ABI_VERSION])
def test_a_library_of_another_build_is_refused_by_name_and_not_by_the_import(copy, tmp_path, version):
    """A kernel library of the ABI before, or one that lacks functions of this one, beside an operator left from it:
    the import (with it the build) works, and what needs the library says what is wrong."""
    where, run = copy
    stub(where / "libmmuon.so", version, tmp_path)
    (where / "libmmuon_torch.so").write_text("an operator of an earlier ABI")
    shutil.copy(_abi.TORCH_LIB_PATH, where)
    expect = f"has ABI {version}" if version != _abi.ABI_VERSION else "lacks a function"
    run(f"""
        import monarch_muon_amd.build
        assert "{expect}" in refused(_abi.lib), refused(_abi.lib)
        assert butterfly._bind() == -1
        assert "ROCm GPU" in refused(m.butterfly_blk, x, w1, w2)
    """)


def test_operator_refuses_functions_of_another_abi():
    assert butterfly._torch_lib.mmuon_torch_bind(_abi.ABI_VERSION + 1, None, None, None, None) == -1


def test_header_and_binding_state_one_abi():
    text = (PACKAGE.parent / "include" / "mmuon.h").read_text()
    assert f"#define MMUON_ABI_VERSION {_abi.ABI_VERSION}\n" in text
    assert _abi.lib().mmuon_abi_version() == _abi.ABI_VERSION
