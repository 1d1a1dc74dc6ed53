"""The compiled call path takes, refuses and raises what the ctypes path it stands in for does."""
import ctypes
import importlib.util
import os
import subprocess
import sys
import sysconfig
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PKG = ROOT / "canopy-foundry_amd"


class Holder:
    def __init__(self, p):
        self.p = p

    def data_ptr(self):
        return self.p


@pytest.mark.parametrize("args", [
    (None, None, None, 0, None), (None, None, None, -1, None), (None, None, None, 4, None), (None, None, None, True, None),
    (0, 0, 0, 1 << 32, 0), (None, None, None, -(1 << 40), None), (Holder(0), Holder(16), None, 0, 0), (Holder(None), None, None, 0, None),
    (None, None, None, ctypes.c_int(0), None), (ctypes.c_void_p(0), None, None, 0, None),
    (None, None, None, 0, None, 7), (None, None, None, 0), (None, None, None, 0.0, None), (object(), None, None, 0, None), (Holder("x"), None, None, 0, 1.5),
])
def test_same_answer_as_ctypes(cf, args):
    def outcome(call):
        try:
            return call(*args)
        except Exception as e:
            return type(e), getattr(e, "code", None)

    assert outcome(cf.cf_swiglu_forward) == outcome(cf._checked("cf_swiglu_forward", cf.raw_cf_swiglu_forward))


def test_floats_sizes_and_outputs(cf):
    n, m = ctypes.c_size_t(7), ctypes.c_size_t(7)
    assert cf.cf_moe_grouped_gelu_workspace_bytes(16, 96, 8, 2048, 1408, ctypes.byref(n)) is None
    assert cf.raw_cf_moe_grouped_gelu_workspace_bytes(16, 96, 8, 2048, 1408, ctypes.byref(m)) == 0 and n.value == m.value > 7
    for value in (448.0, 448, -1, 0.0):          # a float parameter; a null output is refused whatever it is
        with pytest.raises(type(cf)._failed.__globals__["CfError"]):
            cf.cf_fp8_scale_from_amax(None, value, None, None, None)
    assert cf.cf_fp8_quantize_e4m3.__name__ == "cf_fp8_quantize_e4m3"


def build_calls(out, **env):
    """build_call() for a library elsewhere, in a process of its own: the path it returns."""
    code = ("import importlib.util, pathlib; s = importlib.util.spec_from_file_location('b', %r); b = importlib.util.module_from_spec(s); "
            "s.loader.exec_module(b); print(b.build_call(pathlib.Path(%r)))" % (str(PKG / "build.py"), str(out)))
    done = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, env={**os.environ, "CF_LIB_OUT": str(out / "libvariant.so"), **env})
    assert done.returncode == 0, done.stderr
    return done.stdout.strip(), done.stderr


def test_a_variant_has_compiled_calls_of_its_own(tmp_path):
    before = {p.name: p.stat().st_mtime_ns for p in PKG.glob("*.so")}
    made, _ = build_calls(tmp_path)
    assert Path(made).parent == tmp_path and Path(made).exists()
    assert {p.name: p.stat().st_mtime_ns for p in PKG.glob("*.so")} == before
    # another interpreter looks for another file
    assert made.endswith(sysconfig.get_config_var("EXT_SUFFIX"))


def copied_package(tmp_path, header=lambda text: text, calls=True):
    """The package's binding over a copy of the header, the library linked: the module of native.py."""
    pkg, include = tmp_path / "pkg", tmp_path / "include"
    pkg.mkdir()
    include.mkdir()
    (include / "cf_fp8.h").write_text(header((ROOT / "include" / "cf_fp8.h").read_text()))
    (pkg / "native.py").write_text((PKG / "native.py").read_text())
    for lib in PKG.glob("*.so"):
        if calls or lib.name == "libcf_fp8.so":
            (pkg / lib.name).symlink_to(lib)
    spec = importlib.util.spec_from_file_location("cf_native_copy", pkg / "native.py")
    native = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(native)
    return native


def test_loads_without_the_compiled_calls(tmp_path):
    native = copied_package(tmp_path, calls=False)
    with pytest.warns(RuntimeWarning):
        lib = native.Lib()
    assert lib.cf_swiglu_forward(None, None, None, 0, None) is None
    with pytest.raises(native.CfError):
        lib.cf_swiglu_forward(None, None, None, 4, None)
    assert lib.cf_swiglu_forward.__name__ == "cf_swiglu_forward"


def test_goes_by_the_header_that_is_read(tmp_path):
    """A prototype that changed since the compiled calls were built, and a function that was not there then."""
    native = copied_package(tmp_path, lambda text: text.replace("int cf_fp8_scale_from_amax(const float* d_amax, float fp8_max,",
                                                                "int cf_fp8_scale_from_amax(const float* d_amax, int fp8_max,"))
    assert native.parse_header()["cf_fp8_scale_from_amax"][1][1] == ("int", "fp8_max")
    with pytest.warns(RuntimeWarning):
        lib = native.Lib()
    with pytest.raises(ctypes.ArgumentError):
        lib.cf_fp8_scale_from_amax(None, 448.0, None, None, None)


def test_a_build_without_a_host_compiler_has_none(tmp_path):
    earlier, _ = build_calls(tmp_path)
    made, said = build_calls(tmp_path, CXX=str(tmp_path / "no-such-compiler"))
    assert made == "None" and "no-such-compiler" in said and not Path(earlier).exists()
    (tmp_path / "fails").write_text("#!/bin/sh\necho Python.h: not found >&2\nexit 1\n")
    (tmp_path / "fails").chmod(0o755)
    assert build_calls(tmp_path, CXX=str(tmp_path / "fails"))[0] == "None"


@pytest.mark.parametrize("error", [KeyboardInterrupt, RuntimeError, MemoryError])
def test_what_data_ptr_raises_is_raised(cf, error):
    class Once:
        """Raises the first time it is asked (an interrupt that arrives there), and would answer the second."""
        asked = 0

        def data_ptr(self):
            self.asked += 1
            if self.asked == 1:
                raise error
            return 0

    once = Once()
    with pytest.raises(error):
        cf.cf_swiglu_forward(None, once, None, 0, None)
    assert once.asked == 1


def test_a_function_the_compiled_calls_do_not_know(tmp_path, monkeypatch):
    native = copied_package(tmp_path)

    class Calls:
        @staticmethod
        def make(name, address, fallback, failed):
            return None

    monkeypatch.setattr(native, "_call_module", lambda lib: Calls)
    with pytest.raises(native.CfError):
        native.Lib().cf_swiglu_forward(None, None, None, 4, None)
