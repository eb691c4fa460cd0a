"""The C-ABI library loads and exports exactly what include/chadq.h declares.  No GPU, no compute calls."""
import ctypes
import os
import re

import pytest

from chadslab_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "chadq.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(chadq_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_something():
    syms = declared_symbols()
    assert "chadq_gemv_i4g32" in syms and "chadq_version" in syms and len(syms) >= 10


def test_library_is_built_in_tree():
    assert _lib.LIB_PATH.exists(), "run `python -m chadslab_amd.build` (or __graft_entry__.build())"
    assert str(_lib.LIB_PATH).startswith(ROOT)


def test_every_declared_symbol_is_exported():
    lib = ctypes.CDLL(str(_lib.LIB_PATH))
    for name in declared_symbols():
        assert hasattr(lib, name), "libchadq.so does not export %s" % name


def test_python_binding_covers_the_header():
    assert sorted(_lib.SIGNATURES) == declared_symbols()


def test_version_and_arch_without_a_gpu():
    lib = _lib.load()
    assert lib.chadq_version() >= 100
    assert lib.chadq_arch() == b"gfx950"
    assert lib.chadq_last_error() is not None


def test_ops_refuse_cpu_tensors():
    import torch

    from chadslab_amd import QWeightInt4G32, ops

    qw = QWeightInt4G32(torch.zeros(4, 16, dtype=torch.uint8), torch.ones(4, 1, dtype=torch.float16))
    with pytest.raises(ValueError, match="GPU tensor"):
        ops.qgemv(torch.zeros(1, 32, dtype=torch.bfloat16), qw)
    with pytest.raises(ValueError, match="GPU tensor"):
        ops.unpack_int4(torch.zeros(4, 16, dtype=torch.uint8))


def test_host_side_quantizer_matches_oracle():
    import numpy as np
    import torch

    import chadslab_amd as C
    from oracle import chadq_oracle as O

    w = (np.random.Generator(np.random.PCG64(7)).standard_normal((24, 96)) * 0.1).astype(np.float32)
    qw = C.quantize_int4_g32(torch.from_numpy(w))
    p, s = O.quantize_int4_g32(w)
    assert np.array_equal(qw.packed.numpy(), p) and np.array_equal(qw.scale.numpy(), s)
    q8 = C.quantize_int8_row(torch.from_numpy(w))
    w8, s8 = O.quantize_int8_row(w)
    assert np.array_equal(q8.w.numpy(), w8) and np.array_equal(q8.scale.numpy(), s8)
    with pytest.raises(ValueError):
        C.QWeightInt4G32(torch.zeros(4, 16, dtype=torch.uint8), torch.ones(4, 2, dtype=torch.float16))


def test_host_module_has_no_thread_local_storage():
    """Opened late, it would slow every access to thread-local storage in the process: torch's current device, stream, allocator."""
    import struct

    data = _lib.HOST_PATH.read_bytes()
    assert data[:5] == b"\x7fELF\x02"
    start, = struct.unpack_from("<Q", data, 32)
    size, count = struct.unpack_from("<HH", data, 54)
    kinds = [struct.unpack_from("<I", data, start + i * size)[0] for i in range(count)]
    assert 1 in kinds and 7 not in kinds  # PT_LOAD, PT_TLS


def test_ops_go_without_the_host_module(monkeypatch, tmp_path):
    """It holds no kernels: where it is missing, or was built for another torch, the calls take the Python road, and say so."""
    import torch

    from chadslab_amd import QWeightInt4G32, ops

    broken = tmp_path / "_host_call.so"
    qw = QWeightInt4G32(torch.zeros(4, 16, dtype=torch.uint8), torch.ones(4, 1, dtype=torch.float16))
    for content in (None, b"no extension"):
        if content:
            broken.write_bytes(content)
        monkeypatch.setattr(_lib, "HOST_PATH", broken)
        monkeypatch.setattr(_lib, "_native", None)
        monkeypatch.setattr(_lib, "_native_lib", None)
        with pytest.warns(RuntimeWarning, match="host module"), pytest.raises(ValueError, match="GPU tensor"):
            ops.qlinear(torch.zeros(1, 32, dtype=torch.bfloat16), qw)
        with pytest.raises(ValueError, match="GPU tensor"):
            ops.moe_ffn(torch.zeros(1, 32, dtype=torch.bfloat16), torch.zeros(1, 1), [(qw, qw, qw)], top_k=1)


def test_the_library_is_linked_before_the_host_module_can_fail(monkeypatch, tmp_path):
    from chadslab_amd import build

    linked = []

    def run(cmd):
        out = cmd[cmd.index("-o") + 1]
        open(out, "w").close()
        if "-shared" in cmd:
            linked.append(os.path.basename(out))

    def no_headers(verbose=True):
        raise RuntimeError("no torch headers")

    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "build_host", no_headers)
    monkeypatch.setattr(build, "OBJ", tmp_path / "obj")
    monkeypatch.setattr(build, "LIB", tmp_path / "libchadq.so")
    monkeypatch.setattr(build, "ablation_path", lambda name: tmp_path / ("ablate_%s.so" % name))
    with pytest.raises(RuntimeError, match="no torch headers"):
        build.build(verbose=False)
    assert (tmp_path / "libchadq.so").exists() and "libchadq.so.tmp" in linked
    assert build.build(verbose=False, host=False) == tmp_path / "libchadq.so"
