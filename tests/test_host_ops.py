"""Host side of packkv_amd/ops.py: checks that come before any launch, on tensors without a GPU."""
import ctypes
import os
import subprocess
import sys

import pytest
import torch

from packkv_amd import _lib, ops


def test_rotary_tables_on_another_device_than_the_tokens_are_refused():
    """The kernels get bare addresses, so a host table must not pass: the tokens are on the meta device here."""
    like = torch.empty(2, 5, 7, 128, dtype=torch.float16, device="meta")
    here, there = torch.empty(2, 7, 128, dtype=torch.float16, device="meta"), torch.zeros(2, 7, 128, dtype=torch.float16)
    for cos, sin in ((there, there), (there, here), (here, there)):
        with pytest.raises(RuntimeError, match="one device"):
            ops._rotary_rows(cos, sin, like)


def test_dense_rows_have_no_limit_from_head_to_head():
    """2^24 tokens of five heads are 2^31 elements from head to head, which rows that lie 128 apart may have: the call comes
    as far as the check behind that one (8192 sequences are too many; nothing is launched).  Strided K is refused."""
    lib, at, size = _lib.load(), ctypes.c_void_p(4096), ctypes.c_uint64(0)
    T, H, B = 1 << 24, 5, 8192
    for fn in (lib.pkv_k_quant_encode, lib.pkv_v_quant_encode):
        assert fn(at, _lib.F16, B, H, T, 0.1, 4, at, 1 << 20, at, at, at, ctypes.byref(size), None, None) != 0
        assert b"batch x tokens too large" in lib.pkv_last_error()
    side = lambda st, sh: _lib.AppendSide(4096, H * sh, sh, st, 4096, 1 << 20, 0, 4096, 4096, 4096, 0.1, 4)
    for k, v, message in ((side(256, 1 << 31), side(256, 1 << 31), b"4 GiB or more"),
                          (side(256, (1 << 31) - 256), side(256, 1 << 31), b"batch x tokens too large"),
                          (side(128, 1 << 31), side(256, 1 << 31), b"batch x tokens too large")):
        assert lib.pkv_kv_quant_encode_append(ctypes.byref(k), ctypes.byref(v), _lib.F16, B, H, T, T, ctypes.byref(size),
                                              ctypes.byref(size), None) != 0
        assert message in lib.pkv_last_error(), lib.pkv_last_error()


def test_rows_that_the_encoders_cannot_reach_are_copied():
    """What window_cut copies before the encode: the token and head strides that the entry point refuses, and no others."""
    rows = lambda H, sh, st: torch.empty_strided((1, H, 256, 128), (0, sh, st, 1), dtype=torch.float16, device="meta")
    for H, sh, st, want in ((5, 1 << 31, 128, True), (5, 1 << 31, 256, False), (4, 1 << 31, 256, True), (5, (1 << 31) - 136, 256, True),
                            (5, (1 << 31) - 128, 256, False), (5, 128, 1 << 25, False), (4, 128, 1 << 25, False),
                            (5, 128, (1 << 25) - 8, True), (5, 128, 1284, False), (1, 7, 256, True)):
        x = rows(H, sh, st)
        assert ops._encodable(x, ops._strides(x)) == want, (H, sh, st)


def test_import_without_the_private_torch_functions():
    """The two look-ups that torch does not promise: without them the module imports and asks torch.cuda instead."""
    code = """
import types, torch
del torch._C._cuda_getCurrentRawStream, torch._C._cuda_getDevice
torch.cuda.current_device = lambda: 3
torch.cuda.current_stream = lambda device=None: types.SimpleNamespace(cuda_stream=100 + device)
from packkv_amd import ops
assert ops._stream(torch.device("cuda")) == 103 and ops._stream(torch.device("cuda", 1)) == 101
assert ops._on(torch.device("cuda", 3)) is ops._here
"""
    subprocess.run([sys.executable, "-c", code], check=True, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), timeout=300)


@pytest.mark.parametrize("module", ["None", "types.SimpleNamespace(torch='0.0')"])
def test_without_the_native_host_side_the_library_loads_and_the_general_code_serves(module):
    """_host.so missing, not loadable, or built for another torch: a warning, and calls come as far as they do in ops.py."""
    code = """
import sys, types, warnings
import packkv_amd
sys.modules["packkv_amd._host"] = %s
if sys.modules["packkv_amd._host"]:
    packkv_amd._host = sys.modules["packkv_amd._host"]
import torch
from packkv_amd import _lib, ops
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    assert _lib.load().pkv_abi_version() == 3
assert any("_host" in str(w.message) for w in seen), seen
assert _lib.host is _lib.NO_HOST and _lib.host.attn_decode(1, 2) is None
try:
    ops.attn_decode(torch.zeros(1, 8, 128, dtype=torch.float16), None, None)
except RuntimeError as e:
    assert "q must be a contiguous device tensor" in str(e), e
else:
    raise SystemExit("accepted")
""" % module
    subprocess.run([sys.executable, "-c", code], check=True, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))), timeout=300)


def test_the_native_host_side_is_the_one_of_this_torch():
    _lib.load()
    assert _lib.host is not _lib.NO_HOST and _lib.host.torch == torch.__version__


def test_what_is_refused_needs_no_library(monkeypatch):
    """Without libpackkv_hip.so a call that is refused says why, and any other one that the library is missing."""
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "host", None)
    monkeypatch.setattr(_lib, "LIB_PATH", os.path.join(os.path.dirname(_lib.LIB_PATH), "nowhere.so"))
    with pytest.raises(RuntimeError, match="q must be a 2D tensor"):
        ops.fused_kq(*(torch.zeros(2, dtype=torch.float16) for _ in range(5)))
    with pytest.raises(ImportError, match="not built"):
        ops.block_bound(True, 64, 128, 4)


def test_host_tensors_are_refused_by_name():
    """The tensor is looked at before the runtime is asked for its device: there may be no GPU."""
    half = lambda *s: torch.zeros(*s, dtype=torch.float16)
    side = {"stream": torch.zeros(64, dtype=torch.uint8), "info": torch.zeros(2, 2, dtype=torch.uint32), "scale": half(1, 128), "zero": half(1, 128), "bits": 4}
    stream, info = side["stream"], side["info"]
    for call, message in ((lambda: ops.attn_decode(half(1, 8, 128), side, side), "q must be a contiguous device tensor"),
                          (lambda: ops.window_append(half(1, 2, 1, 128), half(1, 2, 1, 128), None, None, half(1, 2, 8, 128), half(1, 2, 8, 128), 0),
                           "K and V must be device tensors"),
                          (lambda: ops.dense_view(side, side), "a compressed cache is on a GPU"),
                          (lambda: ops.kq_mat_vec_mul(stream, info, half(1, 128), half(1, 64), 64, 128, 64, 128, 4), "tensor must be a CUDA tensor"),
                          (lambda: ops.wv_mat_vec_mul(stream, info, half(1, 128), torch.zeros(1, 128), 128, 128, 128, 64, 4), "tensor must be a CUDA tensor"),
                          (lambda: ops.fused_kq(half(1, 64), half(1, 128), half(64), half(64), half(1, 64)), "q must be a CUDA tensor"),
                          (lambda: ops.fused_wv(half(1, 128), half(1, 64), half(64), half(64), half(1, 128)), "w must be a CUDA tensor")):
        with pytest.raises(RuntimeError, match=message):
            call()
    assert _lib.host.plan_step(4096, 0, 1, half(1, 8, 128)) is None


def test_a_plan_that_another_thread_drops_meanwhile_serves_the_step_that_has_it():
    """attend looks at the layer's plan once: an update that cuts drops it at any time."""
    from packkv_amd import cache as pc

    class Plan:
        sm_scale_arg = None

        def step(self, q, rows):
            return q, rows

    class Layer:
        win_len, plans = 3, [Plan()]

        @property
        def plan(self):
            return self.plans.pop() if self.plans else None
    cache = pc.PackKVCompressedCache(1, 2, 128, 1, device="cpu")
    cache.layers[0] = Layer()
    q = torch.zeros(1, 2, 128)
    assert cache.attend(q, 0) == (q, 3)
