"""Host-side checks of the training and masked-prefill entry points: struct
layouts against the header, and argument errors raised before any launch."""

import ctypes

import pytest
import torch

from cyclic_flow_attention import _native
from test_abi import _c_layout


@pytest.mark.parametrize("name", ["CyfaConvGradArgs", "CyfaGatePathArgs", "CyfaNormTrainArgs", "CyfaGatesTrainArgs"])
def test_struct_layout_matches_header(tmp_path, name):
    cls = getattr(_native, name)
    fields = [f for f, _ in cls._fields_]
    got = [ctypes.sizeof(cls)] + [getattr(cls, f).offset for f in fields]
    assert got == _c_layout(tmp_path, name, fields)


def test_short_conv_grad_validates_before_launch():
    lib = _native.load_library()
    n = lib.cyfa_short_conv_grad_workspace_bytes(2, 100, 64, 4)
    assert n >= 2 * 2 * 5 * 64 * 4 and lib.cyfa_short_conv_grad_workspace_bytes(2, 100, 64, 5) == 0
    good = dict(B=2, T=100, D=64, W=4, x=0x10000, x_row=64, weight=0x20000, dy=0x30000, workspace=0x40000,
                workspace_bytes=n)

    def call(dtype=0, **change):
        a = _native.CyfaConvGradArgs(**{**good, **change})
        return lib.cyfa_short_conv_grad(ctypes.byref(a), dtype, None)

    assert call(W=5) == call(D=60) == _native.CYFA_ERR_UNSUPPORTED
    assert call(dtype=7) == call(x=None) == call(T=0) == _native.CYFA_ERR_VALUE
    assert call(x=0x10004) == call(x_row=60) == call(dx=0x50002) == _native.CYFA_ERR_ALIGN
    assert call(workspace_bytes=n - 1) == _native.CYFA_ERR_WORKSPACE
    assert call(split=24) == call(split=16) == call(split=32) == call(D=40, split=20) == _native.CYFA_ERR_VALUE  # 32: no dy1
    assert call(split=32, dy1=0x30004) == call(dx_row=60) == call(dx_row=68) == _native.CYFA_ERR_ALIGN


def test_mask_entry_points_validate_before_launch():
    lib = _native.load_library()
    assert lib.cyfa_mask_rows(None, 1, 4, None, None, None, None) == _native.CYFA_ERR_VALUE
    c = _native.CyfaConvArgs(B=1, T=4, D=64, W=4, split=64, x=0x10000, x_row=64, weight=0x20000, mask=0x30000)
    c.out[0] = 0x40000
    assert lib.cyfa_short_conv(ctypes.byref(c), None) == _native.CYFA_ERR_VALUE  # mask without lengths


def test_norm_train_validates_before_launch():
    lib = _native.load_library()
    n = lib.cyfa_norm_grad_workspace_bytes(100, 256)
    assert n >= 256 * 4
    good = dict(rows=100, D=256, x=0x10000, weight=0x20000, out=0x30000, dy=0x40000, workspace=0x50000, workspace_bytes=n)

    def call(grad, dtype=0, **change):
        a = _native.CyfaNormTrainArgs(**{**good, **change})
        return lib.cyfa_norm_train(ctypes.byref(a), dtype, grad, None)

    assert call(0, D=258) == call(1, D=4096) == _native.CYFA_ERR_UNSUPPORTED
    past = _native.NORM_TRAIN_MAX_ROWS + 1  # past a grid of 2^32 threads
    size = lib.cyfa_norm_grad_workspace_bytes(past, 4)
    assert call(0, rows=past, D=4) == call(1, rows=past, D=4, workspace_bytes=size) == _native.CYFA_ERR_UNSUPPORTED
    assert call(0, out=None) == call(1, dy=None) == call(1, dgate=0x60000) == call(0, dtype=3) == _native.CYFA_ERR_VALUE
    assert call(0, x=0x10008) == _native.CYFA_ERR_ALIGN
    assert call(1, workspace_bytes=n - 4) == _native.CYFA_ERR_WORKSPACE


def test_gates_train_validates_before_launch():
    lib = _native.load_library()
    n = lib.cyfa_gates_grad_workspace_bytes(100, 256, 4)
    assert n >= (100 * 12 + 12 * 256) * 4
    names = [f for f, t in _native.CyfaGatesTrainArgs._fields_ if t is ctypes.c_void_p]
    good = dict(rows=100, K=256, H=4, workspace_bytes=n, **{f: 0x10000 * (i + 1) for i, f in enumerate(names)})

    def call(grad, dtype=0, **change):
        a = _native.CyfaGatesTrainArgs(**{**good, **change})
        return lib.cyfa_gates_train(ctypes.byref(a), dtype, grad, None)

    assert call(0, K=60) == call(1, H=9) == _native.CYFA_ERR_UNSUPPORTED
    assert call(0, rows=0) == call(0, g=None) == call(1, dwa=None) == call(0, dtype=2) == _native.CYFA_ERR_VALUE
    assert call(0, x=0x10008) == call(1, dx=0x10004) == _native.CYFA_ERR_ALIGN
    assert call(1, workspace_bytes=n - 4) == _native.CYFA_ERR_WORKSPACE


class _Recorder:
    """Stands in for the library: keeps the arguments of the one call made."""

    def __getattr__(self, name):
        def call(args, *rest):
            if name.endswith("_workspace_bytes"):
                return 64
            self.args = args._obj
            return _native.CYFA_OK

        return call


# [B, T, D] views whose size-1 dimensions carry strides that mean nothing, and
# ordinary ones: a time-major tensor's single step, one row of a longer batch,
# channels of a wider buffer, one batch row of a strided buffer
@pytest.mark.parametrize("make", [
    lambda: torch.zeros(1, 5, 8).transpose(0, 1), lambda: torch.zeros(5, 1, 24)[..., :8],
    lambda: torch.zeros(5, 3, 8)[:, 1:2], lambda: torch.zeros(1, 3, 11)[:, 1:2, :8],
    lambda: torch.zeros(2, 6, 24)[..., 8:16], lambda: torch.zeros(1, 12, 8)[:, ::2], lambda: torch.zeros(3, 6, 8)])
def test_short_conv_rows_are_where_the_kernels_read_them(monkeypatch, make):
    """The kernels read row (b, t) of x at (b T + t) x_row elements."""
    lib = _Recorder()
    monkeypatch.setattr(_native, "load_library", lambda: lib)
    monkeypatch.setattr(_native, "require_device", lambda *_: torch.device("cpu"))
    monkeypatch.setattr(_native, "stream_handle", lambda _: None)
    x, w = make(), torch.zeros(8, 4)
    seen = []
    monkeypatch.setattr(_native, "ptr", lambda t: seen.append(t) or (None if t is None else t.data_ptr()))

    def rows_read_back():
        xs = next(t for t in seen if t is not None and t.data_ptr() == lib.args.x)  # x, or its copy
        B, T, _ = xs.shape
        assert xs.shape == x.shape and xs.stride(2) == 1
        assert lib.args.x_row % 8 == 0 and lib.args.x_row >= 8
        for b in range(B):
            for t in range(T):
                assert xs[b, t].storage_offset() - xs.storage_offset() == (b * T + t) * lib.args.x_row

    _native.short_conv(x, w, None, torch.zeros(x.shape[0], 5, 11)[:, 1:4, :8].contiguous())
    rows_read_back()
    seen.clear()
    _native.short_conv(x, w[:, :2].contiguous(), None, torch.zeros(x.shape[0], 5, 11)[:, 1:2, :8].contiguous())
    assert lib.args.cache_row % 8 == lib.args.cache_batch % 8 == 0
    rows_read_back()
    seen.clear()
    if x.stride(2) == 1 and (x.is_contiguous() or x.shape[:2] == (2, 6)):  # rows the gradient's callers give it
        seen.clear()
        _native.short_conv_grad(x, w, None, torch.zeros(x.shape), (True, True, False, False))
        rows_read_back()
