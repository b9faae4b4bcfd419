"""Host-side behaviour of enhancers.fused_int8 on the CPU: _Overrides installs and removes the per-call _forward
and the shared-quantisation cache (enhancers/fused_int8.py:311-332 of the reference); _int8_quantised declines
every case outside the reference's eligibility (:129-147), and _shared_forward then runs
torch.nn.functional.linear and counts the fallback (:279-292); a pending input is materialised for the fallback."""
import ctypes

import pytest
import torch

from conftest import sub
from fake_quant import FakeQT, Lin

fi = sub("enhancers.fused_int8")
fs = sub("enhancers.fused_state")
native = sub("_native")


def _weight(n=16, k=256, **kw):
    g = torch.Generator().manual_seed(n + k)
    w_q = torch.randint(-127, 128, (n, k), generator=g, dtype=torch.int64).to(torch.int8)
    return FakeQT(w_q, torch.full((n,), 0.01), **kw)


def test_overrides_install_and_restore():
    lins = [Lin(_weight()), Lin(_weight())]
    special = lambda i, w, b: "special"  # noqa: E731
    with fi._Overrides([lins[0], (lins[1], special)]) as ov:
        assert lins[0].__dict__["_forward"] is fi._shared_forward
        assert lins[1].__dict__["_forward"] is special
        assert fi._tls.qkv == {} and not ov.outer
        with fi._Overrides([lins[0]]) as inner:        # already overridden: left alone; outer cache kept
            assert inner.outer and inner.layers == []
        assert fi._tls.qkv == {}
    assert "_forward" not in lins[0].__dict__ and "_forward" not in lins[1].__dict__
    assert getattr(fi._tls, "qkv", None) is None


def test_ineligible_cases_return_none():
    x = torch.randn(8, 256).to(torch.bfloat16)
    fi._tls.qkv = {}
    try:
        assert fi._int8_quantised(x, _weight(), None) is None                          # CPU input
        assert fi._int8_quantised(x, _weight(), torch.zeros(16)) is None               # bias
        assert fi._int8_quantised(x, _weight(convrot=False), None) is None             # not ConvRot
        assert fi._int8_quantised(x, _weight(transposed=True), None) is None
        assert fi._int8_quantised(x, _weight(groupsize=128), None) is None
        assert fi._int8_quantised(x, torch.zeros(16, 256), None) is None               # not a quantized weight
    finally:
        fi._tls.qkv = None
    assert fi._int8_quantised(x, _weight(), None) is None                              # outside _Overrides


def test_shared_forward_falls_back_and_counts():
    fs.stats(reset=True)
    w = _weight()
    x = torch.randn(4, 256).to(torch.bfloat16)
    lin = Lin(w)
    with fi._Overrides([lin]):
        y = lin(x)
    ref = torch.nn.functional.linear(x, w.as_subclass(torch.Tensor))
    assert torch.equal(y, ref)
    st = fs.stats()
    assert st["qkv"]["fallback"] == 1 and st["qkv"]["used"] == 0 and "FakeQT" in st["qkv"]["why"]


def test_pending_input_is_materialised_for_the_fallback():
    fs.stats(reset=True)
    w = _weight()
    x = torch.randn(4, 256).to(torch.bfloat16)
    scale, shift = torch.full((256,), 0.5).to(torch.bfloat16), torch.full((256,), 0.25).to(torch.bfloat16)
    pre = fi._set_pre(x, "mod", scale=scale, shift=shift)
    lin = Lin(w)
    with fi._Overrides([lin]):
        y = lin(x)
    fi._clear_pre()
    assert pre["used"]
    real = x * (1 + scale) + shift
    assert torch.equal(y, torch.nn.functional.linear(real, w.as_subclass(torch.Tensor)))


def test_residual_forward_without_pending_residual_is_shared_forward():
    w = _weight()
    x = torch.randn(4, 256).to(torch.bfloat16)
    fi._tls.res = None
    y = fi._residual_forward(x, w, None)
    assert torch.equal(y, torch.nn.functional.linear(x, w.as_subclass(torch.Tensor)))


def test_int8_linear_declines_cpu():
    assert fi.int8_linear(torch.randn(4, 256).to(torch.bfloat16), torch.zeros(8, 256, dtype=torch.int8),
                          torch.ones(8)) is None


def _plan(M, N, K, workspace=1 << 62):
    p = native.I8Plan()
    rc = native.lib().wf_linear_i8_plan(M, N, K, workspace, ctypes.byref(p))
    return rc, p


@pytest.mark.parametrize("M,N,K,tile", [
    # the shapes whose modelled tiling measured slower than the one they had
    (600, 13824, 5120, (256, 256)), (135, 8256, 1920, (128, 160)), (197, 6975, 2560, (128, 160)),
    (6, 7744, 7168, (128, 160)), (25, 12560, 6144, (128, 160)), (303, 4848, 2176, (128, 160)),
    (700, 8048, 11264, (256, 128)), (746, 8544, 7680, (256, 128)), (867, 8288, 5888, (256, 256)),
    (219, 11464, 1280, (128, 160)), (2718, 2138, 1152, (256, 128)), (434, 13264, 12928, (256, 128)),
    # those the tests of the tilings name
    (4000, 5000, 512, (256, 320)), (3000, 3000, 384, (256, 256)), (2000, 4000, 640, (256, 128)),
    (1024, 5000, 512, (128, 160)), (1024, 4992, 128, (128, 160))])
def test_plan_keeps_the_tilings_that_measured_faster(M, N, K, tile):
    for workspace in (0, 1 << 62):
        rc, p = _plan(M, N, K, workspace)
        if p.slices == 1:
            assert rc == 0 and (p.tile_rows, p.tile_columns) == tile and p.workspace_bytes == 0


@pytest.mark.parametrize("M,N,K", [(746, 2592, 4608), (746, 8544, 7680), (434, 13264, 12928), (4748, 1404, 11776),
                                   (1275, 5949, 9728), (679, 1888, 3328), (2826, 1936, 9984), (1094, 1464, 6272)])
def test_plan_leaves_out_slices_that_measured_slower(M, N, K):
    rc, p = _plan(M, N, K)
    assert rc == 0 and p.slices == 1 and p.workspace_bytes == 0


def test_plan_query():
    need = ctypes.c_int64()
    for M, N, K in ((256, 5120, 5120), (1560, 5120, 13824), (16, 5120, 5120)):
        rc, p = _plan(M, N, K)
        assert rc == 0 and p.slices > 1 and p.whole_ns > 20000
        assert native.lib().wf_linear_i8_workspace(M, N, K, ctypes.byref(need)) == 0 and need.value == p.workspace_bytes
        rc, q = _plan(M, N, K, p.workspace_bytes - 1)            # fewer slices, or none
        assert rc == 0 and q.workspace_bytes < p.workspace_bytes
        assert _plan(M, N, K, 0)[1].slices == 1
    rc, p = _plan(300, 1000, 208)                                # the kernel for K % 64 != 0
    assert rc == 0 and p.tile_rows == 0 and p.slices == 1 and p.whole_ns == 0
    assert _plan(0, 8, 128)[0] == native.EINVAL and _plan(8, 8, 0)[0] == native.EINVAL
    assert _plan(8, 8, 131088)[0] == native.EUNSUPPORTED and _plan(8, 8, 24)[0] == native.EUNSUPPORTED
    assert native.lib().wf_linear_i8_plan(8, 8, 128, 0, None) == native.EINVAL


class _Calls:
    """The native library with its int8 products recorded instead of run."""

    def __init__(self):
        self.names, self.real = [], native.lib()

    def __getattr__(self, name):
        if name not in ("wf_linear_i8", "wf_linear_i8_residual", "wf_linear_i8_ws"):
            return getattr(self.real, name)
        return lambda *a: self.names.append(name) or self.rc

    rc = 0


def _products(monkeypatch, calls, m, n, k, least_ns, residual=False):
    """The entry points one product goes through."""
    monkeypatch.setattr(native, "lib", lambda: calls)
    monkeypatch.setattr(fi, "_stream", lambda dev: None)
    x_q, w_q = torch.empty((m, k), dtype=torch.int8), torch.empty((n, k), dtype=torch.int8)
    x_s, ws = torch.empty((m, 1)), torch.empty(n)
    out = torch.empty((m, n), dtype=torch.bfloat16)
    gate = out[:1] if residual else None
    assert fi._linear_i8(x_q, x_s, w_q, ws, None, gate, out if residual else None, out, m, least_ns)
    return calls.names


@pytest.mark.parametrize("m,n,k,direct,block", [
    (64, 2048, 2048, False, False), (150, 2048, 2048, False, False), (64, 1111, 4096, False, False),   # shorter than a call
    (16, 5120, 5120, True, False), (256, 5120, 5120, True, False), (300, 2048, 8192, True, False),
    (16, 5120, 13824, True, False),                                                  # longer than int8_linear's call
    (1560, 5120, 13824, True, True), (5152, 2048, 8192, False, False)])              # longer than a block's layer
def test_slices_only_where_the_call_is_longer_than_its_host_time(monkeypatch, m, n, k, direct, block):
    assert _products(monkeypatch, _Calls(), m, n, k, fi._LEAST_NS) == ["wf_linear_i8_ws" if direct else "wf_linear_i8"]
    assert _products(monkeypatch, _Calls(), m, n, k, fi._BLOCK_LEAST_NS) == ["wf_linear_i8_ws" if block else "wf_linear_i8"]
    assert _products(monkeypatch, _Calls(), m, n, k, fi._BLOCK_LEAST_NS, residual=True) == [
        "wf_linear_i8_ws" if block else "wf_linear_i8_residual"]


def test_failures_name_the_entry_point_that_ran(monkeypatch):
    calls = _Calls()
    calls.rc = native.EINVAL
    for m, n, k, residual, name in ((8, 64, 256, False, "wf_linear_i8"), (8, 64, 256, True, "wf_linear_i8_residual"),
                                    (16, 5120, 5120, False, "wf_linear_i8_ws")):
        with pytest.raises(native.NativeError, match=name + " failed"):
            _products(monkeypatch, calls, m, n, k, 0, residual)


def test_no_memory_for_slices_runs_the_product_whole(monkeypatch):
    real, asked = torch.empty, []

    def empty(*shape, **kw):
        if kw.get("dtype") == torch.uint8:
            asked.append(shape)
            raise torch.OutOfMemoryError("no memory")
        return real(*shape, **kw)
    x = [real((16, 13824), dtype=torch.int8), real((16, 1)), real((5120, 13824), dtype=torch.int8), real(5120)]
    calls = _Calls()
    monkeypatch.setattr(native, "lib", lambda: calls)
    monkeypatch.setattr(fi, "_stream", lambda dev: None)
    monkeypatch.setattr(torch, "empty", empty)
    assert fi.gemm(*x) is not None and calls.names == ["wf_linear_i8"] and len(asked) == 1
    out = real((16, 5120), dtype=torch.bfloat16)
    assert fi._linear_i8(*x, None, out[:1], out, out, 16, 0) and calls.names[1:] == ["wf_linear_i8_residual"]
