"""GPU parity of the LoRA add (wf_dequant_add, the role of the reference's _deq_add, enhancers/gguf_dequant.py:
99-133) against the oracle, bit for bit: the first LoRA fused into the dequantisation for every format and every
MID / OUT pair, later LoRAs onto an existing weight (ragged tail included), and the drop-in Python path
(dequantize_lora, the patched get_weight) with two LoRAs whose differences come from the same torch.mm."""
import numpy as np
import pytest
import torch

from conftest import sub
from oracle import lib, np_oracle

encode = sub("gguf_encode")

pytestmark = pytest.mark.gpu

F16, BF16, F32 = 0, 1, 2
TD = {F16: torch.float16, BF16: torch.bfloat16, F32: torch.float32}
ALL_TYPES = [2, 3, 6, 7, 8, 10, 11, 12, 13, 14]
PAIRS = [(m, o) for m in range(3) for o in range(3)]


def _bits(t, D):
    t = t.cpu()
    if D == F32:
        return t.numpy().astype(np.float32).ravel()
    return t.contiguous().view(torch.int16).numpy().view(np.uint16).ravel()


def _same(a, b, D):
    fa, fb = np_oracle.bits_to_f32(a, D), np_oracle.bits_to_f32(b, D)
    eq = np.asarray(a).view(np.uint8).reshape(fa.size, -1) == np.asarray(b).view(np.uint8).reshape(fb.size, -1)
    ok = eq.all(axis=1) | (np.isnan(fa) & np.isnan(fb))
    return bool(ok.all()), np.nonzero(~ok)[0][:8]


@pytest.mark.parametrize("qtype", ALL_TYPES)
def test_first_lora_fused_into_dequant(native, qtype):
    nblk = 2047 if encode.PER_BLOCK[qtype] == 256 else 8191
    n = nblk * encode.PER_BLOCK[qtype]
    raw = encode.random_blocks(qtype, nblk, seed=500 + qtype, family="normal")
    diff = (np.random.default_rng(qtype).standard_normal(n) * 0.02).astype(np.float32)
    raw_dev, diff_dev = torch.from_numpy(raw).cuda(), torch.from_numpy(diff).cuda()
    for mid, out in PAIRS:
        res = torch.empty(n, dtype=TD[out], device="cuda")
        print(f"case qtype={qtype} mid={mid} out={out} n={n}", flush=True)
        rc = native.lib().wf_dequant_add(raw_dev.data_ptr(), raw_dev.numel(), qtype, mid, out, diff_dev.data_ptr(),
                                         0.4375, res.data_ptr(), n, native.stream_of(res.device))
        assert rc == 0, native.last_error()
        torch.cuda.synchronize()
        ok, where = _same(_bits(res, out), lib.dequant_add(raw, qtype, mid, out, diff, 0.4375), out)
        assert ok, (qtype, mid, out, where)


@pytest.mark.parametrize("out", [F16, BF16, F32])
@pytest.mark.parametrize("n", [8, 1_000_003, 5120 * 5120])
def test_later_lora_onto_weight(native, out, n):
    rng = np.random.default_rng(n + out)
    w = torch.from_numpy(rng.standard_normal(n).astype(np.float32) * 0.05).to(TD[out])
    diff = (rng.standard_normal(n) * 0.01).astype(np.float32)
    base = _bits(w, out)
    wd, dd = w.cuda(), torch.from_numpy(diff).cuda()
    print(f"case out={out} n={n}", flush=True)
    rc = native.lib().wf_dequant_add(None, 0, 0, 0, out, dd.data_ptr(), -1.25, wd.data_ptr(), n,
                                     native.stream_of(wd.device))
    assert rc == 0, native.last_error()
    torch.cuda.synchronize()
    ok, where = _same(_bits(wd, out), lib.dequant_add(None, 0, 0, out, diff, -1.25, base=base), out)
    assert ok, where


# rows around the kernel's 32-row tiles, columns around its 256 (one block, a ragged last tile), odd and largest ranks
@pytest.mark.parametrize("qtype,n_out,n_in,rank", [
    (7, 1, 32, 1), (8, 33, 288, 7), (3, 31, 256, 8), (2, 64, 544, 33), (6, 40, 1024, 64), (12, 32, 256, 16),
    (13, 65, 512, 2), (14, 33, 768, 24), (10, 7, 256, 192), (11, 96, 512, 5), (None, 33, 264, 12), (None, 3, 8, 192)])
def test_lora_product_inside_the_kernel(native, qtype, n_out, n_in, rank):
    # factors of small integers: every float32 sum of their products is exact, so the result is one set of bits
    rng = np.random.default_rng(rank + n_in)
    ups, downs = (rng.integers(-8, 9, s).astype(np.float32) for s in ((n_out, rank), (rank, n_in)))
    diff = (ups.astype(np.float64) @ downs).astype(np.float32).ravel()
    n = n_out * n_in
    for mid, out in (PAIRS if qtype is not None else [(F16, o) for o in (F16, BF16, F32)]):
        udt, ddt = TD[(mid + out) % 3], TD[out]
        up, down = torch.from_numpy(ups).to("cuda", udt), torch.from_numpy(downs).to("cuda", ddt)
        if qtype is not None:
            raw = encode.random_blocks(qtype, n // encode.PER_BLOCK[qtype], seed=qtype, family="normal")
            raw_dev, res = torch.from_numpy(raw).cuda(), torch.empty(n, dtype=TD[out], device="cuda")
            blocks, expect = (raw_dev.data_ptr(), raw_dev.numel(), qtype, mid), lib.dequant_add(raw, qtype, mid, out, diff,
                                                                                                0.0078125)
        else:
            w = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).to(TD[out])
            res, blocks = w.cuda(), (None, 0, 0, 0)
            expect = lib.dequant_add(None, 0, 0, out, diff, 0.0078125, base=_bits(w, out))
        print(f"case qtype={qtype} {n_out}x{n_in} rank={rank} mid={mid} out={out}", flush=True)
        rc = native.lib().wf_dequant_lora(*blocks, out, up.data_ptr(), (mid + out) % 3, down.data_ptr(), out, rank,
                                          0.0078125, res.data_ptr(), n_out, n_in, native.stream_of(res.device))
        assert rc == 0, native.last_error()
        torch.cuda.synchronize()
        ok, where = _same(_bits(res, out), expect, out)
        assert ok, (mid, out, where)


class LoRAAdapter:
    def __init__(self, weights):
        self.weights = weights


def _patch(up, down, alpha, strength):
    return (strength, LoRAAdapter((up, down, alpha, None, None, None)), 1.0, None, None)


def _expected(raw, qtype, mid, out, n_out, n_in, loras):
    """the oracle's chain with each difference from the same torch.mm the drop-in calls (float32 on the GPU)"""
    res = None
    for i, (up, down, sa) in enumerate(loras):
        diff = torch.mm(up.to("cuda", torch.float32), down.to("cuda", torch.float32)).cpu().numpy().ravel()
        if i == 0:
            res = lib.dequant_add(raw, qtype, mid, out, diff, sa)
        else:
            res = lib.dequant_add(None, 0, 0, out, diff, sa, base=res)
    return res


@pytest.mark.parametrize("qtype,mid", [(8, torch.float16), (12, torch.float16), (14, torch.bfloat16), (3, None)])
def test_dequantize_lora_two_loras(native, qtype, mid):
    gd = sub("enhancers.gguf_dequant")
    n_out, n_in = 384, 1024
    if qtype in encode.ENCODERS:
        raw = encode.encode(encode.weights((n_out, n_in), seed=qtype), qtype)
    else:
        raw = encode.random_blocks(qtype, n_out * n_in // encode.PER_BLOCK[qtype], seed=qtype, family="normal")
    g = torch.Generator().manual_seed(qtype)
    ups = [torch.randn((n_out, 16), generator=g).to(torch.bfloat16), torch.randn((n_out, 8), generator=g)]
    downs = [torch.randn((16, n_in), generator=g).to(torch.bfloat16), torch.randn((8, n_in), generator=g)]
    loras = gd.lora_factors([_patch(ups[0], downs[0], 8.0, 0.7), _patch(ups[1], downs[1], None, -0.3)], n_out, n_in)
    y = gd.dequantize_lora(torch.from_numpy(raw).cuda(), qtype, (n_out, n_in), mid, torch.bfloat16, loras)
    torch.cuda.synchronize()
    assert y.shape == (n_out, n_in) and y.dtype == torch.bfloat16
    m = {None: F16, torch.float16: F16, torch.bfloat16: BF16}[mid]
    expect = _expected(raw, qtype, m, BF16, n_out, n_in, loras)
    ok, where = _same(_bits(y, BF16), expect, BF16)
    assert ok, where
    # not this path's case: CPU data, no LoRA, a 1-D shape
    assert gd.dequantize_lora(torch.from_numpy(raw), qtype, (n_out, n_in), mid, torch.bfloat16, loras) is None
    assert gd.dequantize_lora(torch.from_numpy(raw).cuda(), qtype, (n_out, n_in), mid, torch.bfloat16, []) is None
    assert gd.dequantize_lora(torch.from_numpy(raw).cuda(), qtype, (n_out * n_in,), mid, torch.bfloat16, loras) is None


def test_patched_get_weight_with_lora(native, fake_gguf):
    gd = sub("enhancers.gguf_dequant")
    ops = fake_gguf
    assert gd.install(force=True)
    try:
        n_out, n_in = 256, 512
        raw = encode.encode(encode.weights((n_out, n_in), seed=3), 13)
        g = torch.Generator().manual_seed(3)
        up, down = torch.randn((n_out, 4), generator=g), torch.randn((4, n_in), generator=g)
        t = ops.GGMLTensor(torch.from_numpy(raw).cuda(), tensor_type=13, tensor_shape=torch.Size((n_out, n_in)),
                           patches=[([_patch(up, down, 2.0, 0.5)], "key")])
        gd.stats(reset=True)
        y = ops.GGMLLayer().get_weight(t, torch.bfloat16)
        torch.cuda.synchronize()
        assert gd.stats().get("lora_used") == 1
        loras = gd.lora_factors([_patch(up, down, 2.0, 0.5)], n_out, n_in)
        ok, where = _same(_bits(y, BF16), _expected(raw, 13, F16, BF16, n_out, n_in, loras), BF16)
        assert ok, where
    finally:
        gd.uninstall()


def test_inference_mode_factors_use_the_kernel(native, fake_gguf):
    # ComfyUI runs under torch.inference_mode and its LoRA factors are inference tensors (no version counter): the
    # pinned-factor path must take them (lora_used), reuse their page-locked copies on the next call, and give the
    # same bits as the oracle's chain
    gd = sub("enhancers.gguf_dequant")
    ops = fake_gguf
    assert gd.install(force=True)
    try:
        n_out, n_in = 256, 512
        raw = encode.encode(encode.weights((n_out, n_in), seed=4), 12)
        g = torch.Generator().manual_seed(4)
        with torch.inference_mode():
            up, down = torch.randn((n_out, 8), generator=g), torch.randn((8, n_in), generator=g)
            t = ops.GGMLTensor(torch.from_numpy(raw).cuda(), tensor_type=12, tensor_shape=torch.Size((n_out, n_in)),
                               patches=[([_patch(up, down, 4.0, 0.75)], "key")])
            gd.stats(reset=True)
            held_before = len(gd._PINNED)
            ys = [ops.GGMLLayer().get_weight(t, torch.bfloat16) for _ in range(2)]
            torch.cuda.synchronize()
        assert gd.stats().get("lora_used") == 2 and "lora_fallback" not in gd.stats()
        assert len(gd._PINNED) == held_before + 2          # one page-locked copy per factor, reused by the 2nd call
        loras = gd.lora_factors([_patch(up, down, 4.0, 0.75)], n_out, n_in)
        expect = _expected(raw, 12, F16, BF16, n_out, n_in, loras)
        for y in ys:
            ok, where = _same(_bits(y, BF16), expect, BF16)
            assert ok, where
    finally:
        gd.uninstall()


def _integer_loras(shapes, n_out, n_in, dtypes):
    """LoRAs whose factors are small integers: every float32 sum is exact, so the result is one set of bits."""
    g = torch.Generator().manual_seed(sum(shapes))
    return [(torch.randint(-8, 9, (n_out, r), generator=g).to(d), torch.randint(-8, 9, (r, n_in), generator=g).to(d), s)
            for r, d, s in zip(shapes, dtypes, (0.0078125, -0.00390625))]


@pytest.mark.parametrize("ranks,dtypes", [
    ((256,), (torch.bfloat16,)), ((130,), (torch.float16,)), ((80,), (torch.float32,)), ((8,), (torch.float64,)),
    ((16, 256), (torch.bfloat16, torch.bfloat16)), ((256, 16), (torch.float32, torch.bfloat16)),
    ((200, 96), (torch.bfloat16, torch.float32))])
def test_loras_beside_the_kernel(native, monkeypatch, ranks, dtypes):
    # LoRAs that take torch.mm's difference (high ranks, float64), alone and before or after one that the kernel computes
    gd = sub("enhancers.gguf_dequant")
    n_out, n_in = 96, 512
    raw = encode.random_blocks(13, n_out * n_in // 256, seed=5, family="normal")
    loras = _integer_loras(ranks, n_out, n_in, dtypes)
    routes, plain = [], gd._add_difference
    monkeypatch.setattr(gd, "_add_difference", lambda *a: routes.append(a[1].shape[1]) or plain(*a))
    for out, D in ((torch.bfloat16, BF16), (torch.float32, F32)):
        del routes[:]
        y = gd.dequantize_lora(torch.from_numpy(raw).cuda(), 13, (n_out, n_in), None, out, loras)
        assert routes == [r for r in ranks if r != 16]
        torch.cuda.synchronize()
        ok, where = _same(_bits(y, D), _expected(raw, 13, F16, D, n_out, n_in, loras), D)
        assert ok, where


def test_lora_factor_the_kernel_declines(native):
    # a device factor that starts at an odd value: not aligned to a pair of values, so the kernel declines it
    gd = sub("enhancers.gguf_dequant")
    n_out, n_in = 64, 256
    raw = encode.random_blocks(8, n_out * n_in // 32, seed=6, family="normal")
    (up, down, s), = _integer_loras((16,), n_out, n_in, (torch.bfloat16,))
    shifted = torch.zeros(down.numel() + 1, dtype=down.dtype, device="cuda")[1:].view(down.shape)
    shifted.copy_(down)
    up = up.cuda()
    assert shifted.data_ptr() % 4 == 2 and shifted.is_contiguous()
    res = torch.zeros((n_out, n_in), dtype=torch.bfloat16, device="cuda")
    rc = native.lib().wf_dequant_lora(None, 0, 0, 0, BF16, up.data_ptr(), BF16, shifted.data_ptr(), BF16, 16, s,
                                      res.data_ptr(), n_out, n_in, native.stream_of(res.device))
    assert rc == native.EUNSUPPORTED
    y = gd.dequantize_lora(torch.from_numpy(raw).cuda(), 8, (n_out, n_in), None, torch.bfloat16, [(up, shifted, s)])
    torch.cuda.synchronize()
    ok, where = _same(_bits(y, BF16), _expected(raw, 8, F16, BF16, n_out, n_in, [(up, down, s)]), BF16)
    assert ok, where
