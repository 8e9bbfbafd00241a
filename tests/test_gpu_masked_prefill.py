"""Right-padded (masked) prefill on the fused path: the masked short
convolution against the unmasked one on masked rows, and the layer against its
general path, which a float mask of the same values takes."""

import pytest
import torch

from cyclic_flow_attention import CyclicFlowAttention, _native

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _mask(B, T, gen, kind):
    lengths = torch.randint(0, T + 1, (B,), generator=gen)
    lengths[0] = T
    lengths[-1] = min(T, 2) if kind == "short" else lengths[-1]
    mask = (torch.arange(T)[None, :] < lengths[:, None]).long()
    if kind == "holes":  # the mask need not be a prefix
        mask = mask * (torch.rand(B, T, generator=gen) < 0.8)
    return mask


# lengths shorter than the window, runs of 8 and 32 tokens with remainders,
# channel blocks with remainders, with and without a carried cache
@pytest.mark.parametrize("B,T,D,W,cache,kind", [(3, 5, 24, 4, True, "short"), (2, 64, 64, 3, False, "prefix"),
                                                (4, 130, 3072, 4, True, "holes"), (1, 33, 520, 2, False, "short"),
                                                (40, 700, 3072, 4, False, "prefix")])
def test_masked_short_conv_equals_convolution_of_masked_rows(B, T, D, W, cache, kind):
    gen = torch.Generator().manual_seed(B + T)
    x = torch.randn(B, T, D, generator=gen).bfloat16().to(DEV)
    w = (0.5 * torch.randn(D, W, generator=gen)).bfloat16().to(DEV)
    c = torch.randn(B, W - 1, D, generator=gen).bfloat16().to(DEV) if cache else None
    mask = _mask(B, T, gen, kind).to(DEV)
    values, valid, lengths = _native.mask_rows(mask)
    assert torch.equal(values, mask.bfloat16().float()) and torch.equal(valid.bool(), mask.bool())
    assert torch.equal(lengths.long(), mask.sum(1))
    xm = x * mask.bfloat16()[..., None]
    out = torch.empty(B, W - 1, D, dtype=torch.bfloat16, device=DEV)
    y, = _native.short_conv(x, w, None, c, cache_out=out, mask=values, lengths=lengths)
    ref, = _native.short_conv(xm, w, None, c)
    assert torch.equal(y, ref)
    history = torch.cat([torch.zeros(B, W - 1, D, dtype=x.dtype, device=DEV) if c is None else c, xm], 1)
    rows = lengths.long()[:, None] + torch.arange(W - 1, device=DEV)
    assert torch.equal(out, history[torch.arange(B, device=DEV)[:, None], rows])
    if cache and T <= 32:  # in place
        _native.short_conv(x, w, None, c, cache_out=c, mask=values, lengths=lengths)
        assert torch.equal(c, out)


@pytest.mark.parametrize("B,T,hidden,H,dtype,kind", [(2, 33, 256, 1, torch.bool, "prefix"),
                                                     (3, 192, 1024, 4, torch.int64, "holes"),
                                                     (5, 130, 1536, 6, torch.int32, "prefix"),
                                                     (2, 320, 2048, 11, torch.uint8, "short")])
@pytest.mark.parametrize("carried", [False, True])
def test_masked_layer_equals_general_path(B, T, hidden, H, dtype, kind, carried):
    """Same roundings on both paths; the fused q|k|v projection may sum in
    another order, which moves a bf16 value by one ulp here and there, and the
    output norm's sum of squares likewise: 2^-8 of the 2-norm (one rounding of
    every value) for y and the caches; the states are sums of such values."""
    gen = torch.Generator().manual_seed(T + H)
    torch.manual_seed(T)
    layer = CyclicFlowAttention(hidden_size=hidden, num_heads=H).eval()
    with torch.no_grad():
        for name, p in layer.named_parameters():
            if name.endswith("weight") and "norm" not in name:
                p.copy_((0.3 if "conv" in name else 0.02) * torch.randn(p.shape, generator=gen))
        for name, p in layer.named_parameters():
            if not any(s in name for s in ("norm.weight", "readout", "A_log", "dt_bias")):
                p.data = p.data.bfloat16()
    layer = layer.to(DEV)
    x = torch.randn(B, T, hidden, generator=gen).bfloat16().to(DEV)
    mask = _mask(B, T, gen, kind).to(DEV)
    with torch.no_grad():
        cache = layer(torch.randn(B, 70, hidden, generator=gen).bfloat16().to(DEV), use_cache=True)[1] if carried else None
        assert layer._fused_mask_ok(x, mask.to(dtype)) and not layer._fused_mask_ok(x, mask.float())
        y, got = layer(x, cache, use_cache=True, attention_mask=mask.to(dtype))
        ry, ref = layer(x, cache, use_cache=True, attention_mask=mask.float())
    pairs = [(y, ry)] + list(zip(got["recurrent_state"], ref["recurrent_state"]))
    pairs += list(zip(got["conv_state"], ref["conv_state"]))
    for a, b in pairs:
        assert a.shape == b.shape and a.dtype == b.dtype
        assert ((a.double() - b.double()).norm() <= 2.0 ** -8 * b.double().norm().clamp_min(1e-30)).item()


def test_masked_call_of_a_layer_with_hooks_calls_its_modules():
    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=256, num_heads=1).eval().bfloat16().to(DEV)
    x = torch.randn(2, 40, 256, dtype=torch.bfloat16, device=DEV)
    mask = torch.ones(2, 40, dtype=torch.long, device=DEV)
    mask[1, 30:] = 0
    seen = []
    with torch.no_grad():
        for m in (layer.q_proj, layer.g_proj[1], layer.k_conv1d, layer.o_norm, layer.o_proj):
            assert layer._fused_mask_ok(x, mask)
            hook = m.register_forward_pre_hook(lambda *_: seen.append(1))
            layer(x, attention_mask=mask)
            hook.remove()
        assert len(seen) == 5
        layer.v_proj = torch.nn.Sequential(layer.v_proj)
        assert not layer._fused_mask_ok(x, mask)


def test_masked_call_sees_weights_written_through_data():
    """An average of the weights copied in through ``.data``, and weights that
    come back at an address used before: no version counter tells of either."""
    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=256, num_heads=1).eval().bfloat16().to(DEV)
    x = torch.randn(2, 40, 256, dtype=torch.bfloat16, device=DEV)
    mask = torch.ones(2, 40, dtype=torch.long, device=DEV)
    mask[1, 30:] = 0
    with torch.no_grad():
        layer(x, attention_mask=mask)
        for p in (layer.q_proj.weight, layer.v_proj.weight, layer.k_conv1d.weight, layer.g_proj[0].weight,
                  layer.b_proj.weight, layer.d_proj.bias):
            p.data.copy_(0.1 * torch.randn(p.shape, device=DEV))
            y, ref = layer(x, attention_mask=mask)[0], layer(x, attention_mask=mask.float())[0]
            # (the paths' own difference, as in test_masked_layer_equals_general_path)
            assert ((y.double() - ref.double()).norm() <= 2.0 ** -8 * ref.double().norm()).item()


def test_masked_call_takes_operands_off_the_16_byte_grid():
    """x, and g_proj[1]'s weight, as views into larger buffers."""
    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=256, num_heads=1).eval().bfloat16().to(DEV)
    x = torch.randn(2, 40, 256, dtype=torch.bfloat16, device=DEV)
    mask = torch.ones(2, 40, dtype=torch.long, device=DEV)
    mask[1, 30:] = 0

    def off(t):
        return torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape).copy_(t)

    with torch.no_grad():
        y = layer(x, attention_mask=mask)[0]
        assert torch.equal(layer(off(x), attention_mask=mask)[0], y)
        layer.g_proj[1].weight.data = off(layer.g_proj[1].weight)
        assert torch.equal(layer(x, attention_mask=mask)[0], y)


def test_masked_call_past_the_convolution_launch_keeps_the_general_path(monkeypatch):
    """More tokens, or batch rows, than a launch of the convolution takes."""
    torch.manual_seed(0)
    layer = CyclicFlowAttention(hidden_size=256, num_heads=1).eval().bfloat16().to(DEV)
    x = torch.randn(3, 96, 256, dtype=torch.bfloat16, device=DEV)
    mask = torch.ones(3, 96, dtype=torch.long, device=DEV)
    with torch.no_grad():
        assert layer._fused_mask_ok(x, mask)
        monkeypatch.setattr(_native, "SHORT_CONV_MAX_GRID", 3)
        assert layer._fused_mask_ok(x, mask) and not layer._fused_mask_ok(x.repeat(2, 1, 1), mask.repeat(2, 1))
        assert not layer._fused_mask_ok(x.repeat(1, 2, 1), mask.repeat(1, 2))


def test_masked_call_applies_the_biases_of_replaced_modules():
    """Against the general path, which a float mask of the same values takes;
    each replacement changes the result, and what it adds is not lost."""
    from cyclic_flow_attention.layers.cyfa import ShortConvolution

    def layer():
        torch.manual_seed(1)
        return CyclicFlowAttention(hidden_size=256, num_heads=1).eval().bfloat16().to(DEV)

    gen = torch.Generator().manual_seed(2)
    x = torch.randn(2, 40, 256, generator=gen).bfloat16().to(DEV)
    mask = _mask(2, 40, gen, "prefix").to(DEV)
    with torch.no_grad():
        plain = layer()(x, attention_mask=mask)[0]

        def linear(n, bias=True):
            m = torch.nn.Linear(256, n, bias=bias)
            if bias:
                m.bias.copy_(torch.randn(n, generator=gen))
            return m

        def conv():
            m = ShortConvolution(256, 4, True)
            m.weight.copy_(0.3 * torch.randn(m.weight.shape, generator=gen))
            m.bias.copy_(torch.randn(256, generator=gen))
            return m

        for name, module in (("q_proj", linear(256)), ("a_proj", linear(1)), ("o_proj", linear(256)),
                             ("k_conv1d", conv()), ("b_proj", linear(1, False))):
            changed = layer()
            setattr(changed, name, module.bfloat16().to(DEV))
            y = changed(x, attention_mask=mask)[0]
            assert torch.equal(y, changed(x, attention_mask=mask.float())[0]), name
            assert _differs(y, plain), name


def _differs(a, b):
    return ((a.double() - b.double()).norm() > 2.0 ** -6 * b.double().norm()).item()
