"""The one-pass norm + RoPE + transposition of the processors' projections (``svoo_qkv_heads``) against the separate
tensor operations it stands in for, and the cases in which those have to run."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


class Layer(torch.nn.Module):
    """Projections and norms under the names the processors read."""

    def __init__(self, heads, d, norm_width, gpu, double=False, fused=False):
        super().__init__()
        dim = heads * d
        kw = dict(dtype=torch.bfloat16, device=gpu)
        self.heads = heads
        self.fused_projections = fused
        if fused:
            self.to_qkv = torch.nn.Linear(dim, 3 * dim, **kw)
            self.cross_attention_dim_head = None
        names = [] if fused else ["to_q", "to_k", "to_v"]
        norms = ["norm_q", "norm_k"]
        if double:
            names += ["add_q_proj", "add_k_proj", "add_v_proj"]
            norms += ["norm_added_q", "norm_added_k"]
        for n in names:
            setattr(self, n, torch.nn.Linear(dim, dim, **kw))
        for n in norms:
            m = torch.nn.RMSNorm(norm_width, eps=1e-6, **kw)
            torch.nn.init.uniform_(m.weight, 0.5, 1.5)
            setattr(self, n, m)
        self.requires_grad_(False)


def _tables(rows, d, gpu):
    ang = torch.rand(rows, d, device=gpu) * 6.0  # each element its own angle: the forms differ in which they take
    return ang.cos(), ang.sin()


def _processor(base):
    """A processor whose attention hands back the heads it was given."""

    class P(base):
        def attention_core_logic(self, query, key, value, *a):
            self.got = (query, key, value)
            return query if base.__name__.startswith("Hunyuan") else query.transpose(1, 2).flatten(2, 3)

        def get_o(self, *a):
            return None

    return P(layer_idx=0)


def _heads(proc, layer, x, separate, monkeypatch, **kw):
    from svoo_amd import _lib, heads

    calls = []
    real = _lib.call
    with monkeypatch.context() as m:
        m.setattr(_lib, "call", lambda name, *a: (calls.append(name), real(name, *a))[1])
        if separate:
            m.setattr(heads, "plain_execution", lambda: False)
        proc(layer, x, timestep=torch.zeros(1), **kw)
    assert all(t.is_contiguous() for t in proc.got)
    return [t.clone() for t in proc.got], calls.count("svoo_qkv_heads")


def _close(got, want):
    """The norm's sums may round differently in another order: rstd moves by a few 2^-24, so a normed element moves by
    at most one bf16 step (2^-8 of it) and a rotated pair by 2^-8 (|x0| + |x1|) and its own rounding."""
    for g, w in zip(got, want):
        g, w = g.double(), w.double()
        pair = w.unflatten(-1, (-1, 2)).abs().sum(-1, keepdim=True).expand(*w.shape[:-1], w.shape[-1] // 2, 2).flatten(-2)
        assert ((g - w).abs() <= 2.0 ** -6 * pair + 1e-30).all()
        assert (g != w).double().mean() < 1e-2


@pytest.mark.parametrize("heads,d,s,fused", [(12, 128, 333, False), (2, 128, 5, True), (5, 64, 130, False),
                                             (40, 128, 65, False), (64, 128, 3, False), (1, 64, 1, False)])
def test_wan_heads_equal_the_operations(gpu, monkeypatch, heads, d, s, fused):
    from svoo_amd.processor import WanAttn_SAPAttn_Processor

    say("wan heads", heads, d, s, fused)
    torch.manual_seed(heads * s)
    layer = Layer(heads, d, heads * d, gpu, fused=fused)
    x = torch.randn(1, s, heads * d, device=gpu, dtype=torch.bfloat16)
    proc = _processor(WanAttn_SAPAttn_Processor)
    cos, sin = _tables(s, d, gpu)
    kw = dict(rotary_emb=(cos[None, :, None], sin[None, :, None]))
    want, n0 = _heads(proc, layer, x, True, monkeypatch, **kw)
    got, n1 = _heads(proc, layer, x, False, monkeypatch, **kw)
    assert (n0, n1) == (0, 1)
    _close(got[:2], want[:2])
    assert torch.equal(got[2], want[2])
    # without the norm in the pass (another norm module) every bit is the operations'
    layer.norm_q, layer.norm_k = torch.nn.Identity(), torch.nn.Identity()
    for kw2 in (kw, {}):
        want, _ = _heads(proc, layer, x, True, monkeypatch, **kw2)
        got, n1 = _heads(proc, layer, x, False, monkeypatch, **kw2)
        assert n1 == 1 and all(torch.equal(g, w) for g, w in zip(got, want))


@pytest.mark.parametrize("double", [False, True])
@pytest.mark.parametrize("heads,d,s,text", [(24, 128, 200, 33), (3, 64, 7, 1)])
def test_hunyuan_heads_equal_the_operations(gpu, monkeypatch, heads, d, s, text, double):
    from svoo_amd.processor import Hunyuan_SAPAttn_Processor

    say("hunyuan heads", heads, d, s, text, double)
    torch.manual_seed(s + text)
    layer = Layer(heads, d, d, gpu, double=double)
    x = torch.randn(1, s, heads * d, device=gpu, dtype=torch.bfloat16)
    txt = torch.randn(1, text, heads * d, device=gpu, dtype=torch.bfloat16)
    proc = _processor(Hunyuan_SAPAttn_Processor)
    for kw in (dict(encoder_hidden_states=txt, image_rotary_emb=_tables(s, d, gpu)),
               dict(encoder_hidden_states=txt), dict(image_rotary_emb=_tables(s, d, gpu))):
        want, n0 = _heads(proc, layer, x, True, monkeypatch, **kw)
        got, n1 = _heads(proc, layer, x, False, monkeypatch, **kw)
        assert n0 == 0 and n1 == (2 if double and "encoder_hidden_states" in kw else 1)
        _close(got[:2], want[:2])
        assert torch.equal(got[2], want[2])


@pytest.mark.parametrize("q_norm,k_norm", [(True, False), (False, True), (False, False)])
def test_hunyuan_text_norms_one_by_one(gpu, monkeypatch, q_norm, k_norm):
    """A double-stream block with a norm for the text's queries only, its keys only or neither: each is normed where it
    has a norm, whichever path runs."""
    from svoo_amd.processor import Hunyuan_SAPAttn_Processor

    say("hunyuan text norms", q_norm, k_norm)
    torch.manual_seed(5)
    heads, d, s, text = 3, 128, 40, 9
    layer = Layer(heads, d, d, gpu, double=True)
    if not q_norm:
        layer.norm_added_q = None
    if not k_norm:
        layer.norm_added_k = None
    x = torch.randn(1, s, heads * d, device=gpu, dtype=torch.bfloat16) * 3
    txt = torch.randn(1, text, heads * d, device=gpu, dtype=torch.bfloat16) * 3
    kw = dict(encoder_hidden_states=txt, image_rotary_emb=_tables(s, d, gpu))
    proc = _processor(Hunyuan_SAPAttn_Processor)
    want, _ = _heads(proc, layer, x, True, monkeypatch, **kw)
    got, _ = _heads(proc, layer, x, False, monkeypatch, **kw)
    _close(got[:2], want[:2])
    assert torch.equal(got[2], want[2])


def test_the_operations_run_where_the_pass_cannot(gpu, monkeypatch):
    """Gradients, hooks, an overridden method, autocast, tables or rows of another type: the tensor operations run, and
    give what they gave."""
    from svoo_amd.processor import WanAttn_SAPAttn_Processor

    say("heads: fallbacks")
    heads, d, s = 2, 128, 40
    layer = Layer(heads, d, heads * d, gpu)
    x = torch.randn(1, s, heads * d, device=gpu, dtype=torch.bfloat16)
    proc = _processor(WanAttn_SAPAttn_Processor)
    cos, sin = (t[None, :, None] for t in _tables(s, d, gpu))
    rope = dict(rotary_emb=(cos, sin))
    assert _heads(proc, layer, x, False, monkeypatch, **rope)[1] == 1
    # gradients: the weights' reach the result
    for weight in (layer.norm_q.weight, layer.to_q.weight):
        layer.requires_grad_(False)
        weight.requires_grad_(True)
        _, n = _heads(proc, layer, x, False, monkeypatch, **rope)
        assert n == 0 and proc.got[0].requires_grad
    with torch.no_grad():
        assert _heads(proc, layer, x, False, monkeypatch, **rope)[1] == 1
    layer.requires_grad_(False)
    # a hook of the norm runs
    seen = []
    hook = layer.norm_k.register_forward_hook(lambda m, i, o: seen.append(1))
    _heads(proc, layer, x, False, monkeypatch, **rope)
    assert seen == [1]
    hook.remove()
    for kw, run in ((dict(rotary_emb=(cos.double(), sin.double())), x), (rope, x.expand(2, -1, -1).contiguous())):
        want, n0 = _heads(proc, layer, run, True, monkeypatch, **kw)
        got, n1 = _heads(proc, layer, run, False, monkeypatch, **kw)
        assert n0 == n1 == 0 and all(torch.equal(a, b) for a, b in zip(got, want))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert _heads(proc, layer, x, False, monkeypatch, **rope)[1] == 0
    type(proc).get_qk_norm = lambda self, attn, q, k: (q, k)
    assert _heads(proc, layer, x, False, monkeypatch, **rope)[1] == 0


@pytest.mark.parametrize("norm_width", [256, 128])
def test_heads_of_non_finite_rows(gpu, monkeypatch, norm_width):
    """Rows with +inf, -inf, NaN and the type's largest values: NaN where the operations give NaN, the same values
    elsewhere (norm over the row, whose sum overflows, and per head)."""
    from svoo_amd.processor import Hunyuan_SAPAttn_Processor, WanAttn_SAPAttn_Processor

    say("heads: non-finite rows", norm_width)
    torch.manual_seed(2)
    wan = norm_width == 256
    layer = Layer(2, 128, norm_width, gpu)
    for n in ("to_q", "to_k", "to_v"):
        setattr(layer, n, torch.nn.Identity())  # the rows themselves
    x = torch.randn(1, 9, 256, device=gpu, dtype=torch.bfloat16)
    x[0, 1, 3], x[0, 2, 200], x[0, 3, 7], x[0, 4, 130], x[0, 5] = np.inf, -np.inf, np.nan, 3.0e38, 0.0
    x[0, 6, :128] = np.nan
    cos, sin = _tables(9, 128, gpu)
    kw = dict(rotary_emb=(cos[None, :, None], sin[None, :, None])) if wan else dict(image_rotary_emb=(cos, sin))
    proc = _processor(WanAttn_SAPAttn_Processor if wan else Hunyuan_SAPAttn_Processor)
    for norms in (True, False):
        if not norms:
            layer.norm_q = layer.norm_k = None
        want, _ = _heads(proc, layer, x, True, monkeypatch, **kw)
        got, n = _heads(proc, layer, x, False, monkeypatch, **kw)
        assert n == 1
        for g, w in zip(got, want):
            assert torch.equal(g.isnan(), w.isnan()) and torch.equal(g.isinf(), w.isinf())
        clean = lambda ts: [t.nan_to_num(0.0, 1.0, -1.0) for t in ts]  # noqa: E731
        g, w = clean(got), clean(want)
        assert torch.equal(g[2], w[2])
        if norms:
            for a, b in zip(g[:2], w[:2]):  # one bf16 step of either of the pair, as in _close
                pair = b.double().unflatten(-1, (-1, 2)).abs().sum(-1, keepdim=True).expand(-1, -1, -1, -1, 2).flatten(-2)
                assert ((a.double() - b.double()).abs() <= 2.0 ** -6 * pair + 1e-30).all()
        else:
            assert torch.equal(g[0], w[0]) and torch.equal(g[1], w[1])


def test_rows_of_another_device_keep_the_operations(gpu, monkeypatch):
    """Rows that are not on the current device: the tensor operations run, which go to their own."""
    from svoo_amd import heads
    from svoo_amd.processor import WanAttn_SAPAttn_Processor

    say("heads: another device")
    layer = Layer(2, 128, 256, gpu)
    x = torch.randn(1, 40, 256, device=gpu, dtype=torch.bfloat16)
    proc = _processor(WanAttn_SAPAttn_Processor)
    assert heads.rows_ok(x, 2) and _heads(proc, layer, x, False, monkeypatch)[1] == 1
    monkeypatch.setattr(torch.cuda, "current_device", lambda: x.device.index + 1)
    assert not heads.rows_ok(x, 2) and _heads(proc, layer, x, False, monkeypatch)[1] == 0
