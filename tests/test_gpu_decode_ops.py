"""Fused decode-step model ops (fl_gemv_bf16, fl_norm_chain, fl_gemv_bf16_chain) against the
torch modules they replace, and the fused engine step against the module step."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

from flashloop_amd import kernels  # noqa: E402
from flashloop_amd.engine import FlashLoopEngine  # noqa: E402
from flashloop_amd.model import OuroConfig, OuroForCausalLM, RMSNorm, apply_rope  # noqa: E402

DEV = "cuda"


def _w(n, k, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(n, k, generator=g, device=DEV) * 0.02).to(torch.bfloat16)


def _x(m, k, seed, dtype=torch.bfloat16):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(m, k, generator=g, device=DEV).to(dtype)


def _close_bf16(got, want, what, cancel=False):
    """Both sides round an fp32 dot product to bf16; summation order may move a value by
    one bf16 ulp (2^-8 relative), nothing more.  With ``cancel`` (RoPE: a sum of two
    rounded products) the ulp is that of the largest value of the row."""
    got, want = got.float(), want.float()
    tol = want.abs() * 2.0 ** -7 + 1e-6
    if cancel:
        tol = tol + want.abs().amax(dim=-1, keepdim=True) * 2.0 ** -7
    bad = ((got - want).abs() > tol).sum().item()
    assert bad == 0, f"{what}: {bad} values beyond one ulp; max diff {(got - want).abs().max().item()}"
    exact = (got == want).float().mean().item()
    assert exact > 0.9, f"{what}: only {exact:.3f} of the values equal the module's"


@pytest.mark.parametrize("m,n,k", [(1, 2048, 2048), (3, 2048, 5632), (8, 512, 2048), (1, 49152, 2048)])
def test_gemv_plain_and_f32(m, n, k):
    print(f"case: gemv m={m} n={n} k={k}", flush=True)
    x, w = _x(m, k, 1), _w(n, k, 2)
    want = F.linear(x, w)
    _close_bf16(kernels.gemv(x, [w]), want, "plain")
    got32 = kernels.gemv(x, [w], epilogue=kernels.EPI_F32)
    assert got32.dtype == torch.float32
    _close_bf16(got32, want.float(), "f32")
    assert torch.equal(got32, got32.bfloat16().float())  # the widened bf16 value


def test_gemv_f32_input_and_add():
    print("case: gemv f32 input + addend", flush=True)
    x32 = _x(2, 2048, 3, torch.float32)
    w = _w(2048, 2048, 4)
    add = _x(2, 2048, 5)
    want = F.linear(x32.to(torch.bfloat16), w) + add
    _close_bf16(kernels.gemv(x32, [w], epilogue=kernels.EPI_ADD, addend=add), want, "f32-in add")


def test_gemv_swiglu():
    print("case: gemv swiglu", flush=True)
    x = _x(2, 2048, 6)
    wg, wu = _w(5632, 2048, 7), _w(5632, 2048, 8)
    want = F.silu(F.linear(x, wg)) * F.linear(x, wu)
    _close_bf16(kernels.gemv(x, [wg, wu], epilogue=kernels.EPI_SWIGLU), want, "swiglu")


def test_gemv_rope_qkv():
    print("case: gemv rope qkv", flush=True)
    cfg = OuroConfig(num_hidden_layers=1, vocab_size=256)
    model = OuroForCausalLM.random_init(cfg, seed=3, device=DEV)
    a = model.model.layers[0].self_attn
    b, hd, heads = 3, 128, cfg.num_attention_heads
    x = _x(b, cfg.hidden_size, 9)
    pos = torch.tensor([[5], [4000], [123456]], device=DEV)
    cos, sin = model.model.rotary_emb(x[:, None], pos)
    q, k, v = kernels.gemv(x, [a.q_proj.weight, a.k_proj.weight, a.v_proj.weight], epilogue=kernels.EPI_ROPE,
                           rope=(cos.reshape(b, hd), sin.reshape(b, hd)))
    rq = a.q_proj(x[:, None]).view(b, 1, heads, hd).transpose(1, 2)
    rk = a.k_proj(x[:, None]).view(b, 1, heads, hd).transpose(1, 2)
    rv = a.v_proj(x[:, None]).view(b, 1, heads, hd).transpose(1, 2)
    rq, rk = apply_rope(rq, rk, cos, sin)
    _close_bf16(q.view(b, heads, 1, hd), rq, "q", cancel=True)
    _close_bf16(k.view(b, heads, 1, hd), rk, "k", cancel=True)
    _close_bf16(v.view(b, heads, 1, hd), rv, "v")


def test_norm_chain_matches_modules():
    print("case: norm chain", flush=True)
    d, eps = 2048, 1e-6
    mods = [RMSNorm(d, eps).to(DEV, torch.bfloat16) for _ in range(3)]
    with torch.no_grad():
        for i, mod in enumerate(mods):
            mod.weight.copy_(1.0 + 0.1 * _x(1, d, 20 + i, torch.float32)[0])
    r, x = _x(4, d, 10), _x(4, d, 11) * 3.0
    h, z = kernels.norm_chain(r, x=x, w_a=mods[0].weight, w_f=mods[1].weight, w_b=mods[2].weight, eps=eps)
    wh = mods[1](r + mods[0](x))
    wz = mods[2](wh)
    _close_bf16(h, wh, "h")
    _close_bf16(z, wz, "z")
    h2, z2 = kernels.norm_chain(r, w_b=mods[2].weight, eps=eps, want_h=False)
    assert h2 is None
    _close_bf16(z2, mods[2](r), "z only")


def test_fused_step_tracks_module_step():
    """The fused decode step and the torch-module step agree to bf16 rounding noise."""
    tiny = OuroConfig(vocab_size=1024, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                      num_attention_heads=2, num_key_value_heads=2)
    model = OuroForCausalLM.random_init(tiny, seed=21, device=DEV)
    g = torch.Generator().manual_seed(21)
    ids = torch.randint(0, tiny.vocab_size, (1, 230), generator=g).to(DEV)
    fused = FlashLoopEngine(model, use_graphs=False)
    mods = FlashLoopEngine(model, use_graphs=False)
    mods.fused_decode = False
    fused.prefill(ids[:, :200], decode_capacity=64)
    mods.prefill(ids[:, :200], decode_capacity=64)
    for i in range(200, 230):
        a = fused.decode(ids[:, i:i + 1]).logits
        b = mods.decode(ids[:, i:i + 1]).logits
        cos = F.cosine_similarity(a.double().flatten(), b.double().flatten(), dim=0).item()
        assert cos > 0.9999, f"step {i}: cos {cos}"
        assert (a - b).abs().max().item() < 2e-2 * max(1.0, b.abs().max().item()), f"step {i}"


@pytest.mark.parametrize("k", [2048, 4096])
@pytest.mark.parametrize("m", [1, 3, 8])
def test_gemv_chain_is_norm_chain_then_gemv(m, k):
    """fl_gemv_bf16_chain equals fl_norm_chain + fl_gemv_bf16 bit for bit (h and the
    output), for every epilogue and every optional part of the chain."""
    print(f"case: gemv chain m={m} k={k}", flush=True)
    eps, hd = 1e-6, 128
    wn = [(1.0 + 0.1 * _x(1, k, 40 + i, torch.float32)[0]).to(torch.bfloat16) for i in range(3)]
    r, x = _x(m, k, 30), _x(m, k, 31) * 3.0
    n = 512
    mats = [_w(n, k, 50 + i) for i in range(3)]
    pos = torch.arange(m, device=DEV) + 7
    inv = 1.0 / (10000.0 ** (torch.arange(0, hd, 2, device=DEV).float() / hd))
    ang = torch.cat([pos[:, None] * inv[None], pos[:, None] * inv[None]], dim=-1)
    rope = (ang.cos().to(torch.bfloat16), ang.sin().to(torch.bfloat16))
    addend = _x(m, n, 32)
    chains = [dict(x=x, w_a=wn[0], w_b=wn[2]), dict(x=x, w_a=wn[0], w_f=wn[1], w_b=wn[2]),
              dict(w_b=wn[2]), dict(x=x, w_a=wn[0], w_f=wn[1])]
    epis = [(kernels.EPI_PLAIN, mats[:1], {}), (kernels.EPI_F32, mats[:1], {}),
            (kernels.EPI_ADD, mats[:1], dict(addend=addend)), (kernels.EPI_SWIGLU, mats[:2], {}),
            (kernels.EPI_ROPE, mats, dict(rope=rope, head_dim=hd))]
    for ci, ch in enumerate(chains):
        h0, z0 = kernels.norm_chain(r, eps=eps, **ch)
        inp = z0 if ch.get("w_b") is not None else h0
        for epi, ws, extra in epis:
            want = kernels.gemv(inp, ws, epilogue=epi, **extra)
            h1, got = kernels.gemv_chain(r, ws, eps=eps, epilogue=epi, **ch, **extra)
            assert torch.equal(h1, h0), f"chain {ci} epilogue {epi}: h differs"
            for g_, w_ in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
                assert torch.equal(g_, w_), f"chain {ci} epilogue {epi}: output differs"
    _, got = kernels.gemv_chain(r, mats[:1], eps=eps, want_h=False, w_b=wn[2])
    _, z0 = kernels.norm_chain(r, eps=eps, w_b=wn[2], want_h=False)
    assert torch.equal(got, kernels.gemv(z0, mats[:1]))


def test_chained_step_equals_unchained_step():
    """The engine's decode step with the chains inside the GEMVs equals the step with
    separate chain launches bit for bit."""
    tiny = OuroConfig(vocab_size=1024, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                      num_attention_heads=2, num_key_value_heads=2)
    model = OuroForCausalLM.random_init(tiny, seed=22, device=DEV)
    g = torch.Generator().manual_seed(22)
    ids = torch.randint(0, tiny.vocab_size, (1, 150), generator=g).to(DEV)
    a_eng = FlashLoopEngine(model, use_graphs=False)
    b_eng = FlashLoopEngine(model, use_graphs=False)
    b_eng.fused_chain = False
    a_eng.prefill(ids[:, :130], decode_capacity=64)
    b_eng.prefill(ids[:, :130], decode_capacity=64)
    for i in range(130, 150):
        a = a_eng.decode(ids[:, i:i + 1]).logits
        b = b_eng.decode(ids[:, i:i + 1]).logits
        assert torch.equal(a, b), f"step {i}: max diff {(a - b).abs().max().item()}"


def _dots(x, w):
    """The Linear's output in float64 (rounded to bf16 once) and the bound of an fp32 sum of k
    products: k * 2^-24 of the sum of their sizes."""
    d = (x.double() @ w.double().t()).float().bfloat16().double()
    return d, (x.double().abs() @ w.double().abs().t()) * x.shape[-1] * 2.0 ** -24


def _near(got, want, slack, what, ulps=1.0):
    """Within the bound of the sums plus ``ulps`` bf16 roundings (2^-8 relative each)."""
    err = (got.double() - want).abs() - (slack + ulps * 2.0 ** -8 * want.abs() + 1e-30)
    assert bool((err <= 0).all()), f"{what}: {err.max().item():.3e} beyond the bound"


@pytest.mark.parametrize("n", [2060, 4108, 8200])
def test_gemv_chain_of_several_units(n):
    """Eight chained rows run on at most 256 workgroups: two, three and five units each, the last
    workgroups fewer (258, 514 and 1025 SwiGLU units); equal to the chain and the GEMV apart."""
    print(f"case: gemv chain units n={n}", flush=True)
    k = 520
    r, x, wn, mats = _x(8, k, 90), _x(8, k, 91), [_x(1, k, 92 + i)[0] for i in range(2)], [_w(n, k, 94 + i) for i in range(2)]
    h0, z0 = kernels.norm_chain(r, eps=1e-6, x=x, w_a=wn[0], w_b=wn[1])
    for epi, ws, extra in ((kernels.EPI_SWIGLU, mats, {}), (kernels.EPI_ADD, mats[:1], dict(addend=_x(8, n, 96)))):
        h1, got = kernels.gemv_chain(r, ws, eps=1e-6, epilogue=epi, x=x, w_a=wn[0], w_b=wn[1], **extra)
        assert torch.equal(h1, h0) and torch.equal(got, kernels.gemv(z0, ws, epilogue=epi, **extra))


@pytest.mark.parametrize("m,n,k", [(1, 4, 8), (1, 516, 200), (2, 12, 520), (5, 516, 2056), (8, 20, 2048), (8, 16388, 1024),
                                   (1, 16388, 2040), (3, 36, 4104), (8, 260, 6152), (1, 260, 8192), (4, 8, 8200)])
def test_gemv_at_tile_and_step_edges(m, n, k):
    """Rows, N and K that end inside a tile, a 512-wide step or an instantiation."""
    print(f"case: gemv edges m={m} n={n} k={k}", flush=True)
    x, x32, add = _x(m, k, 60), _x(m, k, 61, torch.float32), _x(m, n, 62)
    gate, up = _w(n, k, 63), _w(n, k, 64)
    d, s = _dots(x, gate)
    _near(kernels.gemv(x, [gate]), d, s, "plain")
    _near(kernels.gemv(x, [gate], epilogue=kernels.EPI_F32), d, s, "f32")
    df, sf = _dots(x32.bfloat16(), gate)
    got = kernels.gemv(x32, [gate], epilogue=kernels.EPI_ADD, addend=add)
    _near(got, df + add.double(), sf + 2.0 ** -8 * df.abs(), "add")
    # |silu'| < 1.1: an error of the gate carries over, scaled by the up value
    du, su = _dots(x, up)
    silu = F.silu(d)
    slack = 1.1 * (s + 2.0 ** -8 * d.abs()) * du.abs() + silu.abs() * (su + 2.0 ** -8 * du.abs())
    _near(kernels.gemv(x, [gate, up], epilogue=kernels.EPI_SWIGLU), silu * du, slack, "swiglu", ulps=3.0)


@pytest.mark.parametrize("m,heads,hd,k", [(1, 3, 24, 200), (8, 1, 8, 2048), (5, 3, 40, 4104), (8, 4, 128, 2056), (1, 2, 128, 8192)])
def test_gemv_rope_at_head_edges(m, heads, hd, k):
    """Rotary pairs that straddle heads inside a tile, and heads smaller than one."""
    print(f"case: gemv rope edges m={m} heads={heads} hd={hd} k={k}", flush=True)
    n = heads * hd
    x, ws = _x(m, k, 70), [_w(n, k, 71 + i) for i in range(3)]
    ang = torch.rand(m, hd // 2, device=DEV, generator=torch.Generator(device=DEV).manual_seed(74)) * 6.28
    cos, sin = (torch.cat((f, f), dim=-1).bfloat16() for f in (ang.cos(), ang.sin()))
    q, key, v = kernels.gemv(x, ws, epilogue=kernels.EPI_ROPE, rope=(cos, sin), head_dim=hd)
    _near(v, *_dots(x, ws[2]), "v")
    for got, w in ((q, ws[0]), (key, ws[1])):
        d, s = (t.view(m, heads, hd) for t in _dots(x, w))
        rot = torch.cat((-d[..., hd // 2:], d[..., :hd // 2]), dim=-1)
        want = d * cos.double()[:, None] + rot * sin.double()[:, None]
        # the dots' own roundings and each product's (2^-8 of its size, twice)
        slack = s + s.roll(hd // 2, dims=-1) + 2.0 ** -7 * (d.abs() + rot.abs())
        _near(got.view(m, heads, hd), want, slack, "rope")


@pytest.mark.parametrize("b,d,hd,freq", [(1, 8, 2, torch.float32), (3, 2056, 126, torch.bfloat16), (8, 4096, 1024, torch.float32)])
def test_decode_inputs(b, d, hd, freq):
    """Embedding rows exactly; cos and sin of the fp32 angle: 2 ulp of an fp32 function (2^-22 at
    most), then half a bf16 ulp.  A token outside the table gives a row of NaN."""
    print(f"case: decode inputs b={b} d={d} hd={hd}", flush=True)
    table = _x(50, d, 110)
    tok = torch.tensor([[0], [49], [7], [50], [-1], [3], [1 << 40], [49]][:b], device=DEV)
    pos = torch.tensor([[8191], [0], [1], [70000], [12345], [2], [64], [1 << 20]][:b], device=DEV)
    inv = (1.0 / 10000.0 ** (torch.arange(0, hd, 2, device=DEV).float() / hd)).to(freq)
    h, cos, sin = kernels.decode_inputs(tok, pos, table, inv)
    ok = ((tok >= 0) & (tok < 50)).flatten()
    assert torch.equal(h[ok], table[tok[ok]]) and h[~ok].isnan().all()
    angle = (pos.float() * inv.float()[None]).double().cpu()
    for got, want in ((cos, angle.cos()), (sin, angle.sin())):
        want = torch.cat([want, want], -1)
        assert ((got[:, 0].double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -21).all()


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 8])
def test_gemv_of_long_rows(m):
    """K past the matrix-core form: each number of rows on the instantiation that holds it."""
    print(f"case: gemv long rows m={m}", flush=True)
    n, k = 12, 10248
    x, x32, add, w = _x(m, k, 120), _x(m, k, 121, torch.float32), _x(m, n, 122), _w(n, k, 123)
    _near(kernels.gemv(x, [w]), *_dots(x, w), "plain")
    d, s = _dots(x32.bfloat16(), w)
    _near(kernels.gemv(x32, [w], epilogue=kernels.EPI_ADD, addend=add), d + add.double(), s + 2.0 ** -8 * d.abs(), "add")


@pytest.mark.parametrize("m,n,k", [(1, 4, 4104), (2, 12, 6144), (2, 516, 6152), (1, 20, 8192),
                                   (1, 16388, 1024), (2, 16388, 1016), (8, 516, 1024), (2, 16388, 2040), (3, 16388, 1032),
                                   (1, 516, 3072), (5, 516, 2056), (1, 2052, 4096), (1, 2044, 4096), (8, 4104, 4096)])
def test_gemv_forms(m, n, k):
    """Both sides of each line between the forms: one and two rows past K 4096, the steps of K, the
    head-sized N and the f32 rows of two tiles a unit."""
    test_gemv_at_tile_and_step_edges(m, n, k)


@pytest.mark.parametrize("m", [1, 2, 8])
@pytest.mark.parametrize("k", [1016, 2048, 3072, 4096])
def test_gemv_chain_of_a_head(m, k):
    """A head-sized matrix, where a chained call and the GEMV apart take different forms: equal."""
    print(f"case: gemv chain head m={m} k={k}", flush=True)
    n = 16388
    r, x, wn, w = _x(m, k, 130), _x(m, k, 131), [_x(1, k, 132 + i)[0] for i in range(2)], _w(n, k, 134)
    h0, z0 = kernels.norm_chain(r, eps=1e-6, x=x, w_a=wn[0], w_b=wn[1])
    h1, got = kernels.gemv_chain(r, [w], eps=1e-6, epilogue=kernels.EPI_F32, x=x, w_a=wn[0], w_b=wn[1])
    assert torch.equal(h1, h0) and torch.equal(got, kernels.gemv(z0, [w], epilogue=kernels.EPI_F32))
    _near(got, *_dots(z0, w), "head", ulps=2.0)  # both sides are rounded: half an ulp, 2^-8 at most, each
