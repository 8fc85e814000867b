"""Prefill row ops (fl_prefill_attention, fl_rope_store, fl_swiglu) against plain torch."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

from flashloop_amd import _lib, kernels  # noqa: E402
from flashloop_amd.model import apply_rope  # noqa: E402

DEV = "cuda"


def _r(gen, *shape):
    return torch.randn(*shape, generator=gen, device=DEV).to(torch.bfloat16)


@pytest.mark.parametrize("h,n,t", [(1, 1, 1), (2, 5, 5), (3, 64, 64), (2, 65, 65), (1, 129, 129), (2, 1000, 1000),  # dense
                                   (2, 1, 70), (3, 128, 130), (2, 200, 1500), (16, 820, 4100)])  # active rows
def test_prefill_attention(h, n, t):
    """Query blocks, key tiles and key ranges that end early; with positions the rows of a
    token-sparse loop, in order and shuffled.  Bound: every probability is rounded to bf16
    (2^-9 relative) and so is the sum that divides (the same rounded values), the output
    once more; the fp32 sums add far less."""
    print(f"case: prefill attention h={h} n={n} t={t}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(80)
    q = _r(g, n, h, 128).transpose(0, 1)  # the projections' row-major layout
    k, v = _r(g, h, t, 128), _r(g, h, t, 128)
    pos = None if n == t else torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    if pos is not None:
        pos[-1] = t - 1
    for p in ([pos] if pos is None else [pos, pos.flip(0).contiguous()]):
        at = torch.arange(n, device=DEV) if p is None else p.long()
        s = torch.bmm(q.double(), k.double().transpose(1, 2).contiguous()) * 128 ** -0.5
        w = s.masked_fill(torch.arange(t, device=DEV)[None, None] > at[None, :, None], -torch.inf).softmax(-1)
        want = torch.bmm(w, v.double()).transpose(0, 1).reshape(n, h * 128)
        size = torch.bmm(w, v.double().abs()).transpose(0, 1).reshape(n, h * 128)
        got = kernels.prefill_attention(q, k, v, 128 ** -0.5, p)
        err = (got.double() - want).abs() - (2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6)
        assert bool((err <= 0).all()), f"{err.max().item():.3e} beyond the bound"


def _want(q, k, v, at):
    """Attention of queries [H, n, 128] at positions ``at`` in float64, and the same of |v|."""
    s = torch.bmm(q.double(), k.double().transpose(1, 2).contiguous()) * 128 ** -0.5
    w = s.masked_fill(torch.arange(k.shape[1], device=DEV)[None, None] > at[None, :, None], -torch.inf).softmax(-1)
    rows = lambda x: torch.bmm(w, x).transpose(0, 1).reshape(q.shape[1], -1)
    return rows(v.double()), rows(v.double().abs())


def _within(got, want, size, what):
    """The bound of test_prefill_attention."""
    err = (got.double() - want).abs() - (2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6)
    assert bool((err <= 0).all()), f"{what}: {err.max().item():.3e} beyond the bound"


@pytest.mark.parametrize("n,t", [(150, 150), (40, 1000)])
def test_prefill_attention_of_large_scores(n, t):
    """Scores whose base-2 image is past the last fraction of an fp32 value, of both signs: equal
    ones, and ones that differ from key to key."""
    g = torch.Generator(device=DEV).manual_seed(84)
    v = _r(g, 2, t, 128)
    pos = None if n == t else torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    at = torch.arange(n, device=DEV) if pos is None else pos.long()
    for size in (3e2, 3e3, 3e4, 1e7, 1e10, 1e20, 1e31, 1e34):
        for sign in (1.0, -1.0):
            for spread in (0.0, 0.3):
                print(f"case: prefill attention scores n={n} t={t} {sign * size:.0e} {spread}", flush=True)
                a = (size / 128 ** 0.5) ** 0.5
                q = torch.full((2, n, 128), a, device=DEV).bfloat16()
                k = (sign * a * (1.0 + spread * torch.rand(2, t, 1, generator=g, device=DEV))).expand(2, t, 128).bfloat16()
                _within(kernels.prefill_attention(q, k, v, 128 ** -0.5, pos), *_want(q, k, v, at), f"{sign * size:.0e}")


@pytest.mark.parametrize("n,t", [(70, 70), (40, 1000)])
def test_prefill_attention_of_strided_rows(n, t):
    """K and V in any head and row stride: token-major rows, and rows 136 apart."""
    print(f"case: prefill attention strides n={n} t={t}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(85)
    pos = None if n == t else torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    at = torch.arange(n, device=DEV) if pos is None else pos.long()
    q, k, v = _r(g, 3, n, 136)[..., :128], _r(g, t, 3, 128).transpose(0, 1), _r(g, 3, t, 136)[..., :128]
    _within(kernels.prefill_attention(q, k, v, 128 ** -0.5, pos), *_want(q, k, v, at), "strides")


@pytest.mark.parametrize("n,t", [(200, 200), (40, 1000)])
def test_prefill_attention_of_non_finite_rows(n, t):
    """A NaN in a K row reaches the queries that see it and no other; scores of -inf weigh nothing;
    a query whose scores are all -inf, or NaN, gives NaN alone."""
    print(f"case: prefill attention non-finite n={n} t={t}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(86)
    pos = None if n == t else torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    at = torch.arange(n, device=DEV) if pos is None else pos.long()
    q, k, v = _r(g, 2, n, 128).abs(), _r(g, 2, t, 128), _r(g, 2, t, 128)
    scale, hole = 128 ** -0.5, t // 2 + 1
    bad = k.clone()
    bad[0, hole, 5] = torch.nan
    got = kernels.prefill_attention(q, bad, v, scale, pos).view(n, 2, 128)
    sees = at >= hole
    assert sees.any() and not sees.all()
    assert got[sees, 0].isnan().all() and not got[~sees].isnan().any() and not got[:, 1].isnan().any()
    want, size = (x.view(n, 2, 128) for x in _want(q, k, v, at))
    _within(got[~sees], want[~sees], size[~sees], "before a NaN")
    _within(got[:, 1], want[:, 1], size[:, 1], "another head")
    low = k.clone()
    low[:, 1::3] = -torch.inf
    _within(kernels.prefill_attention(q, low, v, scale, pos), *_want(q, low, v, at), "-inf")
    odd = q.clone()
    odd[0, 3], odd[1, n - 1, 0] = -torch.inf, torch.nan
    got = kernels.prefill_attention(odd, k.abs(), v, scale, pos).view(n, 2, 128)
    want, size = (x.view(n, 2, 128) for x in _want(odd, k.abs(), v, at))
    assert got[3, 0].isnan().all() and got[n - 1, 1].isnan().all() and int(got.isnan().sum()) == 2 * 128
    ok = ~got.isnan()
    _within(got[ok], want[ok], size[ok], "other queries")


@pytest.mark.parametrize("h,n,t", [(2, 8200, 8200), (1, 3300, 33000)])
def test_prefill_attention_of_long_prompts(h, n, t):
    """Many query blocks and key tiles; 64 of the queries against float64."""
    print(f"case: prefill attention long h={h} n={n} t={t}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(87)
    q, k, v = _r(g, n, h, 128).transpose(0, 1), _r(g, h, t, 128), _r(g, h, t, 128)
    pos = None if n == t else torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    at = torch.arange(n, device=DEV) if pos is None else pos.long()
    some = torch.cat((torch.randperm(n, generator=g, device=DEV)[:62], torch.tensor([0, n - 1], device=DEV)))
    got = kernels.prefill_attention(q, k, v, 128 ** -0.5, pos)
    _within(got[some], *_want(q[:, some], k, v, at[some]), "long")


@pytest.mark.parametrize("ranges", [0, 1, 2, 5])
def test_prefill_attention_with_less_workspace(ranges):
    """A workspace of fewer key ranges than asked for (or none) divides the keys less."""
    print(f"case: prefill attention ranges={ranges}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(81)
    h, n, t = 2, 150, 4000
    q, k, v = _r(g, h, n, 128), _r(g, h, t, 128), _r(g, h, t, 128)
    pos = torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    lib = _lib.load()
    one = n * h * 130 * 4
    assert lib.fl_prefill_attention_workspace(h, n, t) >= 6 * one
    room = torch.full((ranges * one + 64,), 7, dtype=torch.uint8, device=DEV)
    ws, guard = room, room[ranges * one:]
    out = torch.empty(n, h * 128, dtype=torch.bfloat16, device=DEV)
    _lib.check(lib.fl_prefill_attention(
        q.data_ptr(), q.stride(0), q.stride(1), k.data_ptr(), k.stride(0), k.stride(1), v.data_ptr(), v.stride(0),
        v.stride(1), out.data_ptr(), 128, h * 128, h, n, t, pos.data_ptr(), 128 ** -0.5, ws.data_ptr(), ranges * one,
        torch.cuda.current_stream().cuda_stream), "fl_prefill_attention")
    want = kernels.prefill_attention(q, k, v, 128 ** -0.5, pos).double()
    # a range's probabilities are rounded to bf16 against its own maximum (another power of
    # two times another fraction), so each side has test_prefill_attention's bound
    s = torch.bmm(q.double(), k.double().transpose(1, 2).contiguous()) * 128 ** -0.5
    w = s.masked_fill(torch.arange(t, device=DEV)[None, None] > pos.long()[None, :, None], -torch.inf).softmax(-1)
    size = torch.bmm(w, v.double().abs()).transpose(0, 1).reshape(n, h * 128)
    assert bool(((out.double() - want).abs() <= 2 * (2.0 ** -8 * size + 2.0 ** -8 * want.abs() + 1e-6)).all())
    assert bool((guard == 7).all())


@pytest.mark.parametrize("n,t", [(1, 1), (33, 33), (70, 400)])
def test_rope_store_equals_the_modules(n, t):
    print(f"case: rope store n={n} t={t}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(82)
    h = 3
    rows = [_r(g, n, h * 128) for _ in range(3)]
    ang = torch.rand(t, 64, generator=g, device=DEV) * 6.28
    cos, sin = (torch.cat((f, f), dim=-1).bfloat16() for f in (ang.cos(), ang.sin()))
    pos = None if n == t else torch.randperm(t, generator=g, device=DEV)[:n].sort().values.int()
    at = torch.arange(t, device=DEV) if pos is None else pos.long()
    want = [x.view(n, h, 128).transpose(0, 1) for x in rows]
    wq, wk = apply_rope(want[0][None], want[1][None], cos[at][None], sin[at][None])
    base = _r(g, 2, h, t, 128)
    kd, vd = base.clone().unbind(0)
    q = rows[0].clone()
    kernels.rope_store(q, rows[1], rows[2], (cos, sin), kd, vd, pos)
    assert torch.equal(q.view(n, h, 128).transpose(0, 1), wq[0])
    assert torch.equal(kd, base[0].index_copy(1, at, wk[0]))
    assert torch.equal(vd, base[1].index_copy(1, at, want[2]))


@pytest.mark.parametrize("n,d", [(1, 8), (3, 40), (257, 5632)])
def test_swiglu_rows(n, d):
    print(f"case: swiglu n={n} d={d}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(83)
    gate, up = _r(g, n, d) * 4, _r(g, n, d)
    want = F.silu(gate.double()) * up.double()
    got = kernels.swiglu(gate, up).double()
    # two bf16 roundings
    assert bool(((got - want).abs() <= 2.0 ** -7 * want.abs() + 1e-30).all())
