"""Row movement and token selection at the sizes where their kernels change."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from flashloop_amd import _lib, kernels  # noqa: E402
from oracle import tokens as OT  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("outer,rows,width,n", [(1, 1, 2, 1), (3, 700, 6, 300), (16, 300, 128, 257), (2, 5000, 8, 4097),
                                                (1, 40, 5000, 40)])
def test_rows_move_and_flag(outer, rows, width, n):
    """Rows of 4 bytes to 10 KB (4- and 16-byte pieces), workgroups that cross rows, and the flag:
    written 0 over whatever the memory held, 1 where an index is out of range, whose row stays."""
    print(f"case: rows outer={outer} rows={rows} width={width} n={n}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(96)
    src = torch.randint(0, 1 << 15, (outer, rows, width), generator=g, device=DEV).to(torch.int16)
    pos = torch.randperm(rows, generator=g, device=DEV)[:n].int()
    got, err = kernels.gather_rows(src, pos, 1)
    assert torch.equal(got, src.index_select(1, pos.long())) and int(err) == 0
    new = torch.randint(0, 1 << 15, (outer, pos.numel(), width), generator=g, device=DEV).to(torch.int16)
    dst, err = kernels.scatter_rows_(src.clone(), pos, new, 1)
    assert torch.equal(dst, src.index_copy(1, pos.long(), new)) and int(err) == 0
    for bad in (-1, rows):
        wrong = pos.clone()
        wrong[-1] = bad
        dst, err = kernels.scatter_rows_(src.clone(), wrong, new, 1)
        assert torch.equal(dst, src.index_copy(1, pos[:-1].long(), new[:, :-1])) and int(err) == 1
        _, err = kernels.gather_rows(src, wrong, 1)
        assert int(err) == 1


@pytest.mark.parametrize("width,gap", [(2, 0), (6, 2), (128, 0), (200, 8), (4, 4)])
def test_row_calls_that_only_set_the_flag(width, gap):
    """fl_gather_rows and fl_scatter_rows through the C API, rows apart in 4- and 16-byte pieces:
    a flag of the caller's is set by an index out of range and otherwise left as it was; none may
    be given; no index moves nothing."""
    print(f"case: row calls width={width} gap={gap}", flush=True)
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    g = torch.Generator(device=DEV).manual_seed(98)
    outer, rows, n, pitch = 3, 500, 131, width + gap
    rand = lambda *shape: torch.randint(0, 1 << 15, shape, generator=g, device=DEV).to(torch.int16)
    full, new = rand(outer, rows, pitch), rand(outer, n, pitch)
    pos = torch.randperm(rows, generator=g, device=DEV)[:n].int()
    wrong = pos.clone()
    wrong[7], wrong[100] = rows, -1
    ok = torch.ones(n, dtype=torch.bool, device=DEV)
    ok[7] = ok[100] = False

    def gather(index, count, flag):
        dst = new.clone()
        _lib.check(lib.fl_gather_rows(full.data_ptr(), rows * pitch * 2, pitch * 2, rows, dst.data_ptr(), n * pitch * 2, pitch * 2,
                                      outer, width * 2, index.data_ptr(), count, None if flag is None else flag.data_ptr(), stream),
                   "fl_gather_rows")
        return dst

    def scatter(index, count, flag):
        dst = full.clone()
        _lib.check(lib.fl_scatter_rows(new.data_ptr(), n * pitch * 2, pitch * 2, dst.data_ptr(), rows * pitch * 2, pitch * 2, rows,
                                       outer, width * 2, index.data_ptr(), count, None if flag is None else flag.data_ptr(), stream),
                   "fl_scatter_rows")
        return dst

    for index, moved in ((pos, torch.ones_like(ok)), (wrong, ok)):
        at = index[moved].long()
        got = new.clone()
        got[:, moved, :width] = full[:, at, :width]
        put = full.clone()
        put[:, at, :width] = new[:, moved, :width]
        for held in (0, 5, None):
            flag = None if held is None else torch.full((1,), held, dtype=torch.int32, device=DEV)
            for call, want in ((gather, got), (scatter, put)):
                assert torch.equal(call(index, n, flag), want)
                if flag is not None:
                    assert int(flag) == (held if bool(moved.all()) else 1)
    flag = torch.full((1,), 5, dtype=torch.int32, device=DEV)
    assert torch.equal(gather(wrong, 0, flag), new) and torch.equal(scatter(wrong, 0, flag), full) and int(flag) == 5


def test_rows_past_a_launch():
    """More than 2^32 pieces of 4 bytes (17 GB): the rows of both launches, and the flag, which an
    index of the second one sets."""
    print("case: rows past a launch", flush=True)
    g = torch.Generator(device=DEV).manual_seed(94)
    width, rows = 2 * 1025, 1000
    n = 2 ** 32 // 1025 + 3000
    src = torch.randint(0, 1 << 15, (1, rows, width), generator=g, device=DEV).to(torch.int16)
    pos = torch.randint(0, rows, (n,), generator=g, device=DEV).int()
    got, err = kernels.gather_rows(src, pos, 1)
    assert int(err) == 0
    some = torch.cat((torch.arange(5, device=DEV), torch.arange(n - 6000, n, device=DEV)))
    assert torch.equal(got[0, some], src[0, pos[some].long()])
    back = torch.zeros_like(src)
    pos.fill_(-1)  # (no two alike: the last 1000 rows go to places of their own)
    pos[-rows:] = torch.randperm(rows, generator=g, device=DEV).int()
    pos[0] = rows
    _, err = kernels.scatter_rows_(back, pos, got, 1)
    assert int(err) == 1 and torch.equal(back[0, pos[-rows:].long()], got[0, -rows:])


def _scores(kind, b, t, gen):
    x = torch.randn(b, t, generator=gen, device=DEV)
    if kind == "tied":
        x = (x * 3).round() / 3
    elif kind == "zeros":
        x = torch.where(x > 0, 0.0, -0.0)
    return x


@pytest.mark.parametrize("kind", ["normal", "tied", "zeros"])
@pytest.mark.parametrize("b,t", [(1, 1), (3, 5), (2, 4096), (2, 4097), (1, 8193), (1, 16385), (1, 36864), (1, 36865)])
def test_token_selection_at_instantiation_edges(kind, b, t):
    """Every instantiation's smallest and largest row, ties, signed zeros, eligibility and the
    forced last token, against the oracle's selection."""
    print(f"case: token selection {kind} b={b} t={t}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(97)
    x = _scores(kind, b, t, gen)
    el = torch.rand(b, t, generator=gen, device=DEV) < 0.4
    el[:, -1] = True
    for fraction, eligible in ((0.25, None), (1.0, None), (0.1, el), (0.9, el)):
        mask, pos, counts, err = kernels.select_tokens(x, fraction, eligible=eligible)
        want = OT.select_active_mask(x.cpu().numpy(), fraction, eligible=None if eligible is None else eligible.cpu().numpy())
        assert np.array_equal(mask.cpu().numpy(), want) and int(err) == 0
        for i in range(b):
            on = np.nonzero(want[i])[0]
            assert int(counts[i]) == len(on)
            assert np.array_equal(pos[i].cpu().numpy(), np.concatenate([on, np.zeros(t - len(on), on.dtype)]))
    if b > 1:  # a row whose last token is not eligible is left empty; the others are selected
        el[1, -1] = False
        mask, pos, counts, err = kernels.select_tokens(x, 0.25, eligible=el)
        assert int(err) == 1 and int(counts[1]) == 0 and not bool(mask[1].any()) and not bool(pos[1].any())
        want = OT.select_active_mask(x[:1].cpu().numpy(), 0.25, eligible=el[:1].cpu().numpy())
        assert np.array_equal(mask[:1].cpu().numpy(), want)


@pytest.mark.parametrize("rows,dim", [(1, 8), (5, 2048), (3, 2056), (7, 100), (2, 16384)])
def test_hidden_score_widths(rows, dim):
    print(f"case: hidden score rows={rows} dim={dim}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(98)
    a, b = (torch.randn(rows, dim, generator=g, device=DEV).bfloat16() for _ in range(2))
    got = kernels.hidden_delta_score(a, b).double()
    want = (a.double() - b.double()).norm(dim=-1) / a.double().norm(dim=-1)
    # two fp32 sums of dim positive terms (halved by the root), a division and two roots
    assert bool(((got - want).abs() <= (dim + 8) * 2.0 ** -24 * want).all())


@pytest.mark.parametrize("dim", [1, 64, 248, 256, 264])
def test_hidden_score_at_the_wide_loads_line(dim):
    """Rows on both sides of 256 values, against the bound of test_hidden_score_widths."""
    print(f"case: hidden score line dim={dim}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(99)
    a, b = (torch.randn(9, dim, generator=g, device=DEV).bfloat16() for _ in range(2))
    got = kernels.hidden_delta_score(a, b).double()
    want = (a.double() - b.double()).norm(dim=-1) / a.double().norm(dim=-1)
    assert bool(((got - want).abs() <= (dim + 8) * 2.0 ** -24 * want).all())


@pytest.mark.parametrize("heads,tokens", [(16, 12000), (16, 20000), (8, 9000), (8, 12000)])
def test_sparse_merges_on_both_sides_of_the_wide_line(heads, tokens):
    """20, 33, 31 and 39 parts a row: each head alone (31 parts or more) gives the same loop-3 and
    loop-4 deltas and source sum.  Bound: fp32 sums over k selected keys of weights that add up to
    1, k * 2^-24 of the largest value each way, for the two sums of a delta."""
    print(f"case: sparse merges heads={heads} tokens={tokens}", flush=True)
    from flashloop_amd.cache import CrossLoopKVLayer
    g = torch.Generator(device=DEV).manual_seed(99)
    rand = lambda *shape: torch.randn(shape, generator=g, device=DEV).to(torch.bfloat16)
    ks, vs = [rand(1, heads, tokens, 128) for _ in range(4)], [rand(1, heads, tokens, 128) for _ in range(4)]
    q, k, v, v1 = (rand(1, heads, 1, 128) for _ in range(4))

    def deltas(rows, chosen):
        lc = CrossLoopKVLayer.from_prefill([x[:, rows] for x in ks], [x[:, rows] for x in vs])
        at = lambda x: x[:, rows].contiguous()
        if chosen is None:
            _, _, chosen = lc.dense_source_attention_select(1, query=q, current_key=k, current_value=v1, scaling=0.088,
                                                            fraction=0.1)
        else:
            idx, valid, mass, w, cnt = chosen
            chosen = (at(idx), at(valid), at(mass), at(w), cnt.view(1, -1)[:, rows].flatten().contiguous())
        idx, valid, mass, w, cnt = chosen
        common = dict(query=at(q), current_key=at(k), current_value=at(v), indices=idx, valid=valid, global_mass=mass,
                      scaling=0.088, counts=cnt)
        d3, so = lc.cached_mass_sparse_attention_delta_with_source(2, source_weights=w, source_current_value=at(v1), **common)
        d4 = lc.cached_mass_sparse_attention_delta(3, source_selected_output=so, **common)
        return chosen, (d3, so, d4)

    chosen, together = deltas(slice(0, heads), None)
    bound = 4 * int(chosen[4].max()) * 2.0 ** -24 * max(float(x.abs().max()) for x in vs)
    for h in range(0, heads, 5):
        _, alone = deltas(slice(h, h + 1), chosen)
        for a, b in zip(together, alone):
            assert float((a.view(heads, 128)[h] - b.view(128)).abs().max()) <= bound
