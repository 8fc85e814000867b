"""Set-up of a packed cache on the device (fl_count_active_rows, fl_cache_prepare) and the
rollover passes against the torch expressions they stand for."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from flashloop_amd import CrossLoopKVLayer, packed_prefix_tokens  # noqa: E402
from flashloop_amd.cache import append_layer_rows  # noqa: E402

DEV = "cuda"


def _kv(gen, b, h, t):
    return [torch.randn(b, h, t, 128, generator=gen, device=DEV).to(torch.bfloat16) for _ in range(4)]


@pytest.mark.parametrize("b,h,t,masks,room", [(1, 1, 1, "none", 0), (1, 2, 130, "both", 0), (3, 2, 777, "both", 300),
                                              (2, 1, 9000, "loop4", 64), (70, 1, 200, "both", 128), (70, 1, 150, "none", 0)])
def test_prefill_state_equals_torch(b, h, t, masks, room):
    """Lengths, rank maps, tails, activity and the zeros of the unused capacity, over ragged
    lengths, masks (both, one, none), scan steps of 8192 tokens and launches of 64 sequences."""
    print(f"case: cache build b={b} h={h} t={t} masks={masks} room={room}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(90)
    ks, vs = _kv(g, b, h, t), _kv(g, b, h, t)
    lengths = [t] + torch.randint(1, t + 1, (b - 1,), generator=torch.Generator().manual_seed(91)).tolist()
    every = torch.ones(b, t, dtype=torch.bool, device=DEV)
    m3 = torch.rand(b, t, generator=g, device=DEV) < 0.4 if masks == "both" else every
    m4 = m3 & (torch.rand(b, t, generator=g, device=DEV) < 0.5) if masks != "none" else every
    given = dict(mask_loop3=m3 if masks == "both" else None, mask_loop4=m4 if masks != "none" else None)
    junk = torch.full((64 << 20,), 0xA5, dtype=torch.uint8, device=DEV)  # freed memory is not zero
    del junk
    layer = CrossLoopKVLayer.from_prefill(ks, vs, lengths=lengths, token_capacity=t + room, **given)
    tp = [packed_prefix_tokens(n) for n in lengths]
    assert layer.packed_tokens.tolist() == tp == layer.packed_host
    assert layer.tail_tokens.tolist() == [n - p for n, p in zip(lengths, tp)] == layer.tail_host
    prefix = torch.arange(t, device=DEV)[None] < torch.tensor(tp, device=DEV)[:, None]
    counts = []
    for s, m in enumerate((m3, m4)):
        act = m & prefix
        want = torch.full_like(layer.rank[s], -1)
        n = min(t, want.shape[1])
        want[:, :n] = torch.where(act, act.int().cumsum(1) - 1, -1)[:, :n].int()
        assert torch.equal(layer.rank[s], want), f"rank map {s}"
        counts.append(act.sum(1).tolist())
        assert layer.late_rows[s].tolist() == counts[s] == layer.late_rows_host[s]
    top = max(tp)
    for i, (p, n) in enumerate(zip(tp, lengths)):
        rows = slice(i * h, (i + 1) * h)
        for r in range(4):
            for tail, src in ((layer.tail_key[r], ks[r]), (layer.tail_value[r], vs[r])):
                assert torch.equal(tail[rows, : n - p], src[i, :, p:n])
                assert not bool(tail[rows, n - p:].any())
        for s, m in enumerate((m3, m4)):
            assert torch.equal(layer.tail_active[s][i, : n - p].bool(), m[i, p:n])
            assert not bool(layer.tail_active[s][i, n - p:].any())
        for s in range(4):
            # the groups past a short sequence's prefix are encoded from its padding rows
            used = top if s < 2 else counts[s - 2][i]
            for x, u in ((layer.codes[s], used), (layer.value_meta[s], used), (layer.value_meta_half[s], used),
                         (layer.key_meta[s], top // 64), (layer.key_meta_half[s], top // 64)):
                assert not bool(x[rows, u:].any()), f"stream {s}: unused capacity is not zero"
            rec = layer.value_meta_token[rows][:, :, :, s]
            stored = torch.arange(rec.shape[1], device=DEV) < top
            if s >= 2:
                stored = stored & (layer.rank[s - 2][i] >= 0)
            assert not bool(rec[:, ~stored].any()), f"stream {s}: records of rows not stored"
    if masks == "both":
        again = CrossLoopKVLayer.from_prefill(ks, vs, lengths=lengths, token_capacity=t + room, **given,
                                              late_counts=CrossLoopKVLayer.count_late_rows(m3, m4, lengths))
        for name, x in layer.state_dict()[0].items():
            assert torch.equal(x, again.state_dict()[0][name]), name
        if bool(m4[0, :-1].any()):
            with pytest.raises(ValueError, match="nested"):
                CrossLoopKVLayer.from_prefill(ks, vs, lengths=lengths, mask_loop3=m4, mask_loop4=every)


def test_rollover_of_a_ragged_batch_equals_torch():
    """Of five sequences two roll: their rank rows continue the compact numbering, their tails
    and activity move down, and the others do not change."""
    print("case: ragged rollover", flush=True)
    g = torch.Generator(device=DEV).manual_seed(92)
    b, h, t = 5, 2, 400
    lengths = [383, 400, 255, 130, 70]  # tails of 127, 80, 127, 66 and 70 rows
    ks, vs = _kv(g, b, h, t), _kv(g, b, h, t)
    m3 = torch.rand(b, t, generator=g, device=DEV) < 0.5
    m4 = m3 & (torch.rand(b, t, generator=g, device=DEV) < 0.5)
    layer = CrossLoopKVLayer.from_prefill(ks, vs, lengths=lengths, mask_loop3=m3, mask_loop4=m4, token_capacity=512)
    new = [[torch.randn(b, h, 1, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(4)] for _ in range(2)]
    layer.append_rows(*new)
    before = {k: x.clone() for k, x in layer.state_dict()[0].items()}
    layer.commit_append()
    after = layer.state_dict()[0]
    assert layer.packed_host == [320, 320, 192, 64, 0] == after["packed_tokens"].tolist()
    assert layer.tail_host == [64, 81, 64, 67, 71] == after["tail_tokens"].tolist()
    for s in range(2):
        for i in range(b):
            want = before[f"rank.{s}"][i].clone()
            count = int(before["late_rows"][s, i])
            act = before[f"tail_active.{s}"][i].clone()
            if i in (0, 2):
                p = layer.packed_host[i] - 64
                on = act[:64].bool()
                want[p:p + 64] = torch.where(on, on.int().cumsum(0) - 1 + count, -1).int()
                count += int(on.sum())
                act = torch.cat((act[64:], torch.zeros_like(act[:64])))
            assert torch.equal(after[f"rank.{s}"][i], want) and int(after["late_rows"][s, i]) == count
            assert torch.equal(after[f"tail_active.{s}"][i], act)
    for r in range(4):
        for name in (f"tail_key.{r}", f"tail_value.{r}"):
            for i in range(b):
                rows = slice(i * h, (i + 1) * h)
                want = before[name][rows]
                n = layer.tail_host[i]
                assert torch.equal(after[name][rows, :n], want[:, 64:64 + n] if i in (0, 2) else want[:, :n]), name
    assert layer.late_rows_host == after["late_rows"].tolist()


@pytest.mark.parametrize("layers,b,h", [(1, 1, 1), (16, 3, 17), (18, 2, 2)])
def test_append_of_many_layers_equals_torch(layers, b, h):
    """One launch per 16 layers, a layer of another geometry in a launch of its own, more chunks
    than threads (17 heads): rows and flags at each sequence's tail, lengths one up."""
    print(f"case: append layers={layers} b={b} h={h}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(95)
    kv = [_kv(g, b, h, 150) for _ in range(2)]
    lengths = [150, 70, 129][:b]
    ls = [CrossLoopKVLayer.from_prefill(*kv, lengths=lengths) for _ in range(layers)]
    ls.append(CrossLoopKVLayer.from_prefill(*([x[:1] for x in y] for y in kv)))
    rows = [[[torch.randn(x.batch, h, 1, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(4)] for x in ls] for _ in range(2)]
    want = [{k: v.clone() for k, v in x.state_dict()[0].items()} for x in ls]
    append_layer_rows(ls, *rows)
    for i, (layer, w) in enumerate(zip(ls, want)):
        for b_ in range(layer.batch):
            at = int(w["tail_tokens"][b_])
            for r in range(4):
                w[f"tail_key.{r}"][b_ * h:(b_ + 1) * h, at] = rows[0][i][r][b_, :, 0]
                w[f"tail_value.{r}"][b_ * h:(b_ + 1) * h, at] = rows[1][i][r][b_, :, 0]
            for s in range(2):
                w[f"tail_active.{s}"][b_, at] = 1
            w["tail_tokens"][b_] += 1
        got = layer.state_dict()[0]
        assert got.keys() == w.keys()  # (bytes: the tails' unused rows may hold anything)
        assert [k for k in w if not torch.equal(got[k].contiguous().view(torch.uint8), w[k].contiguous().view(torch.uint8))] == [], i


def test_late_rows_beyond_a_given_count_are_dropped():
    """Counts below the masks': the surplus rows of loops 3/4 are left out (rank -1), so the rows
    that a rollover adds never share a compact row with them; a count above them leaves rows free."""
    print("case: late counts that differ from the masks", flush=True)
    g = torch.Generator(device=DEV).manual_seed(96)
    b, h, t = 3, 2, 255  # tails of 127 rows
    ks, vs = _kv(g, b, h, t), _kv(g, b, h, t)
    m3 = torch.rand(b, t, generator=g, device=DEV) < 0.6
    m4 = m3 & (torch.rand(b, t, generator=g, device=DEV) < 0.6)
    true = CrossLoopKVLayer.count_late_rows(m3, m4)
    given = [[max(0, n - d) for n, d in zip(true[s], (20 + s, 0, -5))] for s in range(2)]
    layer = CrossLoopKVLayer.from_prefill(ks, vs, mask_loop3=m3, mask_loop4=m4, token_capacity=512, late_counts=given)
    for s, m in enumerate((m3, m4)):
        for i in range(b):
            on = m[i, :128]
            want = torch.where(on, on.int().cumsum(0) - 1, -1)
            want = torch.where(want < given[s][i], want, -1).int()
            assert torch.equal(layer.rank[s][i, :128], want), f"rank map {s} of sequence {i}"
    assert layer.late_rows.tolist() == given == layer.late_rows_host
    new = [[torch.randn(b, h, 1, 128, generator=g, device=DEV).to(torch.bfloat16) for _ in range(4)] for _ in range(2)]
    layer.append_rows(*new)
    layer.commit_append()
    assert layer.packed_host == [192] * b
    for s in range(2):
        for i in range(b):
            rows = layer.rank[s][i][layer.rank[s][i] >= 0].tolist()
            assert len(set(rows)) == len(rows) and max(rows) < int(layer.late_rows[s, i]), f"rank map {s} of sequence {i}"


@pytest.mark.parametrize("t", [1, 100])
def test_short_prompts_of_misaligned_rows(t):
    """Prompts without a packed group, from K/V that start two bytes into their storage."""
    print(f"case: misaligned short prompt t={t}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(97)
    shape = (2, 3, t, 128)
    off = [torch.randn(2 * 3 * t * 128 + 1, generator=g, device=DEV).bfloat16()[1:].view(shape) for _ in range(8)]
    assert all(x.data_ptr() % 16 == 2 for x in off)
    layer = CrossLoopKVLayer.from_prefill(off[:4], off[4:])
    for r in range(4):
        assert torch.equal(layer.tail_key[r].view(2, 3, -1, 128)[:, :, :t], off[r])
        assert torch.equal(layer.tail_value[r].view(2, 3, -1, 128)[:, :, :t], off[4 + r])


def test_capacity_past_a_launch_is_cleared():
    """64 sequences of 16 heads with room for 131,072 tokens (103 GB): the clears are more than a
    launch's 2^32 threads."""
    print("case: capacity past a launch", flush=True)
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 180 << 30:
        pytest.skip("needs 180 GB of free device memory")
    g = torch.Generator(device=DEV).manual_seed(95)
    b, h, t = 64, 16, 130
    ks = _kv(g, b, h, t)
    junk = [torch.full((n << 30,), 0xA5, dtype=torch.uint8, device=DEV) for n in [16] * 4 + [8] + [2] * 14]
    del junk  # (freed memory is not zero)
    layer = CrossLoopKVLayer.from_prefill(ks, ks, token_capacity=131072)
    assert layer.packed_tokens.tolist() == [64] * b and layer.tail_tokens.tolist() == [t - 64] * b
    for s in range(4):
        for x in (layer.codes[s][:, 64:], layer.value_meta[s][:, 64:], layer.value_meta_half[s][:, 64:], layer.key_meta[s][:, 1:],
                  layer.key_meta_half[s][:, 1:]):
            for row in x.reshape(x.shape[0], -1).split(64):  # (a copy of a sixteenth at a time)
                assert not bool(row.view(torch.int64).any())
    assert not bool(layer.value_meta_token[:, 64:].any())
    for r in layer.rank:
        assert torch.equal(r[:, :64], torch.arange(64, device=DEV, dtype=torch.int32).expand(b, 64)) and bool((r[:, 64:] == -1).all())
    for got, want in zip((*layer.tail_key, *layer.tail_value), (*ks, *ks)):
        assert torch.equal(got[:, : t - 64], want.view(b * h, t, 128)[:, 64:]) and not bool(got[:, t - 64:].any())
    del layer, got, r, x, row
    torch.cuda.empty_cache()
