"""fl_decode_topk_long (a row over several workgroups) against fl_decode_topk (one workgroup
per row): the same keys, counts and non-finite counts bit for bit; the masses sum in
another order (at most k fp32 additions of positive terms: k * 2^-24 relative)."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from flashloop_amd import CrossLoopKVLayer, _lib, decode_attention_step, kernels  # noqa: E402
from flashloop_amd.synthetic import SCALING, loop_chain  # noqa: E402

DEV = "cuda"


def _rows(kind, rows, stride, gen):
    x = torch.randn(rows, stride, generator=gen, device=DEV)
    if kind == "peaked":
        x *= 40.0
    elif kind == "tied":
        x = (x * 4.0).round() / 4.0
    elif kind == "equal":
        x = torch.full_like(x, 0.25)
    elif kind == "mixed":  # NaN, infinities, only -inf and signed zeros, among ordinary rows
        x[0, stride // 3] = float("nan")
        x[1, 7] = float("inf")
        x[2] = float("-inf")
        x[3, ::2] = float("-inf")
        x[4] = torch.where(torch.arange(stride, device=DEV) % 2 == 0, 0.0, -0.0)
    return x


@pytest.mark.parametrize("kind", ["normal", "peaked", "tied", "equal", "mixed"])
@pytest.mark.parametrize("stride,fraction", [(36865, 0.1), (40961, 0.001), (70144, 0.1), (4096, 1.0), (12289, 0.9)])
def test_long_rows_equal_one_workgroup_per_row(kind, stride, fraction):
    print(f"case: long top-k {kind} stride={stride} fraction={fraction}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(95)
    rows = 7
    x = _rows(kind, rows, stride, gen)
    n = torch.tensor([stride, stride - 1, stride, stride - 4096, min(stride, 4097), 5, 0], dtype=torch.int32, device=DEV)
    cap = kernels.decode_capacity(stride, fraction)
    lib = _lib.load()
    st = torch.cuda.current_stream().cuda_stream

    def outputs():
        return [torch.full((rows, cap), 77, dtype=torch.int32, device=DEV), torch.full((rows, cap), 77, dtype=torch.uint8, device=DEV),
                torch.zeros(rows, device=DEV), torch.full((rows, cap), 77.0, device=DEV),
                torch.zeros(rows, dtype=torch.int32, device=DEV), torch.zeros(rows, dtype=torch.int32, device=DEV)]

    want, got = outputs(), outputs()
    _lib.check(lib.fl_decode_topk(x.data_ptr(), stride, rows, n.data_ptr(), 1, fraction, cap, *(t.data_ptr() for t in want), st),
               "fl_decode_topk")
    # the workspace function answers 0 for rows that the other call takes; the slices do not mind
    nbytes = rows * 4 * (6 * (-(-stride // 4096)) + 16 + 1024 + 4 + 2048 + 4)
    assert lib.fl_decode_topk_workspace(rows, stride, fraction) <= nbytes
    ws = torch.full((nbytes,), 0xA5, dtype=torch.uint8, device=DEV)
    part = torch.full_like(n, 3)
    _lib.check(lib.fl_decode_topk_long(x.data_ptr(), stride, rows, (n - 4).data_ptr(), part.data_ptr(), 1, 1, fraction, cap,
                                       *(t.data_ptr() for t in got), ws.data_ptr(), nbytes, st), "fl_decode_topk_long")
    for name, a, b in zip(("indices", "valid", "counts", "nonfinite"), (got[0], got[1], got[4], got[5]), (want[0], want[1], want[4], want[5])):
        assert torch.equal(a, b), f"{name} differ in rows {(a != b).reshape(rows, -1).any(1).nonzero().flatten().tolist()}"
    for a, b in ((got[2], want[2]), (got[3], want[3])):
        a, b = a.double().cpu().numpy(), b.double().cpu().numpy()
        assert np.array_equal(np.isnan(a), np.isnan(b))
        assert np.all(np.isnan(b) | (np.abs(a - b) <= 2 * cap * 2.0 ** -24 * np.abs(b)))


def test_long_row_alone_equals_the_row_in_a_batch():
    """A long sequence alone merges its many partials on another path (and divides its top-k over
    workgroups) than as one of a batch: the fp32 sums are grouped differently, nothing else.
    An output is a mix of V rows with weights that add up to 1, so its sums' sizes are at most
    max |v|; a partial adds at most 1250 keys in fp32 (40,000 over 32 waves a row), whose
    roundings average to sqrt(1250) * 2^-24 = 2.1e-6 of that; 4e-6 allows both sides."""
    print("case: long row alone, t=40000", flush=True)
    h, t = 16, 40000
    gen = torch.Generator(device=DEV).manual_seed(99)
    ks, vs = loop_chain(gen, (1, h, t, 128), device=DEV), loop_chain(gen, (1, h, t, 128), device=DEV)
    q, kc, vc = ([x for x in loop_chain(gen, (1, h, 1, 128), device=DEV)] for _ in range(3))
    one = decode_attention_step(CrossLoopKVLayer.from_prefill(ks, vs), q, kc, vc, SCALING)
    many = decode_attention_step(CrossLoopKVLayer.from_prefill([x.expand(6, -1, -1, -1) for x in ks], [x.expand(6, -1, -1, -1) for x in vs]),
                                 *([x.expand(6, -1, -1, -1).contiguous() for x in y] for y in (q, kc, vc)), SCALING)
    size = max(x.float().abs().max().item() for x in vs)
    for i in (0, 5):
        same = (one.indices[0] == many.indices[i]).all(-1)  # (a swap at the boundary changes a head's selection)
        assert int(same.sum()) >= h // 2
        for name in ("out0", "out1", "selected_output", "delta2", "delta3"):
            a, b = getattr(one, name)[0], getattr(many, name)[i]
            if name[:3] != "out":
                a, b = a[same], b[same]
            assert (a - b).abs().max().item() <= 4e-6 * size, name
        # logits are sums of 128 products of sizes up to |q||k| / sqrt(128), about 40
        assert (one.logits1[0, ..., : t + 1] - many.logits1[i, ..., : t + 1]).abs().max().item() <= 128 * 2.0 ** -24 * 40


@pytest.mark.parametrize("rows,stride,n,long", [(16, 70144, 2000, 0), (16, 70144, 70144, 1), (1, 36865, 6000, 0), (1, 36865, 20000, 1),
                                                (192, 40960, 40960, 0), (9, 131072, 131000, 1), (9, 65536, 30000, 1),
                                                (256, 36868, 36868, 0)])
def test_route_by_rows_and_length(rows, stride, n, long):
    """Short, ordinary and many rows of a wide logits buffer on the call that is faster for them;
    either way what one workgroup per row selects (numbers of slices that are multiples of 8 among them)."""
    print(f"case: top-k route rows={rows} stride={stride} n={n}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(98)
    fraction = 0.1
    x = _rows("tied", rows, stride, gen)
    cap = kernels.decode_capacity(n, fraction)
    lib = _lib.load()
    assert lib.fl_decode_topk_long_pays(rows, stride, int(min(stride, cap / fraction)), fraction) == long
    lengths = torch.randint(n // 2, n + 1, (rows,), generator=gen, device=DEV, dtype=torch.int32)
    lengths[0] = n
    idx, valid, mass, w, counts = kernels.decode_topk(x, lengths, fraction, cap)
    want = [torch.empty_like(t) for t in (idx, valid, mass, w, counts)]
    _lib.check(lib.fl_decode_topk(x.data_ptr(), stride, rows, lengths.data_ptr(), 1, fraction, cap, *(t.data_ptr() for t in want),
                                  None, torch.cuda.current_stream().cuda_stream), "fl_decode_topk")
    assert torch.equal(idx, want[0]) and torch.equal(valid, want[1]) and torch.equal(counts, want[4])
    for got, ref in ((mass, want[2]), (w, want[3])):  # the masses sum in another order (see above)
        assert bool(((got - ref).abs() <= 2 * cap * 2.0 ** -24 * ref.abs()).all())
