"""Which prefill path a model takes: the HIP row kernels for plain modules, the modules themselves
where one is replaced, hooked or laid out otherwise.  The reference is the dense looped model
(``dense_forward``), which always calls the modules."""

import pytest
import torch

pytestmark = pytest.mark.gpu

from flashloop_amd.config import FlashLoopConfig  # noqa: E402
from flashloop_amd.engine import FlashLoopEngine  # noqa: E402
from flashloop_amd.model import OuroConfig, OuroForCausalLM, RMSNorm  # noqa: E402

TINY = OuroConfig(vocab_size=1024, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                  num_attention_heads=2, num_key_value_heads=2)
ALL_ROWS = FlashLoopConfig(prefill_fraction_loop3=1.0, prefill_fraction_loop4=1.0)
IDS = torch.randint(0, TINY.vocab_size, (1, 150), generator=torch.Generator().manual_seed(120))


def _model():
    return OuroForCausalLM.random_init(TINY, seed=121, device="cuda")


def _rel(got, want):
    return float((got.double() - want.double()).norm() / want.double().norm())


def _like_the_modules(model, what):
    """Prefill with every row active equals the dense model.  Bound: about ten bf16 roundings
    (2^-9 each) in each of 2 layers x 4 loops, adding up at random: sqrt(80) * 2^-9 = 1.8e-2."""
    ids = IDS.cuda()
    got, want = FlashLoopEngine(model, config=ALL_ROWS).prefill(ids).logits, model.dense_forward(ids)
    assert _rel(got, want) < 3e-2, f"{what}: {_rel(got, want):.3e} from the modules"
    return want


def test_hooked_final_norm_is_called():
    print("case: hooked final norm", flush=True)
    model = _model()
    calls = []
    model.model.norm.register_forward_hook(lambda m, a, out: (calls.append(1), out * 3.0)[1])
    plain = _like_the_modules(_model(), "plain")
    hooked = _like_the_modules(model, "hooked final norm")
    assert len(calls) == 8 and _rel(hooked, plain) > 0.1  # (both models, four loops each; the change is well past the bound)


def test_final_norm_of_another_class_is_called():
    """A subclass with its own eps, large enough to matter."""
    print("case: final norm of another class", flush=True)

    class Other(RMSNorm):
        pass

    model = _model()
    model.model.norm = Other(TINY.hidden_size, 4.0).to("cuda", torch.bfloat16)
    assert _rel(_like_the_modules(model, "another class"), _like_the_modules(_model(), "plain")) > 0.1


REPLACED = ["model.layers.1.self_attn.q_proj", "model.layers.0.self_attn.o_proj", "model.layers.0.mlp.up_proj",
            "model.layers.1.mlp", "model.layers.0.input_layernorm", "model.layers.1.post_attention_layernorm_2", "model.norm"]


@pytest.mark.parametrize("name", REPLACED)
def test_replaced_forward_is_called(name):
    """A ``forward`` replaced on the instance, as wrapping and offloading tools do it."""
    print(f"case: replaced forward {name}", flush=True)
    model = _model()
    m = model.get_submodule(name)
    calls, forward = [], m.forward
    m.forward = lambda x: (calls.append(1), forward(x) * 2.0)[1]
    _like_the_modules(model, name)
    assert len(calls) == 8  # (both models, four loops each)


def test_class_forward_and_global_hook_are_called():
    """A class whose ``forward`` was replaced, and a hook on every module."""
    print("case: replaced class forward, global hook", flush=True)
    plain = _like_the_modules(_model(), "plain")
    forward = RMSNorm.forward
    RMSNorm.forward = lambda self, x: forward(self, x) * 2.0
    try:
        assert _rel(_like_the_modules(_model(), "class forward"), plain) > 0.1
    finally:
        RMSNorm.forward = forward
    hook = torch.nn.modules.module.register_module_forward_hook(
        lambda m, a, out: out * 2.0 if isinstance(m, RMSNorm) else None)
    try:
        assert _rel(_like_the_modules(_model(), "global hook"), plain) > 0.1
    finally:
        hook.remove()


def test_replaced_embedding_and_rotary_of_a_decode_step_are_called():
    print("case: replaced embedding and rotary", flush=True)
    ids = IDS.cuda()
    for name in ("model.embed_tokens", "model.rotary_emb"):
        model = _model()
        eng = FlashLoopEngine(model, use_graphs=False)
        eng.prefill(ids)
        m = model.get_submodule(name)
        calls, forward = [], type(m).forward
        type(m).forward = lambda self, *a: (calls.append(1), forward(self, *a))[1]
        try:
            eng.decode(ids[:, :1])
        finally:
            type(m).forward = forward
        assert len(calls) == 1, name


@pytest.mark.parametrize("name", ["model.norm", "model.layers.1.post_attention_layernorm"])
def test_misaligned_norm_weight(name):
    """A norm weight that starts two bytes into its storage, which a 16-byte load cannot take."""
    print(f"case: misaligned {name}", flush=True)
    model = _model()
    w = torch.rand(TINY.hidden_size + 1, device="cuda", generator=torch.Generator("cuda").manual_seed(122)).add_(0.5).bfloat16()[1:]
    assert w.data_ptr() % 16 == 2
    model.get_submodule(name).weight = torch.nn.Parameter(w)
    _like_the_modules(model, "misaligned norm weight")


def test_rotary_tables_of_another_layout():
    """A rotary module whose tables are not contiguous."""
    print("case: strided rotary tables", flush=True)
    model = _model()
    rot = model.model.rotary_emb
    forward = rot.forward
    rot.forward = lambda x, p: torch.stack(forward(x, p), dim=-1).unbind(-1)
    _like_the_modules(model, "strided rotary tables")


def test_embedding_rows_of_another_layout():
    """An embedding module whose rows are two bytes off, or lie apart."""
    print("case: embedding rows of another layout", flush=True)
    for offset, gap in ((1, 0), (0, 8)):
        model = _model()
        emb = model.model.embed_tokens
        forward = emb.forward

        def apart(ids, forward=forward, offset=offset, gap=gap):
            h = forward(ids)
            room = h.new_zeros(offset + h.shape[0] * h.shape[1] * (h.shape[2] + gap))[offset:]
            out = room.view(h.shape[0], h.shape[1], h.shape[2] + gap)[..., : h.shape[2]]
            return out.copy_(h)

        emb.forward = apart
        _like_the_modules(model, f"embedding rows offset={offset} gap={gap}")


def test_prefill_attention_scale_is_that_of_the_modules():
    """The modules' attention divides by sqrt(head_dim), whatever ``scaling`` says."""
    print("case: scaling attribute", flush=True)
    model = _model()
    for layer in model.model.layers:
        layer.self_attn.scaling *= 16.0
    with torch.no_grad():
        for layer in model.model.layers:  # scores that matter
            layer.self_attn.q_proj.weight.mul_(10.0)
    _like_the_modules(model, "scaling attribute")


def test_module_path_equals_the_kernels():
    """Token-sparse loops over the same rows on both paths (a hook without effect keeps the
    modules): K/V of every loop and layer, and the logits.  1000 keys: the kernels divide the
    250 and 100 active rows' keys over several workgroups."""
    print("case: module path and kernels", flush=True)
    model = _model()
    ids = torch.randint(0, TINY.vocab_size, (1, 1000), generator=torch.Generator().manual_seed(123)).cuda()
    eng = FlashLoopEngine(model)
    chosen, calls = [], []
    select = eng._select

    def keep(*args, **kw):
        chosen.append(select(*args, **kw))
        return chosen[-1]

    with torch.inference_mode():
        eng._select = keep
        a = eng._prefill_loops(ids, all_logits=True)
        model.model.layers[0].mlp.up_proj.register_forward_hook(lambda m, x, out: calls.append(1))
        rows = iter(chosen)
        eng._select = lambda *args, **kw: next(rows)
        b = eng._prefill_loops(ids, all_logits=True)
    assert len(calls) == 4 and [r.active_rows for r in a.receipts] == [1000, 1000, 250, 100]
    assert torch.equal(a.mask3, b.mask3) and torch.equal(a.mask4, b.mask4)
    # the bound of _like_the_modules
    assert _rel(a.logits, b.logits) < 3e-2
    for loop in range(4):
        for li in range(TINY.num_hidden_layers):
            for x, y in ((a.keys, b.keys), (a.values, b.values)):
                assert _rel(x[loop][li], y[loop][li]) < 3e-2, f"loop {loop + 1} layer {li}"
