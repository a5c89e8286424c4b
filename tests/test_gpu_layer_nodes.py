"""What the one-node decoder layers (``layer.py``) must keep of the layers put together from their parts: autograd's
check of what a backward pass reads, the modules a program may hook or replace, parameters in any storage order."""

import pytest
import torch

pytestmark = pytest.mark.gpu

FAMILIES = ("eagle3", "eagle3x2", "dflash", "mtp")
LAYER = {"eagle3": "layers.0", "eagle3x2": "layers.1", "dflash": "layers.1", "mtp": "mtp_layers.0"}


def _family(name):
    """``(model, position_ids, forward)`` of a small bf16 model; ``forward()`` returns the loss."""
    dev = "cuda"
    g = torch.Generator().manual_seed(21)
    torch.manual_seed(20)
    kw = dict(hidden_size=256, num_attention_heads=4, num_key_value_heads=2, head_dim=64, intermediate_size=320)
    t = 150

    def randn(*shape):
        return torch.randn(*shape, generator=g).bfloat16().to(dev)

    ids = torch.randint(0, 512, (1, t), generator=g).to(dev)
    mask = (torch.rand(1, t, generator=g) < 0.7).to(dev)
    doc = torch.arange(t).div(80, rounding_mode="floor").view(1, t).to(dev)
    pos = (torch.arange(t) % 80).view(1, t).to(dev)
    if name.startswith("eagle3"):
        from speculators_amd.eagle3 import Eagle3Config, Eagle3DraftModel

        model = Eagle3DraftModel(Eagle3Config(vocab_size=512, draft_vocab_size=512,
                                              num_hidden_layers=2 if name.endswith("x2") else 1, **kw))
        batch = dict(hidden_states=randn(1, t, 768), input_ids=ids, document_ids=doc, loss_mask=mask,
                     position_ids=pos, verifier_last_hidden_states=randn(1, t, 256), ttt_steps=3)
        at = 1
    elif name == "dflash":
        from speculators_amd.dflash import DFlashConfig, DFlashDraftModel

        model = DFlashDraftModel(DFlashConfig(vocab_size=512, draft_vocab_size=512, num_aux=2, num_hidden_layers=2,
                                              block_size=8, mask_token_id=7, **kw))
        anchors = torch.tensor([3, 20, 41, 77, 90, 120], device=dev)
        batch = dict(hidden_states=randn(1, t, 512), input_ids=ids, document_ids=doc, loss_mask=mask.float(),
                     position_ids=pos, verifier_last_hidden_states=randn(1, t, 256),
                     anchors=(anchors, torch.ones(6, dtype=torch.bool, device=dev)))
        at = 1
    else:
        from speculators_amd.mtp import MTPConfig, MTPDraftModel

        model = MTPDraftModel(MTPConfig(vocab_size=512, num_speculative_steps=2, **kw))
        batch = dict(input_ids=ids, hidden_states=randn(1, t, 256), position_ids=pos, loss_mask=mask.float())
        at = 1
    model = model.to(dev).bfloat16()
    return model, pos, lambda: model(**batch)[at]


def _grads(model, forward):
    model.zero_grad()
    loss = forward()
    loss.backward()
    return loss.detach(), {n: p.grad for n, p in model.named_parameters() if p.grad is not None}


def _same(got, want):
    assert torch.equal(got[0], want[0])
    assert got[1].keys() == want[1].keys() and len(want[1]) >= 8
    for n, w in want[1].items():
        assert torch.equal(got[1][n], w), n


@pytest.mark.parametrize("family,what", [("eagle3", "self_attn.o_proj"), ("eagle3", "mlp.down_proj"),
                                         ("eagle3", "positions"), ("eagle3x2", "mlp.down_proj"),
                                         ("dflash", "self_attn.q_proj"), ("dflash", "self_attn.o_proj"),
                                         ("dflash", "mlp.down_proj"), ("mtp", "self_attn.o_proj"),
                                         ("mtp", "mlp.down_proj"), ("mtp", "positions")])
def test_a_value_changed_in_place_before_the_backward_is_refused(family, what):
    """bf16 parameters used as they lie and the caller's positions: changed between forward and backward they would give
    the gradient of another function, and autograd says so -- also in the second pass over a retained graph."""
    model, pos, forward = _family(family)
    value = pos if what == "positions" else model.get_parameter(f"{LAYER[family]}.{what}.weight")
    loss = forward()
    loss.backward(retain_graph=True)  # unchanged: fine
    with torch.no_grad():
        value.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def test_parameters_the_layer_reads_a_copy_of_may_change():
    """The merged q/k/v and gate/up weights are copies: the gradient is that of the values the forward saw."""
    model, _, forward = _family("eagle3")
    want = _grads(model, forward)
    model.zero_grad()
    loss = forward()
    with torch.no_grad():
        model.layers[0].self_attn.k_proj.weight.mul_(2)
        model.layers[0].mlp.up_proj.weight.zero_()
    loss.backward()
    _same((loss.detach(), {n: p.grad for n, p in model.named_parameters() if p.grad is not None}), want)


CALLED = {"eagle3": ("self_attn", "mlp"), "eagle3x2": ("self_attn", "mlp"),
          "dflash": ("self_attn", "mlp", "self_attn.q_norm", "self_attn.k_norm"),
          "mtp": ("self_attn", "mlp", "input_layernorm", "self_attn.q_norm", "self_attn.k_norm")}


@pytest.mark.parametrize("family,path", [(f, p) for f in FAMILIES for p in CALLED[f]])
@pytest.mark.parametrize("way", ["hook", "pre_hook", "backward_hook", "instance", "replaced"])
def test_modules_inside_a_layer_are_called_when_a_program_watches_them(family, path, way):
    """Hooks on the modules inside a layer run, a replaced module or method is used, and what they change counts."""
    model, _, forward = _family(family)
    plain = forward().detach()
    layer = model.get_submodule(LAYER[family])
    module, calls = layer.get_submodule(path), []

    def doubled(out):
        calls.append(path)
        return out * 2

    if way == "hook":
        module.register_forward_hook(lambda m, a, out: doubled(out))
    elif way == "pre_hook":
        module.register_forward_pre_hook(lambda m, a: (doubled(a[0]), *a[1:]))
    elif way == "backward_hook":
        module.register_full_backward_hook(lambda m, gi, go: calls.append(path))
    elif way == "instance":
        own = module.forward
        module.forward = lambda *a: doubled(own(*a))
    else:
        class Wrapped(torch.nn.Module):
            def __init__(self):
                super().__init__()
                self.inner = module

            def __getattr__(self, name):
                try:
                    return super().__getattr__(name)
                except AttributeError:
                    return getattr(super().__getattr__("inner"), name)

            def forward(self, *a):
                return doubled(self.inner(*a))

        parent, _, leaf = path.rpartition(".")
        setattr(layer.get_submodule(parent) if parent else layer, leaf, Wrapped())
    loss = forward()
    loss.backward()
    assert calls and torch.isfinite(loss)
    # (an input norm of twice its input is the same norm)
    norm_in = way == "pre_hook" and path.endswith("norm")
    assert torch.equal(loss.detach(), plain) == (way == "backward_hook") or norm_in


def test_global_hooks_and_a_class_method_replaced_see_the_inner_modules(monkeypatch):
    from speculators_amd import eagle3 as E

    model, _, forward = _family("eagle3")
    plain = _grads(model, forward)
    seen = []
    handle = torch.nn.modules.module.register_module_forward_hook(lambda m, a, out: seen.append(type(m).__name__))
    try:
        _same(_grads(model, forward), plain)  # the layer put together from its parts is the same function
    finally:
        handle.remove()
    assert seen.count("Attention") == seen.count("MLP") == 3
    own = E.MLP.forward
    monkeypatch.setattr(E.MLP, "forward", lambda self, x: own(self, x) * 2)
    assert not torch.equal(forward().detach(), plain[0])


def test_a_layer_output_replaced_by_a_hook_keeps_its_gradient():
    """A forward hook on a layer that scales the normed state handed to the next layer: the scaling saves that state, which
    later steps must not overwrite."""
    from speculators_amd import eagle3 as E

    losses, grads = [], []
    for parts in (False, True):
        model, _, forward = _family("eagle3x2")
        scale = torch.nn.Parameter(torch.full((256,), 1.25, device="cuda", dtype=torch.bfloat16))
        model.layers[0].register_forward_hook(lambda m, a, out: (out[0], out[1] * scale))
        step = E.DecoderLayer._step
        if parts:
            E.DecoderLayer._step = lambda self, *a: None
        try:
            loss = forward()
            loss.backward()
        finally:
            E.DecoderLayer._step = step
        losses.append(loss.detach())
        grads.append(scale.grad.float())
    assert torch.equal(losses[0], losses[1])
    assert (grads[0] - grads[1]).abs().max() <= 2e-2 * grads[1].abs().max()


LONE = {"eagle3": ("self_attn.o_proj", "mlp.down_proj"),
        "dflash": ("self_attn.q_proj", "self_attn.o_proj", "mlp.down_proj"),
        "mtp": ("input_proj", "self_attn.o_proj", "mlp.down_proj")}


@pytest.mark.parametrize("family", sorted(LONE))
@pytest.mark.parametrize("order", ["columns", "odd_address", "odd_rows", "wide_rows"])
def test_bf16_weights_in_any_storage_order(family, order):
    """Weights that lie column by column, at an address or with a row stride the kernels do not take, or with a gap between
    the rows: the same results, bit for bit."""
    model, _, forward = _family(family)
    want = _grads(model, forward)
    layer = model.get_submodule(LAYER[family])
    for path in LONE[family]:
        lin = layer.get_submodule(path)
        w = lin.weight.detach()
        n, k = w.shape
        if order == "columns":
            new = w.t().contiguous().t()
        elif order == "odd_address":
            new = torch.empty(n * k + 1, device=w.device, dtype=w.dtype)[1:].view(n, k).copy_(w)
        else:
            new = torch.empty(n, k + (3 if order == "odd_rows" else 64), device=w.device, dtype=w.dtype)[:, :k].copy_(w)
        assert torch.equal(new, w) and new.stride() + (new.data_ptr() % 16,) != w.stride() + (0,)
        lin.weight = torch.nn.Parameter(new)
    _same(_grads(model, forward), want)
    with torch.no_grad():
        assert torch.isfinite(forward())


def test_native_sequences_run_without_the_interpreter_lock():
    """What launches several kernels or allocates from C++ lets other Python threads run meanwhile: with forced switches out
    of the picture a second thread gets its turn only where a call gives the interpreter's lock up.  (The call is refused
    behind that point: the allocator may give the lock up by itself.)"""
    import sys
    import threading

    from speculators_amd import _lib

    a, b = torch.zeros(64, 64, device="cuda").bfloat16(), torch.zeros(64, 32, device="cuda").bfloat16()
    native = _lib.native()
    gate, ran, attempts = threading.Lock(), [], 0
    gate.acquire()

    def other():
        with gate:
            ran.append(True)

    thread = threading.Thread(target=other)
    thread.start()
    interval = sys.getswitchinterval()
    try:
        sys.setswitchinterval(1000.0)
        gate.release()
        while not ran and attempts < 20000:
            attempts += 1
            try:
                native.product(0, a, b, None, 1, None)
            except ValueError:
                pass
        got = bool(ran)
    finally:
        sys.setswitchinterval(interval)
    thread.join()
    assert got


@pytest.mark.parametrize("family,frozen", [(f, n) for f in FAMILIES for n in (
    "norm", "post_attention_layernorm", "input_layernorm", "hidden_norm" if f.startswith("eagle3") else "q_norm")])
def test_gains_that_do_not_train(family, frozen, monkeypatch):
    """Frozen norms (all, or one of a layer's): no gradient for them, every other gradient that of the layer put together
    from its parts."""
    from speculators_amd import dflash, eagle3, mtp

    results = []
    for parts in (False, True):
        model, _, forward = _family(family)
        names = [n for n, p in model.named_parameters() if frozen in n and p.requires_grad]
        assert names
        for n in names:
            model.get_parameter(n).requires_grad_(False)
        if parts:
            for cls in (eagle3.DecoderLayer, dflash.DFlashDecoderLayer, mtp.MTPLayer):
                monkeypatch.setattr(cls, "_step", lambda self, *a: None)
        results.append(_grads(model, forward))
    (loss, grads), (want_loss, want) = results
    assert abs(loss.item() - want_loss.item()) <= 2e-3 * abs(want_loss.item())
    assert grads.keys() == want.keys() and not any(frozen in n for n in grads) and len(want) >= 5
    for n, w in want.items():
        assert (grads[n].float() - w.float()).abs().max() <= 2e-2 * w.float().abs().max() + 1e-6, n
