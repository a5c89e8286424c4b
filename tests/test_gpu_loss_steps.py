"""Head and loss of all steps of a TTT loop in one node against the same steps one by one (``metrics.compute_metrics``)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

H = 64


def _case(t, steps, vocab, seed, mask_dtype=torch.float32, live=0.6):
    g = torch.Generator().manual_seed(seed)
    x = [torch.randn(1, t, H, generator=g).bfloat16().cuda() for _ in range(steps)]
    w = (torch.randn(vocab, H, generator=g) * 0.4).bfloat16().cuda()
    y = (torch.randn(1, t, vocab, generator=g) * 2).bfloat16().cuda()
    # some draft rows agree with their target, so that the acceptance chain has something to count
    for k in range(steps):
        n = t - k
        for r in range(0, n, 3):
            y[0, r + k, int((x[k][0, r].float() @ w.float().T).argmax())] += 12
    mask = (torch.rand(1, t, generator=g) < live).to(mask_dtype).cuda()
    return x, w, y, mask


def _one_by_one(x, w, y, mask, decay, config):
    from speculators_amd import metrics as MT

    xs = [v.clone().requires_grad_(True) for v in x]
    prev, cache, loss, metrics, tokens = mask.clone(), {}, None, {}, []
    for k, v in enumerate(xs):
        loss, m, tok = MT.compute_metrics(MT.Head(v, w, w.t().contiguous()), y, mask, prev, k, decay, loss_config=config,
                                          target_stats_cache=cache, total_in=loss, return_tokens=True)
        metrics.update(m)
        tokens.append(tok)
    grads = torch.autograd.grad(loss, xs)
    return loss, metrics, tokens, prev, grads


def _together(x, w, y, mask, decay, config, grad=True):
    from speculators_amd import metrics as MT

    xs = [v.clone().requires_grad_(grad) for v in x]
    prev = mask.clone()
    run = MT.TTTSteps.take(xs[0], w, y, mask, prev, len(xs), decay, config)
    assert run is not None
    for v in xs:
        run.add(v)
    loss, metrics, tokens = run.finish(w, w.t().contiguous())
    return loss, metrics, tokens, prev, torch.autograd.grad(loss, xs) if grad else None


def _close(a, b, rel):
    a, b = a.double(), b.double()
    assert (a - b).norm() <= rel * b.norm() + 1e-12


# edges of a workgroup's chunks (512 x 8 columns), of the reduction's 256 rows and of the rows that have no target
@pytest.mark.parametrize("t,steps,vocab", [(2, 2, 4096), (7, 7, 4104), (255, 3, 32000), (257, 5, 32768), (600, 32, 4160)])
@pytest.mark.parametrize("name", ["kl_div", "ce", "tv", '{"ce": 0.1, "tv": 0.9}', '{"kl_div": 0.5, "ce": 0.2}',
                                  '{"tv": 1.5, "kl_div": 0.25, "ce": 0.125}'])
def test_steps_together(t, steps, vocab, name):
    from speculators_amd import losses as L

    config = L.resolve_loss_config(name)
    case = _case(t, steps, vocab, t + steps)
    want = _one_by_one(*case, 0.9, config)
    got = _together(*case, 0.9, config)
    # sums of fp32 in another order over at most 600 rows of 32768 columns: 2^-24 * (log2 of the length + a few)
    _close(got[0], want[0], 4e-6)
    assert got[1].keys() == want[1].keys() and list(got[1]) == list(want[1])
    for key, v in want[1].items():
        if "acc" in key or key.endswith("total"):
            assert torch.equal(got[1][key], v), key
        else:
            _close(got[1][key], v, 4e-6)
    for a, b in zip(got[2], want[2], strict=True):
        assert a.dtype == b.dtype and torch.equal(a, b)
    assert torch.equal(got[3], want[3])
    for a, b in zip(got[4], want[4], strict=True):
        assert a.shape == b.shape and a.dtype == b.dtype
        # the packed bf16 gradient rows differ by a rounding here and there, the products by the order of their parts
        _close(a, b, 2.0 ** -8)
    # without gradients: the same numbers (masked rows are formed, but weigh nothing)
    plain = _together(*case, 0.9, config, grad=False)
    _close(plain[0], got[0], 1e-6)
    assert all(torch.equal(a, b) for a, b in zip(plain[2], got[2], strict=True)) and torch.equal(plain[3], got[3])


@pytest.mark.parametrize("dtype,live", [(torch.bool, 0.5), (torch.int64, 0.5), (torch.bfloat16, 1.0), (torch.float32, 0.0)])
def test_masks(dtype, live):
    from speculators_amd import losses as L

    config = {"kl_div": (L.kl_div_loss, 0.7)}
    case = _case(130, 4, 4096, 3, dtype, live)
    want, got = _one_by_one(*case, 1.0, config), _together(*case, 1.0, config)
    _close(got[0], want[0], 4e-6)
    for key, v in want[1].items():
        torch.testing.assert_close(got[1][key], v, rtol=4e-6, atol=0)
    assert torch.equal(got[3], want[3])
    for a, b in zip(got[4], want[4], strict=True):
        assert torch.isfinite(a).all()
        _close(a, b, 2.0 ** -8)


def test_steps_in_several_passes_and_extreme_rows(monkeypatch):
    """Few logits at a time give the same bits; a masked row of infinities and NaN reaches neither loss nor gradient behind
    the first step, a target without a value above -infinity counts as column 0."""
    from speculators_amd import losses as L

    config = L.resolve_loss_config("ce")
    x, w, y, mask = _case(40, 5, 4096, 11)
    mask[0, 20] = 0
    x[2][0, 18] = float("nan")
    y[0, 7] = -float("inf")
    got = _together(x, w, y, mask, 0.8, config)
    want = _one_by_one(x, w, y, mask, 0.8, config)
    assert torch.isfinite(got[0])
    _close(got[0], want[0], 4e-6)
    assert all(torch.equal(a, b) for a, b in zip(got[2], want[2], strict=True))
    monkeypatch.setattr(L, "STEPS_LOGITS_BYTES", 2 * 40 * 4096 * 2)
    again = _together(x, w, y, mask, 0.8, config)
    assert torch.equal(again[0], got[0]) and all(torch.equal(a, b) for a, b in zip(again[4], got[4], strict=True))


@pytest.mark.parametrize("name", ["kl_div", "ce", '{"ce": 0.1, "tv": 0.9}'])
def test_targets_gathered_from_the_full_vocabulary(name):
    from speculators_amd import losses as L
    from speculators_amd import metrics as MT

    x, w, y, mask = _case(70, 3, 4096, 5)
    g = torch.Generator().manual_seed(2)
    ids = torch.randperm(9000, generator=g)[:4096].sort().values.cuda()
    full = torch.randn(1, 70, 9000, generator=g).bfloat16().cuda()
    full[..., ids] = y
    d2t = ids - torch.arange(4096, device="cuda")
    config = L.resolve_loss_config(name)
    want = _together(x, w, y, mask, 0.9, config)
    got = _together(x, w, MT.TargetGather(full, d2t), mask, 0.9, config)
    assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) for a, b in zip(got[2] + list(got[4]), want[2] + list(want[4])))
    old = _one_by_one(x, w, MT.TargetGather(full, d2t), mask, 0.9, config)
    _close(got[0], old[0], 4e-6)
    for a, b in zip(got[4], old[4], strict=True):
        _close(a, b, 2.0 ** -8)


def test_what_goes_step_by_step():
    from speculators_amd import losses as L
    from speculators_amd import metrics as MT

    x, w, y, mask = _case(24, 3, 4096, 1)
    kl = L.resolve_loss_config("kl_div")

    def taken(steps=3, targets=y, m=mask, config=kl, weight=w):
        return MT.TTTSteps.take(x[0], weight, targets, m, mask.clone(), steps, 1.0, config) is not None

    assert taken() and taken(config=None)
    assert not taken(steps=1) and not taken(steps=25) and not taken(steps=33) and not taken(m=None)
    assert taken(config=L.resolve_loss_config("tv")) and not taken(config=L.resolve_loss_config('{"ce": 1, "rkl": 1}'))
    assert not taken(config=L.resolve_loss_config("jsd")) and not taken(config=L.resolve_loss_config("nla"))
    assert not taken(config={"kl_div": (lambda a, b: a, 1.0)}) and not taken(targets=y.float())
    assert not taken(targets=y[..., 1:], weight=w[1:]) and not taken(targets=y[..., :4088], weight=w[:4088])


# (a chunk, a last chunk that a part of one wave holds, all chunks of all threads)
@pytest.mark.parametrize("vocab", [4096, 4104, 32768])
@pytest.mark.parametrize("name", ["kl_div", '{"tv": 1.5, "kl_div": 0.25, "ce": 0.125}'])
def test_target_rows_held_as_probabilities(vocab, name):
    """Rows that nearly agree, columns of the type's lowest value, and an infinite target: as step by step."""
    from speculators_amd import losses as L

    config = L.resolve_loss_config(name)
    x, w, y, mask = _case(50, 3, vocab, 5)
    y[0] = (x[0][0].float() @ w.float().T).bfloat16()
    y[0, :, vocab // 2:] = torch.finfo(torch.bfloat16).min
    want, got = _one_by_one(x, w, y, mask, 0.9, config), _together(x, w, y, mask, 0.9, config)
    # differences of two log-sum-exps of magnitude <= 16 (ulp 2^-20 at most), each within two units, over three steps
    assert (got[0] - want[0]).abs() <= 12 * 2.0 ** -20 + 4e-6 * want[0].abs()
    for a, b in zip(got[4], want[4], strict=True):
        _close(a, b, 2.0 ** -8)
    y[0, 25, 3] = -float("inf")
    mask[0, 25] = 1
    want, got = _one_by_one(x, w, y, mask, 0.9, config), _together(x, w, y, mask, 0.9, config)
    assert torch.equal(got[0].isnan(), want[0].isnan())


@pytest.mark.parametrize("top", [2.0 ** 100, 2.0 ** 121, 2.0 ** 125, 1.5 * 2.0 ** 121])
@pytest.mark.parametrize("name", ["kl_div", '{"tv": 1.5, "kl_div": 0.25, "ce": 0.125}'])
def test_a_target_row_at_the_edges_of_the_type(top, name):
    """A largest logit beyond 1.3e36 beside the lowest value.  A power of two times log2(e) is exact, and so are the log-sum-exp and
    the probability of one: the loss is finite as step by step.  Others round to probabilities of zero: no NaN from these."""
    from speculators_amd import losses as L

    config = L.resolve_loss_config(name)
    x, w, y, mask = _case(20, 2, 4104, 6)
    y[0, 11], mask[0, 11] = torch.finfo(torch.bfloat16).min, 1
    y[0, 11, 40] = top
    want, got = _one_by_one(x, w, y, mask, 0.9, config), _together(x, w, y, mask, 0.9, config)
    assert not got[0].isnan()
    if top == 1.5 * 2.0 ** 121:
        return
    assert got[0].isfinite() and want[0].isfinite()
    # sums of terms of the size of top, each rounded to 24 bits, and the log-sum-exp of that size
    assert (got[0] - want[0]).abs() <= 16 * 2.0 ** -24 * abs(top)
    for a, b in zip(got[4], want[4], strict=True):
        _close(a, b, 2.0 ** -8)
