"""Calls of the anchored-block model and its metrics off the common form: inputs of other lengths and shapes, anchors counted
from the end, decay rates that are not positive, and anchors whose block leaves the sequence."""

import pytest
import torch

from speculators_amd import losses as L
from speculators_amd import metrics as MT
from speculators_amd.dflash import DFlashConfig, DFlashDraftModel

pytestmark = pytest.mark.gpu

T, BS = 64, 4


def _model(from_anchor=False):
    torch.manual_seed(3)
    model = DFlashDraftModel(DFlashConfig(hidden_size=64, num_attention_heads=2, num_key_value_heads=1, head_dim=64,
                                          intermediate_size=64, vocab_size=500, draft_vocab_size=64, num_aux=1,
                                          num_hidden_layers=1, block_size=BS, mask_token_id=499,
                                          sample_from_anchor=from_anchor))
    return model.to(torch.bfloat16).cuda()


def _batch(extra_ids=0, extra_mask=0):
    g = torch.Generator().manual_seed(5)
    return dict(hidden_states=torch.randn(1, T, 64, generator=g).bfloat16().cuda(),
                verifier_last_hidden_states=torch.randn(1, T, 64, generator=g).bfloat16().cuda(),
                document_ids=torch.zeros(1, T, dtype=torch.int64, device="cuda"),
                position_ids=torch.randint(0, 1000, (1, T), generator=g).cuda(),
                input_ids=torch.randint(0, 499, (1, T + extra_ids), generator=g).cuda(),
                loss_mask=(torch.rand(1, T + extra_mask, generator=g) < 0.7).float().cuda())


def _step(model, batch, anchors):
    model.zero_grad(set_to_none=True)
    a = torch.tensor(anchors, device="cuda")
    _, loss, _ = model(**batch, anchors=(a, torch.ones(len(anchors), dtype=torch.bool, device="cuda")))
    loss.backward()
    return loss.detach(), [p.grad for p in model.parameters() if p.requires_grad]


@pytest.mark.parametrize("extra_ids,extra_mask", [(7, 0), (0, 9), (7, 9)])
def test_longer_ids_and_masks(extra_ids, extra_mask):
    model, batch, anchors = _model(), _batch(extra_ids, extra_mask), [1, 17, 33]
    got = _step(model, batch, anchors)
    cut = dict(batch, input_ids=batch["input_ids"][:, :T], loss_mask=batch["loss_mask"][:, :T])
    want = _step(model, cut, anchors)
    assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) for a, b in zip(got[1], want[1], strict=True))


def test_ids_up_to_the_last_anchor():
    model, batch, anchors = _model(), _batch(), [1, 17, 33]
    want = _step(model, batch, anchors)
    got = _step(model, dict(batch, input_ids=batch["input_ids"][:, :34], loss_mask=batch["loss_mask"][:, :37]), anchors)
    assert torch.equal(got[0], want[0]) and all(torch.equal(a, b) for a, b in zip(got[1], want[1], strict=True))


@pytest.mark.parametrize("from_anchor", [False, True])
@pytest.mark.parametrize("ids_len,mask_len", [(T, T), (T + 5, T + 3)])
def test_inputs_are_those_of_plain_indexing(from_anchor, ids_len, mask_len):
    """Rows count from the end of the tensor they are taken of; a block that begins in front of the end wraps."""
    b = _batch(ids_len - T, mask_len - T)
    ids, pos, mask = b["input_ids"], b["position_ids"], b["loss_mask"]
    a, v = torch.tensor([5, -2, 60, -64], device="cuda"), torch.tensor([True, True, False, True], device="cuda")
    model = _model(from_anchor)
    got_ids, q_pos, kv_pos, idx, aligned = (model._inputs if ids_len == T else model._indexed_inputs)(ids, pos, mask, a, v, T)
    rows = (a[:, None] + torch.arange(BS, device="cuda")).reshape(-1)
    want = torch.full((1, a.numel() * BS), 499, device="cuda")
    want[:, ::BS] = ids[:, a]
    block_pos = (pos[0, a][:, None] + torch.arange(BS, device="cuda")).reshape(-1)
    w = mask[:, rows] * v.repeat_interleave(BS)
    if not from_anchor:
        w[:, ::BS] = 0
    assert torch.equal(got_ids, want) and torch.equal(q_pos, block_pos) and torch.equal(kv_pos, torch.cat([pos[0], block_pos]))
    assert torch.equal(idx % T, rows % T if from_anchor else (rows - 1) % T)
    assert torch.equal(aligned, w)


def test_two_rows_of_ids_are_refused():
    b = _batch()
    with pytest.raises((RuntimeError, ValueError)):
        _step(_model(), dict(b, input_ids=b["input_ids"].view(2, T // 2)), [1, 17])


@pytest.mark.parametrize("anchors", [[1, T - BS + 1], [T + 3], [-T - 1, 4]])
@pytest.mark.parametrize("where", ["cuda", "cpu"])
@pytest.mark.parametrize("extra", [0, 7])
def test_a_block_that_leaves_the_sequence_is_refused(anchors, where, extra):
    model, batch = _model(), _batch(extra, 0)
    a = torch.tensor(anchors, device=where)
    with pytest.raises(IndexError):
        model(**batch, anchors=(a, torch.ones(len(anchors), dtype=torch.bool, device=where)))
    _step(model, batch, [1, T - BS])  # (the last one that fits; nothing is left behind)


def test_under_a_default_device():
    model, batch = _model(), _batch()
    want = _step(model, batch, [1, 17])
    with torch.device("cuda"):
        got = _step(model, batch, [1, 17])
    assert torch.equal(got[0], want[0])


@pytest.mark.parametrize("gamma", [-3.0, float("inf"), 0.0, float("nan")])
@pytest.mark.parametrize("from_anchor", [False, True])
def test_decay_rates_that_are_not_positive(gamma, from_anchor):
    g = torch.Generator().manual_seed(2)
    n, vocab = 24, 96
    x, y = (torch.randn(1, n, vocab, generator=g).cuda() for _ in range(2))
    mask = (torch.rand(1, n, generator=g) < 0.8).float().cuda()
    loss, _ = MT.dflash_compute_metrics(x, y, mask, BS, gamma, sample_from_anchor=from_anchor)
    rows = L.kl_div_loss(x, y).double().reshape(-1)
    slot = torch.arange(n, device="cuda").double() % BS
    # (losses/utils.py:17-48)
    w = torch.exp(-slot / gamma) if from_anchor else torch.exp(-(slot - 1).clamp_min(0) / gamma).masked_fill(slot == 0, 0)
    want = (rows * mask.double().reshape(-1) * w).sum() / (mask.double().sum() + 1e-5)
    assert torch.isnan(want) == torch.isnan(loss)
    assert torch.isnan(want) or abs(loss.item() - want.item()) <= 2e-6 * abs(want.item())
