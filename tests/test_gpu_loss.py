"""HIP fused vocabulary loss against the CPU oracle (through the C ABI)."""

import pytest
import torch

from oracle import losses as OL
from oracle import metrics as OM
from oracle import vocab as OV

pytestmark = pytest.mark.gpu

LOSS_TOL = dict(atol=1e-4, rtol=1e-3)  # tests/unit/models/test_fused_losses.py:35
GRAD_TOL = dict(atol=1e-3, rtol=1e-2)  # tests/unit/models/test_fused_losses.py:36
NAMES = ["kl_div", "rkl", "jsd", "ce", "tv", "nla", "lk_hybrid"]


def _check(name, logits, targets, loss_tol=LOSS_TOL, grad_tol=GRAD_TOL):
    from speculators_amd import losses as L

    fn = L.resolve_loss_config(name)[name][0]
    lg = logits.cuda().detach().clone().requires_grad_(True)
    out = fn(lg, targets.cuda())
    assert out.dtype == torch.float32 and out.shape == logits.shape[:-1]
    lo = logits.float().detach().clone().requires_grad_(True)
    ref = OL.LOSS_FNS[name](lo, targets.float())
    torch.testing.assert_close(out.cpu(), ref.detach(), **loss_tol)
    g = torch.Generator().manual_seed(9)
    go = torch.randn(ref.shape, generator=g)
    go[:, ::3] = 0.0  # rows that take the zero-gradient early-out
    (ref * go).sum().backward()
    (out * go.cuda()).sum().backward()
    got = lg.grad.float().cpu()
    torch.testing.assert_close(got, lo.grad, **grad_tol)
    assert (got[:, ::3] == 0).all()


@pytest.mark.parametrize("name", NAMES)
def test_fp32_with_saturated_rows(name):
    # the regime of tests/unit/models/test_fused_losses.py:71-79
    g = torch.Generator().manual_seed(0)
    a = torch.randn(1, 32, 512, generator=g) * 3
    b = torch.randn(1, 32, 512, generator=g) * 3
    a[0, -2:] = -30.0; b[0, -2:] = -30.0
    a[0, -2:, 0] = 30.0; b[0, -2, 0] = 30.0; b[0, -1, 7] = 30.0
    _check(name, a, b)


@pytest.mark.parametrize("name", NAMES)
def test_bf16(name):
    g = torch.Generator().manual_seed(1)
    a = (torch.randn(1, 64, 512, generator=g) * 3).bfloat16()
    b = (torch.randn(1, 64, 512, generator=g) * 3).bfloat16()
    # the oracle computes in fp32 from the same bf16 inputs; the gradient is rounded to bf16
    _check(name, a, b, grad_tol=dict(atol=1e-3, rtol=1e-2))


@pytest.mark.parametrize("name", NAMES)
def test_wide_vocab_151936(name):
    g = torch.Generator().manual_seed(2)
    a = torch.randn(1, 3, 151936, generator=g) * 3
    b = torch.randn(1, 3, 151936, generator=g) * 3
    _check(name, a, b)


@pytest.mark.parametrize("vocab", [1, 7, 8, 9, 250, 32000 + 3])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ragged_vocab_and_unaligned_rows(vocab, dtype):
    from speculators_amd import losses as L

    g = torch.Generator().manual_seed(vocab)
    a = (torch.randn(1, 5, vocab, generator=g) * 2).to(dtype)
    b = (torch.randn(1, 5, vocab, generator=g) * 2).to(dtype)
    rows, am_d, am_t, _ = L.fused_rows(L.OP_KL, a.cuda(), b.cuda())
    torch.testing.assert_close(rows.cpu(), OL.kl_div(a, b), **LOSS_TOL)
    assert torch.equal(am_d.cpu().long(), a.float().argmax(-1))
    assert torch.equal(am_t.cpu().long(), b.float().argmax(-1))


def _float64(name, x, y):
    """Row losses in float64 and the gradient of their sum."""
    x = x.double().requires_grad_(True)
    lp, lq = torch.log_softmax(x, -1), torch.log_softmax(y.double(), -1)
    p, q = lp.exp(), lq.exp()
    if name == "jsd":
        lm = ((p + q) / 2).log()
        rows = 0.5 * ((p * (lp - lm)).sum(-1) + (q * (lq - lm)).sum(-1))
    else:
        rows = (p * (lp - lq)).sum(-1) if name == "rkl" else 1 - torch.minimum(p, q).sum(-1)
    (grad,) = torch.autograd.grad(rows.sum(), x)
    return rows.detach(), grad


@pytest.mark.parametrize("name", ["rkl", "jsd", "tv"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", [(3, 32768), (3, 32775), (3, 32776), (256, 4100), (257, 4100), (257, 5), (520, 1000),
                                        (257, 14336), (257, 14344), (520, 14344), (257, 18432), (257, 18440), (520, 18440)])
def test_two_walks_at_the_edges_of_what_is_held(name, dtype, rows, vocab):
    """Around the narrowest and the widest row that a workgroup keeps, and where the threads of a row change.  Sums of some thousand fp32 terms of one sign against float64: 1e-5 of the row loss; the gradient as the type rounds
    it (bf16: 2^-9 of each value), and tv's where p = q is a tie for one of the two."""
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    x = (torch.randn(1, rows, vocab, device="cuda", generator=g) * 2).to(dtype).requires_grad_(True)
    y = (torch.randn(1, rows, vocab, device="cuda", generator=g) * 2).to(dtype)
    out = L.resolve_loss_config(name)[name][0](x, y)
    (grad,) = torch.autograd.grad(out.sum(), x)
    want, want_grad = _float64(name, x.detach(), y)
    torch.testing.assert_close(out.double(), want, atol=1e-6, rtol=1e-5)
    off = grad.double() - want_grad
    if name == "tv":  # (of the larger rows, too, some columns lie that near: logarithms up to 16, 2^-20 of rounding each)
        lp, lq = (torch.log_softmax(t.detach().double(), -1) for t in (x, y))
        off = off * ((lp - lq).abs() > 2 ** -19)
    err = off.norm() / want_grad.norm()
    assert err < (2e-5 if dtype == torch.float32 else 4e-3), err


@pytest.mark.parametrize("name", ["rkl", "jsd", "tv"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", [(3, 32775), (260, 32775), (3, 18435), (260, 14341)])
def test_columns_behind_the_last_whole_chunk_of_rows_that_are_held(name, dtype, rows, vocab):
    """Rows that begin at 16 bytes and end inside a chunk; their largest value there."""
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    x, y = ((torch.randn(rows, vocab + 8 - vocab % 8, device="cuda", generator=g) * 2).to(dtype)[:, :vocab] for _ in range(2))
    x[:, -1], y[:, -2] = 13.0, 12.0
    loss, lse_d, lse_t, _, am_d, am_t, _, _ = L.fused_loss_forward(L.PRIMITIVE_OP[name], x, y)
    want, _ = _float64(name, x, y)
    torch.testing.assert_close(loss.double(), want, atol=1e-6, rtol=1e-5)
    torch.testing.assert_close(lse_d.double(), x.double().logsumexp(-1), atol=1e-6, rtol=1e-6)
    torch.testing.assert_close(lse_t.double(), y.double().logsumexp(-1), atol=1e-6, rtol=1e-6)
    assert (am_d == vocab - 1).all() and (am_t == vocab - 2).all()


@pytest.mark.parametrize("name", ["jsd", "tv"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", [(300, 4096), (600, 4096), (300, 20000), (600, 20000)])
def test_gathered_rows_are_summed_like_plain_ones(name, dtype, rows, vocab):
    """Bit for bit, but where the fp32 form has fewer threads than the plain one (sums of some thousand terms: 1e-5)."""
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(rows + vocab)
    full = (torch.randn(rows, 2 * vocab, device="cuda", generator=g) * 2).to(dtype)
    x = (torch.randn(rows, vocab, device="cuda", generator=g) * 2).to(dtype)
    d2t = torch.randperm(2 * vocab, device="cuda", generator=g)[:vocab].sort().values - torch.arange(vocab, device="cuda")
    op = L.PRIMITIVE_OP[name]
    step = L.StepPass(d2t=d2t, mask=None, prev=None, counts=torch.zeros(3, device="cuda", dtype=torch.int32))
    got = L.fused_loss_forward(op, x, full, None, step)
    want = L.fused_loss_forward(op, x, L.vocab_gather(full, d2t))
    assert torch.equal(step.gathered, want[7]) and torch.equal(got[4], want[4]) and torch.equal(got[5], want[5])
    for a, b in zip(got[:4], want[:4]):
        if dtype == torch.bfloat16 or vocab == 4096:
            assert torch.equal(a, b)
        torch.testing.assert_close(a, b, atol=1e-6, rtol=1e-5)


def _closed(name, x, y):
    """Row losses and the gradient of their sum in float64, where a probability of nothing has no term."""
    lp, lq = torch.log_softmax(x.double().cpu(), -1), torch.log_softmax(y.double().cpu(), -1)
    p, q = lp.exp(), lq.exp()
    if name == "rkl":
        a = torch.where(p > 0, lp - lq, 0.0)
        rows = (p * a).sum(-1)
        return rows, p * (a - rows[..., None])
    lm = torch.logaddexp(lp, lq) - torch.log(torch.tensor(2.0, dtype=torch.float64))
    a, b = torch.where(p > 0, lp - lm, 0.0), torch.where(q > 0, lq - lm, 0.0)
    ext = (p * a).sum(-1)
    return 0.5 * (ext + (q * b).sum(-1)), 0.5 * p * (a - ext[..., None])


def _ruled_out(rows, vocab, dtype, side, value):
    g = torch.Generator().manual_seed(rows + vocab)
    x, y = (torch.randn(1, rows, vocab, generator=g) * 2 for _ in range(2))
    out = torch.rand(vocab, generator=g) < 0.5
    value = max(value, torch.finfo(dtype).min)
    if side != "target":
        x[..., out] = value
    if side != "draft":
        y[..., out.roll(1) if side == "both" else out] = value
    return x.to(dtype), y.to(dtype)


# one row a workgroup with the pair held, more threads and fewer, the streaming walk, unaligned rows
LOWEST = [(3, 4096), (300, 4096), (600, 4096), (3, 33000), (3, 1001)]


@pytest.mark.parametrize("side", ["draft", "target", "both"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", LOWEST)
@pytest.mark.parametrize("value", [-1e39, -2.4e38, -1e9])
def test_jsd_where_columns_are_ruled_out(rows, vocab, dtype, side, value):
    """Half of the columns at the type's lowest value (or above 2^128 / log2(e), or at a usual mask's): they have no term on
    their side, and the loss stays within log 2."""
    from speculators_amd import losses as L

    x, y = _ruled_out(rows, vocab, dtype, side, value)
    xg = x.cuda().requires_grad_(True)
    out = L.resolve_loss_config("jsd")["jsd"][0](xg, y.cuda())
    (grad,) = torch.autograd.grad(out, xg, torch.ones_like(out))
    want, want_grad = _closed("jsd", x, y)
    torch.testing.assert_close(out.double().cpu(), want, atol=1e-6, rtol=1e-5)
    assert (grad.double().cpu() - want_grad).norm() <= (2e-5 if dtype == torch.float32 else 4e-3) * want_grad.norm()


@pytest.mark.parametrize("side", ["draft", "target", "both"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,vocab", LOWEST)
@pytest.mark.parametrize("value", [-1e39, -1e30, -1e9])
def test_rkl_where_columns_are_ruled_out(rows, vocab, dtype, side, value):
    """Columns that the target rules out and the draft gives weight: the loss is that weight times the value, though the terms
    before the division by the soft-max's sum are too large for the type.  (fp32 sums of terms of one sign: 1e-5.  A gradient's
    rounding is that of the values' differences, 2^-23 of the value times the probability.  Where the draft rules columns out, too,
    their logarithm at the type's lowest value less such a loss is none of the type, and the row has no gradient.)"""
    from speculators_amd import losses as L

    x, y = _ruled_out(rows, vocab, dtype, side, value)
    xg = x.cuda().requires_grad_(True)
    out = L.resolve_loss_config("rkl")["rkl"][0](xg, y.cuda())
    (grad,) = torch.autograd.grad(out, xg, torch.ones_like(out))
    want, want_grad = _closed("rkl", x, y)
    torch.testing.assert_close(out.double().cpu(), want, atol=1e-6, rtol=1e-5)
    if side != "both" or value > -1e38:
        assert (grad.double().cpu() - want_grad).norm() <= (2e-5 if dtype == torch.float32 else 4e-3) * want_grad.norm()


@pytest.mark.parametrize("rows", [5, 300])
@pytest.mark.parametrize("name", ["jsd", "rkl"])
def test_gathered_losses_where_target_columns_are_ruled_out(rows, name):
    from speculators_amd import losses as L

    for dtype in (torch.float32, torch.bfloat16):
        x, y = _ruled_out(rows, 2048, dtype, "target", -1e39)
        full = torch.zeros(rows, 4096, dtype=dtype)
        full[:, ::2] = y[0]
        step = L.StepPass(d2t=torch.arange(2048, device="cuda"), mask=None, prev=None,
                          counts=torch.zeros(3, device="cuda", dtype=torch.int32))
        loss = L.fused_loss_forward(L.PRIMITIVE_OP[name], x[0].cuda(), full.cuda(), None, step)[0]
        torch.testing.assert_close(loss.double().cpu(), _closed(name, x, y)[0][0], atol=1e-6, rtol=1e-5)


def test_reverse_kl_of_rows_a_constant_apart():
    """Rows that differ by little but a constant of 30, whose loss is a difference of 1e-4 beside terms of 30; and columns that
    one side or both rule out (-inf), where it is infinite or not a number as the sum of its terms is."""
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(5)
    y = torch.randn(1, 40, 3000, device="cuda", generator=g)
    x = y + 30 + 0.02 * torch.randn(1, 40, 3000, device="cuda", generator=g)
    fn = L.resolve_loss_config("rkl")["rkl"][0]
    x = x.requires_grad_(True)
    out = fn(x, y)
    (grad,) = torch.autograd.grad(out.sum(), x)
    want, want_grad = _float64("rkl", x.detach(), y)
    # a logit of 30 is rounded by 2^-20, a difference of two of them by as much: 1e-6 of terms of 0.02
    torch.testing.assert_close(out.double(), want, atol=1e-7, rtol=1e-3)
    assert (grad.double() - want_grad).norm() < 1e-3 * want_grad.norm()
    y[0, 0, 7] = -float("inf")
    x.data[0, 1, 9] = y[0, 1, 9] = -float("inf")
    out = fn(x.detach(), y)
    assert out[0, 0] == float("inf") and out[0, 1].isnan() and out[0, 2:].isfinite().all()


def test_argmax_first_index_on_ties_bit_exact():
    from speculators_amd import losses as L
    from speculators_amd.metrics import argmax_rows

    g = torch.Generator().manual_seed(3)
    # coarse bf16 values: many exact ties per row
    a = (torch.randint(-4, 5, (1, 257, 32000), generator=g).float() * 0.5).bfloat16()
    b = (torch.randint(-4, 5, (1, 257, 32000), generator=g).float() * 0.5).bfloat16()
    _, am_d, am_t, _ = L.fused_rows(L.OP_KL, a.cuda(), b.cuda())
    assert torch.equal(am_d.cpu().long(), a.float().argmax(-1))
    assert torch.equal(am_t.cpu().long(), b.float().argmax(-1))
    assert torch.equal(argmax_rows(a.cuda()).cpu(), a.float().argmax(-1))
    # a late unique maximum and an early one
    a[0, 0, :] = 0; a[0, 0, 31999] = 1
    a[0, 1, :] = 0; a[0, 1, 0] = 1
    assert argmax_rows(a.cuda())[0, :2].tolist() == [31999, 0]


def test_vocab_gather_bit_exact():
    from speculators_amd import losses as L

    g = torch.Generator().manual_seed(4)
    vt, vd = 128256, 32000
    sel = torch.randperm(vt, generator=g)[:vd]
    d2t, t2d = OV.build_vocab_mappings(sel.tolist(), vt)
    full = (torch.randn(1, 9, vt, generator=g) * 2).bfloat16()
    got = L.vocab_gather(full.cuda(), d2t.cuda()).cpu()
    assert torch.equal(got, OV.gather_targets(full, d2t))
    assert torch.equal(got, full[..., t2d])
    full32 = torch.randn(3, vt, generator=g)
    assert torch.equal(L.vocab_gather(full32.cuda(), d2t.cuda()).cpu(), full32[..., t2d])


@pytest.mark.parametrize("op_name", ["kl_div", "rkl", "jsd", "ce", "tv"])
@pytest.mark.parametrize("dtype,vt,vd", [(torch.bfloat16, 128256, 32000), (torch.float32, 1000, 333),
                                         (torch.bfloat16, 5003, 1001)])
def test_step_pass_gathers_and_counts_in_the_row_pass(op_name, dtype, vt, vd):
    """The one-pass form (targets read through d2t, acceptance chain inside the row pass) against
    the three-kernel form (gather, loss, chain reduce): gathered rows bit-exact against the
    oracle's index mapping, row losses / statistics / arg-maxes bit-identical, counts and the
    in-place ``prev_correct`` identical."""
    from speculators_amd import _lib
    from speculators_amd import losses as L

    g = torch.Generator().manual_seed(vt + vd)
    rows = 37
    sel = torch.randperm(vt, generator=g)[:vd]
    d2t, t2d = OV.build_vocab_mappings(sel.tolist(), vt)
    full = (torch.randn(rows, vt, generator=g) * 2).to(dtype).cuda()
    logits = (torch.randn(rows, vd, generator=g) * 2).to(dtype).cuda()
    compact = L.vocab_gather(full, d2t.cuda())
    assert torch.equal(compact.cpu(), OV.gather_targets(full.cpu(), d2t))
    for i in range(0, rows, 3):  # a third of the rows agree with their target
        logits[i, compact[i].float().argmax()] = 30.0
    mask = (torch.rand(rows, generator=g) < 0.7).float().cuda()
    prev0 = (torch.rand(rows, generator=g) < 0.8).cuda()
    op = L.PRIMITIVE_OP[op_name]

    ref = L.fused_loss_forward(op, logits, compact)
    out = torch.empty(6, device="cuda")
    prev_ref = prev0.clone()
    _lib.call("spx_ttt_step_reduce", _lib.ptr(ref[0]), _lib.ptr(ref[4]), _lib.ptr(ref[5]), _lib.ptr(mask),
              _lib.kind_code(mask), _lib.ptr(prev_ref), _lib.kind_code(prev_ref), rows, 0.7,
              _lib.ptr(out), None, _lib.stream_ptr(mask.device))

    prev_got = prev0.clone()
    step = L.StepPass(d2t=d2t.cuda(), mask=mask, prev=prev_got,
                      counts=torch.zeros(3, dtype=torch.int32, device="cuda"))
    got = L.fused_loss_forward(op, logits, full, step=step)
    assert torch.equal(step.gathered, compact)
    for a, b in zip(got[:6], ref[:6], strict=True):
        assert torch.equal(a, b)
    assert torch.equal(prev_got, prev_ref)
    assert step.counts.tolist() == [int(out[1]), int(out[2]), int(out[4])]
    out2 = torch.empty(6, device="cuda")
    _lib.call("spx_ttt_step_mean", _lib.ptr(got[0]), _lib.ptr(mask), _lib.kind_code(mask), rows, 0.7,
              _lib.ptr(step.counts), _lib.ptr(out2), None, _lib.stream_ptr(mask.device))
    assert torch.equal(out2, out)


@pytest.mark.parametrize("op_name", ["kl_div", "ce"])
@pytest.mark.parametrize("known", [False, True])
@pytest.mark.parametrize("vocab", [32000, 32768, 8, 1000])
def test_row_pass_that_also_writes_the_logits_gradient(op_name, known, vocab):
    """``spx_vocab_loss_step_fwd_grad`` (a workgroup keeps the row pair in registers: loss, statistics,
    acceptance chain and the unit-weight logits gradient of the unmasked rows in ONE read of the rows)
    against the streaming kernels: arg-maxes, counts and ``prev_correct`` identical, row losses and
    log-sum-exps within 1e-5 (another summation order), masked rows with known statistics report a
    zero loss; the packed gradient rows against ``softmax(x) - softmax(y)`` / ``softmax(x) - onehot``
    in fp32 (one bf16 rounding); the scaled unpack."""
    from speculators_amd import _lib
    from speculators_amd import losses as L

    g = torch.Generator().manual_seed(vocab + 7 * known)
    rows = 41
    logits = (torch.randn(rows, vocab, generator=g) * 2).bfloat16().cuda()
    targets = (torch.randn(rows, vocab, generator=g) * 2).bfloat16().cuda()
    for i in range(0, rows, 3):
        logits[i, targets[i].float().argmax()] = 30.0
    targets[5, 1] = targets[5].float().max()  # a tie inside the target row: the first index wins
    targets[5, 0] = targets[5, 1]
    mask = (torch.rand(rows, generator=g) < 0.7).float().cuda()
    mask[0], mask[1] = 0.0, 1.0
    prev0 = (torch.rand(rows, generator=g) < 0.8).cuda()
    op = L.PRIMITIVE_OP[op_name]

    base = L.fused_loss_forward(op, logits, targets)  # the statistics of step 0
    stats = (base[2].clone(), base[5].clone()) if known else None
    prev_ref = prev0.clone()
    step_ref = L.StepPass(mask=mask, prev=prev_ref, counts=torch.zeros(3, dtype=torch.int32, device="cuda"))
    ref = L.fused_loss_forward(op, logits, targets, stats, step=step_ref)

    prev_got = prev0.clone()
    step = L.StepPass(mask=mask, prev=prev_got, counts=torch.zeros(3, dtype=torch.int32, device="cuda"),
                      grad_in_pass=True)
    assert L._one_pass_ok(op, logits, targets, step)
    loss, lse_t, am_d, am_t, packed, row_map, count = L._loss_forward_with_grad(
        op, logits, None if (known and op_name == "ce") else targets, stats, step)
    live = mask.bool()
    n_live = int(live.sum())
    assert int(count) == n_live
    assert torch.equal(am_d, ref[4]) and torch.equal(am_t, ref[5])
    assert torch.equal(prev_got, prev_ref) and step.counts.tolist() == step_ref.counts.tolist()
    want_loss = ref[0] if not known else torch.where(live, ref[0], torch.zeros_like(ref[0]))
    if op_name == "ce" and not known:
        want_loss = ref[0]  # without known statistics every row is reduced in full
    assert (loss - want_loss).abs().max().item() <= 1e-5 * max(1.0, want_loss.abs().max().item())
    assert (lse_t - ref[2]).abs().max().item() <= 1e-5 * max(1.0, ref[2].abs().max().item())

    p = torch.softmax(logits.float(), -1)
    if op_name == "ce":
        q = torch.nn.functional.one_hot(ref[5].long(), vocab).float()
    else:
        q = torch.softmax(targets.float(), -1)
    want = (p - q)[live]
    got = packed[:n_live].float()
    assert (got - want).abs().max().item() <= 2 ** -8 * want.abs().max().item() + 1e-6
    assert torch.equal(row_map[live].long().cpu(), torch.arange(n_live)) and (row_map[~live] == -1).all()

    scale = torch.randn(rows, generator=g).cuda()
    cols = packed[:, :8].contiguous()
    out = L._unpack_rows_scaled(cols, row_map, scale, rows + 3)
    want_out = torch.zeros(rows + 3, 8, device="cuda")
    want_out[:rows][live] = cols[:n_live].float() * scale[live, None]
    assert torch.equal(out, want_out.bfloat16())


def test_compute_metrics_with_target_gather_equals_materialised_targets():
    """compute_metrics over three TTT steps with the targets given as full-vocabulary logits +
    d2t (first step reads through the table and leaves the draft-vocabulary rows behind) against
    the same call on gathered targets: every metric, the loss and the gradients bit for bit."""
    from speculators_amd import losses as L
    from speculators_amd.metrics import TargetGather, compute_metrics

    g = torch.Generator().manual_seed(8)
    t, vt, vd, steps = 130, 4000, 1000, 3
    sel = torch.randperm(vt, generator=g)[:vd]
    d2t, _ = OV.build_vocab_mappings(sel.tolist(), vt)
    full = (torch.randn(1, t, vt, generator=g) * 2).bfloat16().cuda()
    mask = (torch.rand(1, t, generator=g) < 0.7).float().cuda()
    logits = [(torch.randn(1, t, vd, generator=g) * 2).bfloat16().cuda() for _ in range(steps)]
    runs = []
    for form in ("gather", "materialised"):
        tg = TargetGather(full, d2t.cuda()) if form == "gather" else L.vocab_gather(full, d2t.cuda())
        prev, cache, res = mask.clone(), {}, []
        for k in range(steps):
            lg = logits[k].clone().requires_grad_(True)
            loss, m = compute_metrics(lg, tg, mask, prev, k, 0.9, L.resolve_loss_config("kl_div"),
                                      target_stats_cache=cache)
            loss.backward()
            res.append((loss.detach(), m, lg.grad, prev.clone()))
        if form == "gather":
            assert torch.equal(tg.compact, L.vocab_gather(full, d2t.cuda()))
        runs.append(res)
    for (la, ma, ga, pa), (lb, mb, gb, pb) in zip(*runs, strict=True):
        assert torch.equal(la, lb) and torch.equal(ga, gb) and torch.equal(pa, pb)
        assert ma.keys() == mb.keys()
        for key in ma:
            assert torch.equal(ma[key], mb[key]), key


@pytest.mark.parametrize("mask_dtype", [torch.float32, torch.bool, torch.int64, torch.bfloat16])
def test_eagle3_compute_metrics_chain_matches_oracle(mask_dtype):
    from speculators_amd import losses as L
    from speculators_amd.metrics import compute_metrics

    g = torch.Generator().manual_seed(5)
    t, v, steps = 300, 1000, 4
    targets = (torch.randn(1, t, v, generator=g) * 2).bfloat16()
    mask = (torch.rand(1, t, generator=g) < 0.7).to(mask_dtype)
    prev_ref = mask.clone()
    prev_gpu = mask.clone().cuda()
    for k in range(steps):
        logits = (torch.randn(1, t, v, generator=g) * 2).bfloat16()
        for i in range(0, t - k, 2):  # make half the rows agree with the shifted target
            logits[0, i, targets[0, i + k].float().argmax()] = 20.0
        lg = logits.cuda().requires_grad_(True)
        loss, m = compute_metrics(lg, targets.cuda(), mask.cuda(), prev_gpu, k, 0.8,
                                  L.resolve_loss_config("kl_div"))
        lo = logits.float().requires_grad_(True)
        rloss, rm = OM.eagle3_compute_metrics(lo, targets.float(), mask, prev_ref, k, 0.8)
        assert loss.item() == pytest.approx(rloss.item(), rel=1e-3)
        for key in rm:
            if "acc" in key:  # integer counts: bit exact
                assert m[key].item() == rm[key].item(), key
            else:
                assert m[key].item() == pytest.approx(rm[key].item(), rel=1e-3), key
        assert set(m) == set(rm)
        assert torch.equal(prev_gpu.cpu(), prev_ref) and prev_gpu.dtype == mask_dtype
        loss.backward(); rloss.backward()
        torch.testing.assert_close(lg.grad.float().cpu(), lo.grad, atol=1e-5, rtol=2e-2)


def test_compound_loss_config_and_no_mask():
    from speculators_amd import losses as L
    from speculators_amd.metrics import compute_metrics

    g = torch.Generator().manual_seed(6)
    logits = torch.randn(1, 40, 333, generator=g)
    targets = torch.randn(1, 40, 333, generator=g)
    cfg = L.resolve_loss_config('{"ce": 0.25, "tv": 0.75}')
    loss, m = compute_metrics(logits.cuda(), targets.cuda(), None, None, 2, 0.5, cfg)
    rloss, rm = OM.eagle3_compute_metrics(logits, targets, None, None, 2, 0.5,
                                          OL.resolve_loss_config({"ce": 0.25, "tv": 0.75}))
    assert set(m) == set(rm)
    for key in rm:
        assert m[key].item() == pytest.approx(rm[key].item(), rel=1e-3, abs=1e-6), key


@pytest.mark.parametrize("weighting", ["fixed-exp-decay", "dpace"])
def test_dflash_compute_metrics_matches_oracle(weighting):
    from speculators_amd import losses as L
    from speculators_amd.metrics import dflash_compute_metrics

    g = torch.Generator().manual_seed(7)
    bs, a, v = 8, 37, 2000
    logits = (torch.randn(1, a * bs, v, generator=g) * 2).bfloat16()
    targets = (torch.randn(1, a * bs, v, generator=g) * 2).bfloat16()
    for i in range(0, a * bs, 3):
        logits[0, i, targets[0, i].float().argmax()] = 20.0
    mask = (torch.rand(1, a * bs, generator=g) < 0.8).float()
    mask[:, ::bs] = 0
    name = "ce" if weighting == "dpace" else "kl_div"
    lg = logits.cuda().requires_grad_(True)
    loss, m = dflash_compute_metrics(lg, targets.cuda(), mask.cuda(), bs, 4.0,
                                     L.resolve_loss_config(name), weighting, 0.5)
    lo = logits.float().requires_grad_(True)
    rloss, rm = OM.dflash_compute_metrics(lo, targets.float(), mask, bs, 4.0,
                                          OL.resolve_loss_config(name), weighting, 0.5)
    assert set(m) == set(rm)
    for key in rm:
        if "acc" in key:
            assert m[key].item() == rm[key].item(), key
        else:
            assert m[key].item() == pytest.approx(rm[key].item(), rel=1e-3, abs=1e-6), key
    loss.backward(); rloss.backward()
    torch.testing.assert_close(lg.grad.float().cpu(), lo.grad, atol=1e-5, rtol=2e-2)


def test_full_size_rows_properties():
    """Config[1] row shape (32000-wide bf16): properties that need no oracle at size --
    KL(x, x) == 0, loss >= 0, gradient rows sum to ~0, determinism."""
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(8)
    x = (torch.randn(1, 4096, 32000, device="cuda", generator=g) * 2).bfloat16().requires_grad_(True)
    y = (torch.randn(1, 4096, 32000, device="cuda", generator=g) * 2).bfloat16()
    same = L.kl_div_loss(x.detach(), x.detach())
    assert same.abs().max().item() < 1e-4
    rows, am_d, _, _ = L.fused_rows(L.OP_KL, x, y)
    rows2, am_d2, _, _ = L.fused_rows(L.OP_KL, x, y)
    assert torch.equal(rows, rows2) and torch.equal(am_d, am_d2)
    assert (rows >= 0).all()
    rows.sum().backward()
    assert x.grad.float().sum(-1).abs().max().item() < 2e-2
    # a 64-row sample against the oracle
    idx = torch.arange(0, 4096, 64)
    ref = OL.kl_div(x.detach()[:, idx].cpu(), y[:, idx].cpu())
    torch.testing.assert_close(rows[:, idx].detach().cpu(), ref, **LOSS_TOL)


def test_full_size_row_pass_with_gradient_properties():
    """The one-read row pass at the 8B draft's row shape (4096 x 32000 bf16, 70 % of the rows live, target
    statistics of an earlier step handed in): against the streaming kernels on the same rows -- arg-maxes,
    counts and chain identical, row losses within 1e-5 -- and through what needs no oracle at size: KL rows
    >= 0, every gradient row sums to ~0 (two soft-maxes), the gradient of a row paired with itself is zero,
    two runs agree bit for bit."""
    from speculators_amd import losses as L

    g = torch.Generator(device="cuda").manual_seed(9)
    t, v = 4096, 32000
    x = (torch.randn(t, v, device="cuda", generator=g) * 2).bfloat16()
    y = (torch.randn(t, v, device="cuda", generator=g) * 2).bfloat16()
    y[7] = x[7]  # a row paired with itself
    mask = (torch.rand(t, device="cuda", generator=g) < 0.7).float()
    mask[7] = 1.0
    base = L.fused_loss_forward(L.OP_KL, x, y)
    known = (base[2].clone(), base[5].clone())
    prev0 = torch.rand(t, device="cuda", generator=g) < 0.8

    def run(one_pass):
        prev = prev0.clone()
        step = L.StepPass(mask=mask, prev=prev, counts=torch.zeros(3, dtype=torch.int32, device="cuda"),
                          grad_in_pass=one_pass)
        if one_pass:
            out = L._loss_forward_with_grad(L.OP_KL, x, y, known, step)
            return out, prev, step.counts
        return L.fused_loss_forward(L.OP_KL, x, y, known, step=step), prev, step.counts

    (loss, _lse_t, am_d, am_t, packed, row_map, count), prev_a, counts_a = run(True)
    ref, prev_b, counts_b = run(False)
    live = mask.bool()
    n_live = int(live.sum())
    assert int(count) == n_live and counts_a.tolist() == counts_b.tolist() and torch.equal(prev_a, prev_b)
    assert torch.equal(am_d, ref[4]) and torch.equal(am_t, ref[5])
    assert (loss[live] - ref[0][live]).abs().max().item() <= 1e-5 * ref[0].abs().max().item()
    assert (loss[~live] == 0).all() and (loss >= -1e-5).all()
    grad = packed[:n_live].float()
    assert grad.sum(-1).abs().max().item() < 2e-2
    assert grad[int(row_map[7])].abs().max().item() == 0.0
    packed2 = L._loss_forward_with_grad(L.OP_KL, x, y, known, L.StepPass(
        mask=mask, prev=prev0.clone(), counts=torch.zeros(3, dtype=torch.int32, device="cuda"), grad_in_pass=True))[4]
    assert torch.equal(packed2[:n_live], packed[:n_live])
    # a 32-row sample against the closed form in fp32
    idx = torch.nonzero(live).flatten()[::97][:32]
    want = torch.softmax(x[idx].float(), -1) - torch.softmax(y[idx].float(), -1)
    got = packed[row_map[idx].long()].float()
    assert (got - want).abs().max().item() <= 2 ** -8 * want.abs().max().item() + 1e-7


@pytest.mark.parametrize("op_name", ["kl_div", "ce"])
def test_reused_target_statistics_give_the_same_rows(op_name):
    """Steps >= 1 reuse the verifier rows' lse / arg-max from step 0: same loss, arg-maxes
    and gradient as recomputing them."""
    from speculators_amd import losses as L

    op = L.PRIMITIVE_OP[op_name]
    g = torch.Generator().manual_seed(11)
    t, v, k = 200, 4000, 3
    logits = (torch.randn(1, t, v, generator=g) * 2).bfloat16().cuda()
    targets = (torch.randn(1, t, v, generator=g) * 2).bfloat16().cuda()
    _, _, am_full, lse_full = L.fused_rows(op, logits, targets)
    a = logits[:, : t - k].detach().clone().requires_grad_(True)
    b = logits[:, : t - k].detach().clone().requires_grad_(True)
    fresh, pd_f, pt_f, _ = L.fused_rows(op, a, targets[:, k:])
    known = (lse_full.reshape(-1)[k:], am_full.reshape(-1)[k:])
    reused, pd_r, pt_r, _ = L.fused_rows(op, b, targets[:, k:], known)
    assert torch.equal(pd_f, pd_r) and torch.equal(pt_f, pt_r)
    torch.testing.assert_close(reused, fresh, atol=2e-6, rtol=1e-5)
    go = torch.randn_like(fresh)
    (fresh * go).sum().backward(); (reused * go).sum().backward()
    torch.testing.assert_close(b.grad.float(), a.grad.float(), atol=1e-6, rtol=1e-3)


@pytest.mark.parametrize("live_fraction", [0.15, 0.45, 1.0])
def test_head_and_loss_node_with_the_input_gradient_in_parts(live_fraction, monkeypatch):
    """The frozen head + loss node over a sparse loss mask: its input-gradient product runs over the
    packed live rows and, when their tiles are few, with the contraction cut into parts
    (``spx_gemm_bf16_nt_rows_split``).  Against the same node with the cut switched off (one rounding of
    a bf16 value apart) and against autograd through the fp32 oracle loss; dead rows get exact zeros."""
    from speculators_amd import gemm as G
    from speculators_amd import losses as L

    t, h, vd = 1024, 512, 4096
    g = torch.Generator().manual_seed(int(live_fraction * 100))
    x = (torch.randn(1, t, h, generator=g) * 0.5).bfloat16()
    w = (torch.randn(vd, h, generator=g) * 0.05).bfloat16()
    tg = (torch.randn(1, t, vd, generator=g) * 2).bfloat16()
    mask = (torch.rand(1, t, generator=g) < live_fraction).float()
    grads = {}
    for parts in (4, 1):
        monkeypatch.setattr(G, "SPLIT_PARTS", parts)
        xg = x.cuda().requires_grad_(True)
        wc = w.cuda()
        loss = L.head_fused_rows(L.OP_KL, xg, wc, wc.t().contiguous(), tg.cuda())[0]
        (loss * mask.cuda()).sum().backward()
        grads[parts] = xg.grad.float().cpu()
    xr = x.float().requires_grad_(True)
    # (the oracle sees the logits the kernel sees: rounded to bf16, gradient straight through)
    logits = xr @ w.float().t()
    logits = logits + (logits.detach().bfloat16().float() - logits.detach())
    ref = OL.kl_div(logits, tg.float())
    (ref * mask).sum().backward()
    want = xr.grad
    scale = want.abs().max().item()
    dead = mask[0] == 0
    for parts in (4, 1):
        assert (grads[parts][0][dead] == 0).all()
        assert (grads[parts] - want).abs().max().item() <= 2e-2 * scale + 1e-6, parts
    assert (grads[4] - grads[1]).abs().max().item() <= 1e-2 * scale + 1e-6


@pytest.mark.parametrize("op_name", ["kl_div", "ce"])
@pytest.mark.parametrize("case", ["even", "skewed", "ragged", "one_tile", "clustered"])
def test_pipelined_gather_pass_on_the_edges_of_its_tiling(op_name, case):
    """The pipelined form of the one-pass kernel (bf16, 16-byte aligned rows, kl / ce: spans of the
    full row staged two tiles deep, picks with lane = id) against the three-kernel form, bit for bit:
    a table spread evenly; one that is dense at the low ids and sparse at the high ones, so that
    the spans of the late tiles do not fit a buffer and are read directly; a draft vocabulary that
    ends inside a chunk of 8 (rows kept aligned by their stride); one smaller than a tile; ids
    clustered in two far-apart runs (a span boundary inside a tile)."""
    from speculators_amd import _lib
    from speculators_amd import losses as L

    g = torch.Generator().manual_seed(len(case) * 7 + len(op_name))
    rows = 21
    if case == "even":
        vt, vd = 40000, 9000
        sel = torch.randperm(vt, generator=g)[:vd]
    elif case == "skewed":
        vt, vd = 200000, 6144
        dense = torch.arange(4000)                                  # ids 0..3999 map to themselves
        sparse = 4000 + torch.randperm(vt - 4000, generator=g)[:vd - 4000]  # 2144 ids over 196000 columns
        sel = torch.cat([dense, sparse])
    elif case == "ragged":
        vt, vd = 30000, 4099
        sel = torch.randperm(vt, generator=g)[:vd]
    elif case == "one_tile":
        vt, vd = 3000, 700
        sel = torch.randperm(vt, generator=g)[:vd]
    else:
        vt, vd = 150000, 5000
        sel = torch.cat([torch.arange(100, 2600), torch.arange(140000, 142500)])
    d2t, _ = OV.build_vocab_mappings(sel.tolist(), vt)
    vt_ld, vd_ld = -(-vt // 8) * 8, -(-vd // 8) * 8
    full = (torch.randn(rows, vt_ld, generator=g) * 2).bfloat16().cuda()[:, :vt]
    logits = (torch.randn(rows, vd_ld, generator=g) * 2).bfloat16().cuda()[:, :vd]
    compact = L.vocab_gather(full.contiguous(), d2t.cuda())
    assert torch.equal(compact.cpu(), OV.gather_targets(full.cpu(), d2t))
    for i in range(0, rows, 3):
        logits[i, compact[i].float().argmax()] = 30.0
    mask = (torch.rand(rows, generator=g) < 0.7).float().cuda()
    prev0 = (torch.rand(rows, generator=g) < 0.8).cuda()
    op = L.PRIMITIVE_OP[op_name]
    ref = L.fused_loss_forward(op, logits, compact)
    out = torch.empty(6, device="cuda")
    prev_ref = prev0.clone()
    _lib.call("spx_ttt_step_reduce", _lib.ptr(ref[0]), _lib.ptr(ref[4]), _lib.ptr(ref[5]), _lib.ptr(mask),
              _lib.kind_code(mask), _lib.ptr(prev_ref), _lib.kind_code(prev_ref), rows, 0.7,
              _lib.ptr(out), None, _lib.stream_ptr(mask.device))
    prev_got = prev0.clone()
    step = L.StepPass(d2t=d2t.cuda(), mask=mask, prev=prev_got,
                      counts=torch.zeros(3, dtype=torch.int32, device="cuda"))
    assert full.stride(0) % 8 == 0 and logits.stride(0) % 8 == 0  # the pipelined kernel's precondition
    got = L.fused_loss_forward(op, logits, full, step=step)
    assert torch.equal(step.gathered, compact)
    names = ("loss", "lse_draft", "lse_target", "extra", "argmax_draft", "argmax_target")
    for name, a, b in zip(names, got[:6], ref[:6], strict=True):
        if op_name == "ce" and name in ("lse_target", "extra"):
            continue  # not defined for ce
        assert torch.equal(a, b), name
    assert torch.equal(prev_got, prev_ref)
    assert step.counts.tolist() == [int(out[1]), int(out[2]), int(out[4])]


@pytest.mark.parametrize("n,tail,vocab,dtype", [(0, 3, 5, torch.float32), (1, 0, 8, torch.bfloat16),
                                                (255, 1, 2047, torch.bfloat16), (257, 4, 32000, torch.bfloat16),
                                                (300, 2, 2056, torch.float32)])
def test_row_tokens_widen_the_known_and_find_the_rest(n, tail, vocab, dtype):
    from speculators_amd.metrics import row_tokens

    g = torch.Generator().manual_seed(n + vocab)
    known = torch.randint(0, vocab, (n,), generator=g, dtype=torch.int32)
    rows = torch.randint(-4, 5, (n + tail, vocab), generator=g).to(dtype)  # many equal maxima: the first one counts
    got = row_tokens(known.cuda(), rows.cuda()[n:])
    want = torch.cat([known.long(), torch.tensor([int((r == r.max()).nonzero()[0]) for r in rows[n:].float()],
                                                 dtype=torch.int64)])
    assert got.shape == (1, n + tail) and torch.equal(got[0].cpu(), want)


@pytest.mark.parametrize("rows", [1, 1023, 1025, 3000])
@pytest.mark.parametrize("kind", [torch.bool, torch.int64, torch.bfloat16])
def test_mask_row_map_and_step_total(rows, kind):
    from speculators_amd import _lib

    g = torch.Generator().manual_seed(rows)
    mask = (torch.rand(rows, generator=g) < 0.6).to(kind).cuda()
    out = torch.full((rows + 4,), 7, device="cuda", dtype=torch.int32)
    st = _lib.stream_ptr(mask.device)
    _lib.call("spx_mask_row_map", mask, _lib.kind_code(mask), rows, out, out[rows:], out[rows + 1:], st)
    live = mask.cpu().float() != 0
    want = torch.where(live, live.long().cumsum(0) - 1, torch.tensor(-1))
    assert torch.equal(out[:rows].cpu().long(), want) and out[rows:].tolist() == [int(live.sum()), 0, 0, 0]
    loss = torch.randn(rows, generator=g).cuda()
    counts = torch.tensor([3, 5, 9], device="cuda", dtype=torch.int32)
    a, b = torch.empty(8, device="cuda"), torch.empty(6, device="cuda")
    rw = torch.empty(2, rows, device="cuda")
    before, total = torch.tensor(2.5, device="cuda"), torch.empty((), device="cuda")
    _lib.call("spx_ttt_step_mean", loss, mask, _lib.kind_code(mask), rows, 0.7, counts, b, rw[0], st)
    _lib.call("spx_ttt_step_total", loss, None, None, mask, _lib.kind_code(mask), None, 0, rows, 0.7, counts, 0.25,
              before, total, a, rw[1], st)
    assert torch.equal(a[:6], b) and torch.equal(rw[0], rw[1]) and a[7].item() == 1.0
    assert a[6].item() == b[0].item() * 0.25 and abs(total.item() - (2.5 + a[6].item())) < 1e-6


def _rows_without_a_maximum(vocab, dtype):
    """Rows of -infinity, NaN, both, and the type's lowest value with one larger value or none; plain rows between them."""
    g = torch.Generator().manual_seed(vocab)
    x = torch.randn(9, vocab, generator=g)
    x[0], x[2], x[4, :] = float("-inf"), float("nan"), torch.finfo(dtype).min
    x[6, :] = torch.finfo(dtype).min
    x[6, vocab - 1] = -2.0
    x[8, : vocab // 2], x[8, vocab // 2:] = float("nan"), float("-inf")
    return x.to(dtype)


@pytest.mark.parametrize("vocab,dtype", [(50, torch.bfloat16), (1000, torch.float32), (32000, torch.bfloat16),
                                         (33000, torch.bfloat16), (7, torch.float32)])
def test_arg_max_outputs_are_columns_of_the_row(vocab, dtype):
    """Rows of -infinity, NaN or the type's lowest value (a masked-out vocabulary, a draft that diverged): every arg-max is
    a column, torch's where it is defined, and a statistic handed in that is none reads nothing outside the row."""
    from speculators_amd import gemm
    from speculators_amd import losses as L
    from speculators_amd import metrics as MT

    x = _rows_without_a_maximum(vocab, dtype)
    y = x.flip(0).contiguous()
    want_x, want_y = (t.masked_fill(t.isnan(), float("-inf")).argmax(-1) for t in (x, y))
    xg, yg = x.cuda().unsqueeze(0), y.cuda().unsqueeze(0)
    assert torch.equal(MT.argmax_rows(xg)[0].cpu(), want_x)
    for op in (L.OP_KL, L.OP_CE, L.OP_RKL, L.OP_JSD, L.OP_TV):
        rows, am_d, am_t, lse_t = L.fused_rows(op, xg, yg)
        assert torch.equal(am_d[0].cpu().long(), want_x) and torch.equal(am_t[0].cpu().long(), want_y)
    # cross-entropy of a target row without a maximum: the draft's value in column 0
    rows, _, _, _ = L.fused_rows(L.OP_CE, xg[:, 1:2], yg[:, 8:9])
    ref = torch.logsumexp(x[1].double(), -1) - x[1, 0].double()
    assert abs(rows.item() - ref.item()) <= 1e-5 * abs(ref.item()) + 1e-5
    # known statistics of such a row, as an earlier pass of another program may have left them
    for bad in (0x7fffffff, vocab, -1):
        known = (torch.zeros(9, device="cuda"), torch.full((9,), bad, device="cuda", dtype=torch.int32))
        rows, am_d, _, _ = L.fused_rows(L.OP_CE, xg, yg, known)
        assert torch.equal(am_d[0].cpu().long(), want_x)
        assert abs(rows[0, 1].item() - ref.item()) <= 1e-5 * abs(ref.item()) + 1e-5
        if dtype == torch.bfloat16 and vocab % 8 == 0 and vocab <= 32768:
            step = L.StepPass(mask=torch.ones(9, device="cuda"), counts=torch.zeros(3, device="cuda", dtype=torch.int32),
                              grad_in_pass=True)
            loss, _, am_d, *_ = L._loss_forward_with_grad(L.OP_CE, xg[0], None, known, step)
            assert torch.equal(am_d.cpu().long(), want_x)
            assert abs(loss[1].item() - ref.item()) <= 1e-5 * abs(ref.item()) + 1e-5
    # the head product's epilogue: a row of NaN and one of -infinity (the product of -inf and ones)
    a = torch.ones(4, 64, device="cuda").bfloat16()
    a[1], a[2] = float("nan"), float("-inf")
    _, _, am = gemm.gemm_nt_stats(a, torch.ones(max(vocab, 8), 64, device="cuda").bfloat16())
    assert am.tolist() == [0, 0, 0, 0]


def test_arg_max_of_gathered_targets_is_a_column():
    """The pass that reads full-vocabulary targets through the offset table, with a target row of -infinity."""
    from speculators_amd import losses as L

    vt, vd = 4096, 1024
    x = torch.randn(5, vd, device="cuda").bfloat16()
    full = torch.randn(5, vt, device="cuda").bfloat16()
    full[1] = float("-inf")
    x[3] = float("-inf")
    d2t = torch.arange(vd, device="cuda") * 3
    for op in (L.OP_KL, L.OP_CE):
        step = L.StepPass(d2t=d2t, mask=None, prev=None, counts=torch.zeros(3, device="cuda", dtype=torch.int32))
        _, _, _, _, am_d, am_t, _, _ = L.fused_loss_forward(op, x, full, None, step)
        assert torch.equal(am_d.long(), x.argmax(-1))
        assert torch.equal(am_t.long(), full[:, torch.arange(vd, device="cuda") * 4].argmax(-1))
