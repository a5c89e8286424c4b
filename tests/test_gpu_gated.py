"""The first product of a gated MLP with its activation (spx_gemm_bf16_gated) against the product and the SwiGLU launch."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _operands(m, f, k, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(m, k, generator=g).bfloat16().cuda()
    w = (torch.randn(2 * f, k, generator=g) * 4 * k ** -0.5).bfloat16().cuda()
    return a, w


def _separately(a, w):
    from speculators_amd import _lib

    m, f, k = a.shape[0], w.shape[0] // 2, a.shape[1]
    gu = torch.empty(m, 2 * f, device="cuda", dtype=torch.bfloat16)
    _lib.call("spx_gemm_bf16_nt", a, k, w, k, gu, 2 * f, m, 2 * f, k, _lib.stream_ptr(a.device))
    return gu, _activation(gu)


def _activation(gu):
    from speculators_amd import _lib

    m, f = gu.shape[0], gu.shape[1] // 2
    act = torch.empty(m, f, device="cuda", dtype=torch.bfloat16)
    _lib.call("spx_swiglu_rows_fwd", gu, 2 * f, gu[:, f:], 2 * f, act, f, m, f, _lib.stream_ptr(gu.device))
    return act


# one slab beyond the first two; rows at the edges of a tile and of its 16-row blocks; one to five tiles for a workgroup; results
# past the caches (> 256 MiB)
@pytest.mark.parametrize("m,f,k", [(1, 256, 192), (15, 512, 256), (257, 768, 192), (255, 256, 1024), (700, 16384, 192), (2300, 16384, 320),
                                   (8200, 8192, 256)])
@pytest.mark.parametrize("keep", [False, True])
def test_against_two_launches(m, f, k, keep):
    a, w = _operands(m, f, k, m + f)
    gu, act = _separately(a, w)
    got, kept = _at_once(a, w, keep)
    if keep:
        assert torch.equal(kept, gu)  # the same sums in the same order
    assert torch.equal(got, act)  # (the activation's bits: test_every_value_of_a_gate)


# last rounds in two, three and four parts: four cut tiles behind 256 whole ones, 128 of them, and nothing but cut tiles
@pytest.mark.parametrize("m,f,k,parts", [(257, 16640, 2048, 2), (700, 16384, 2048, 4), (1, 256, 3136, 3), (700, 2560, 4096, 4)])
def test_a_cut_last_round(m, f, k, parts):
    a, w = _operands(m, f, k, m + f)
    want, _ = _separately(a, w)
    got, gu = _at_once(a, w, True, parts)
    # fp32 sums of the parts' sums, 2^-24 sqrt(k) of 4 |x| at most apart from the whole's: now and then the next bf16
    assert ((gu.double() - want.double()).abs() <= 2 ** -7 * want.double().abs() + 2 ** -20 * k ** 0.5).all()
    assert (gu != want).double().mean() <= 0.02
    assert torch.equal(got, _activation(gu))
    assert torch.equal(_at_once(a, w, False, parts)[0], got)


def _at_once(a, w, keep, parts=1):
    from speculators_amd import _lib

    m, f, k = a.shape[0], w.shape[0] // 2, a.shape[1]
    ws = torch.full((_lib.load().spx_gemm_tail_workspace_bytes() // 4,), float("nan"), device="cuda") if parts > 1 else None
    up = w[f:].clone()  # (the two weights need not lie behind one another)
    gu = torch.full((m + 1, 2 * f), 7.0, device="cuda", dtype=torch.bfloat16)
    out = torch.full((m + 1, f + 8), 7.0, device="cuda", dtype=torch.bfloat16)
    _lib.call("spx_gemm_bf16_gated", a, k, w, up, k, gu if keep else None, 2 * f, out, f + 8, m, f, k, parts, ws,
              0 if ws is None else ws.nbytes, _lib.stream_ptr(a.device))
    assert (out[m] == 7).all() and (out[:m, f:] == 7).all() and (gu[m] == 7).all()
    return out[:m, :f], gu[:m]


def test_extremes_of_the_gate():
    from speculators_amd import _lib

    f, k = 256, 192
    a = torch.zeros(8, k, device="cuda", dtype=torch.bfloat16)
    a[:, 0] = torch.tensor([0.0, 88.0, -87.5, -88.5, -120.0, 3e38, -3e38, float("nan")])
    w = torch.zeros(2 * f, k, device="cuda", dtype=torch.bfloat16)
    w[:, 0] = 1
    w[f:, 1] = 0
    _, want = _separately(a, w)
    got = torch.empty_like(want)
    _lib.call("spx_gemm_bf16_gated", a, k, w, w[f:], k, None, 2 * f, got, f, 8, f, k, 1, None, 0, _lib.stream_ptr(a.device))
    assert torch.equal(got.isnan(), want.isnan())
    assert ((got - want).double().abs() <= 2 ** -6 * want.double().abs() + 1e-36).logical_or(want.isnan() | (got == want)).all()


@pytest.mark.parametrize("keep", [False, True])
def test_every_value_of_a_gate(keep):
    """All 2^16 values that a gate can have, under three values beside each: the bits of the pass that divides.  (Gates below -87.3,
    where 1 / (1 + e^-x) is no normal number: to the last bit.)"""
    f, k = 1 << 16, 192
    w = torch.zeros(2 * f, k, device="cuda", dtype=torch.bfloat16)
    w[:f, 0] = torch.arange(f, device="cuda").to(torch.int16).view(torch.bfloat16)
    w[f:, 1:4] = torch.randn(f, 3, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3)).bfloat16()
    a = torch.zeros(3, k, device="cuda", dtype=torch.bfloat16)
    a[:, 0] = 1
    a[0, 1] = a[1, 2] = a[2, 3] = 1
    gu, want = _separately(a, w)
    whole = w[:f, 0].abs() >= 2 ** -126  # (what a product may flush to zero aside)
    assert torch.equal(gu[0, :f][whole], w[:f, 0][whole]) and gu[0, :f].isnan().sum() == w[:f, 0].isnan().sum()
    got, _ = _at_once(a, w, keep)
    same = (got == want) | (got.isnan() & want.isnan())
    low = gu[:, :f] < -87
    assert same[~low].all(), (~same & ~low).nonzero()
    assert (((got - want).abs() <= 2 ** -7 * want.abs()) | same)[low].all()


@pytest.mark.parametrize("m,f,k", [(1999, 8192, 2048), (512, 8192, 2048), (3001, 14336, 4096), (4096, 14336, 4096), (888, 8192, 2048)])
def test_what_is_taken(m, f, k):
    """Large tiles (512 rows run on smaller ones), with a workspace where the last round is cut."""
    from speculators_amd import gemm

    ws = gemm._gated("mixed", gemm.TAIL_PARTS, m, f, k)
    assert ws is None if m == 512 else (ws > 0) == (m == 3001)
    assert gemm._gated("hipblaslt", gemm.TAIL_PARTS, m, f, k) is None


# bf16: gate's and up's weights as they lie; autocast: their merged copy.  888 and 1999 rows have whole rounds, of 2560 the last one is cut
@pytest.mark.parametrize("seq,regime,train", [(888, "bf16", True), (888, "autocast", True), (1999, "bf16", False), (1999, "autocast", False),
                                              (2560, "bf16", True), (2560, "autocast", True)])
def test_a_draft_with_it_and_without(seq, regime, train, monkeypatch):
    """Loss, tokens, metrics and every gradient of a draft whose layers form the activation in the product, against the product by its
    own route and the pass: the same bits, but where sums of a cut round are added elsewhere (bf16 activations: 1e-2)."""
    from perf import cases
    from speculators_amd import gemm

    case = {"kind": "eagle3", "shape": "1b", "seq": seq, "steps": 2, "docs": 2, "window": 0, "regime": regime, "loss": "kl_div",
            "targets": "hidden", "train": train}
    state = cases.prepare(case, 3)
    asked, plain = [], gemm.gated
    monkeypatch.setattr(gemm, "gated", lambda m, staged, pair: asked.append((plain(m, staged, pair), pair)) or asked[-1][0])
    got = cases.run(state)
    assert len(asked) == 2 and all(ws is not None and (ws > 0) == (seq == 2560) for ws, _ in asked)
    assert all((pair is not None) == (regime == "bf16") for _, pair in asked)
    monkeypatch.setattr(gemm, "gated", lambda m, staged, pair: None)
    want = cases.run(state)
    pairs = [(got["loss"], want["loss"]), (got["metrics"], want["metrics"])]
    if train:
        assert got["grads"].keys() == want["grads"].keys() and len(want["grads"]) > 8
        pairs += [(got["grads"][n], want["grads"][n]) for n in want["grads"]]
    for a, b in pairs:
        assert bool(b.any())
        if seq == 2560:
            assert (a.double() - b.double()).norm() <= 1e-2 * b.double().norm()
        else:
            assert torch.equal(a, b)
    for a, b in zip(got["steps"], want["steps"], strict=True):
        assert (a != b).double().mean() <= (2e-3 if seq == 2560 else 0)
