"""Products against the weights of two projections as they lie: the same bits as against their concatenation."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pair(form, a, b, b2, parts):
    from speculators_amd import _lib, gemm

    m, k = a.shape
    n = b.shape[1] if form else 2 * b.shape[0]
    out = torch.empty(m, n, device=a.device, dtype=torch.bfloat16)
    nbytes = max(int(_lib.load().spx_gemm_auto_workspace_bytes(form, m, n, k, parts)), 256)
    ws = torch.empty(nbytes, device=a.device, dtype=torch.uint8)
    _lib.call("spx_gemm_bf16_pair", form, a, a.stride(0), b, b2, b.stride(0), out, n, m, n, k, parts, ws, nbytes, None,
              _lib.stream_ptr(a.device))
    return out


# whole rounds, a cut last round, a ragged last tile row; of the second form: the turn in the middle of a tile's contraction and between
# the parts of one that is cut whole, in the first slabs and with a ragged row of tiles
@pytest.mark.parametrize("form,m,n,k,parts", [(0, 888, 16384, 192, 4), (0, 4096, 16384, 2048, 4), (0, 1999, 10240, 4096, 4),
                                              (0, 4096, 16384, 2048, 1), (1, 4096, 8192, 384, 4), (1, 4001, 8192, 2176, 4),
                                              (1, 888, 2048, 16384, 4), (1, 1300, 2048, 16512, 4)])
def test_same_bits_as_the_concatenation(form, m, n, k, parts):
    from speculators_amd import _lib, gemm

    assert _lib.load().spx_gemm_pair_takes(form, m, n, k, n if form else k, parts)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randn(m, k, device="cuda", generator=g).bfloat16()
    rows = (k if form else n) // 2
    b, b2 = (torch.randn(rows, n if form else k, device="cuda", generator=g).bfloat16() for _ in range(2))
    whole = torch.cat([b, b2])
    out = torch.empty(m, n, device="cuda", dtype=torch.bfloat16)
    nbytes = max(int(_lib.load().spx_gemm_auto_workspace_bytes(form, m, n, k, parts)), 256)
    ws = torch.empty(nbytes, device="cuda", dtype=torch.uint8)
    _lib.call("spx_gemm_bf16_auto", form, a, k, whole, whole.stride(0), out, n, m, n, k, None, parts, ws, nbytes,
              _lib.stream_ptr(a.device))
    assert torch.equal(_pair(form, a, b, b2, parts), out)


@pytest.mark.parametrize("form,m,n,k", [(0, 888, 16384 + 256, 2048), (0, 64, 16384, 2048), (1, 888, 2048, 16384 + 64), (1, 64, 2048, 16384), (1, 4096, 8192, 256)])
def test_sizes_that_are_refused(form, m, n, k):
    from speculators_amd import _lib

    assert not _lib.load().spx_gemm_pair_takes(form, m, n, k, n if form else k, 4)
    a = torch.zeros(m, k, device="cuda", dtype=torch.bfloat16)
    b = torch.zeros((k if form else n) // 2, n if form else k, device="cuda", dtype=torch.bfloat16)
    with pytest.raises(_lib.SpxError):
        _pair(form, a, b, b, 4)


@pytest.mark.parametrize("train", [False, True])
def test_a_bf16_layer(train, monkeypatch):
    """A draft whose gate and up weights are read as they lie gives the bits it gives with their concatenation, and a weight that
    changes between forward and backward raises."""
    from speculators_amd import gemm
    from perf import cases

    case = next(c for c in cases.listed() if c["name"] == ("dflash-1b-1777" if train else "eagle3-1b-validate-1999"))
    state = cases.prepare(case, 1)
    taken = []
    plain = gemm.pair_routes
    monkeypatch.setattr(gemm, "pair_routes", lambda m, s: taken.append(plain(m, s)) or taken[-1])
    got = cases.run(state)
    assert taken and all(t is not None for t in taken)
    monkeypatch.setattr(gemm, "pair_routes", lambda m, s: None)
    want = cases.run(state)
    assert torch.equal(got["loss"], want["loss"])
    if train:
        assert all(torch.equal(got["grads"][n], want["grads"][n]) for n in want["grads"])
        monkeypatch.setattr(gemm, "pair_routes", plain)
        model = state["model"]
        _, loss, _ = model(**state["batch"], **state["kw"])
        with torch.no_grad():
            next(p for n, p in model.named_parameters() if "gate_proj" in n).mul_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            loss.backward()
