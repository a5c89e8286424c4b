"""Several fp32 weights cast in one launch, against a cast each."""

import pytest
import torch

pytestmark = pytest.mark.gpu


# five to eight parts: parts of one chunk of eight, ends inside and at the edges of a workgroup's 8192 values, bf16 between
@pytest.mark.parametrize("sizes,dtypes", [((8, 8, 16, 8, 8), "fbfbf"), ((8192, 8192, 8184, 8, 16384, 24), "ffffff"),
                                          ((8200, 40960, 8, 8192, 100008, 8, 8, 65536), "fbffbfff"), ((1 << 20,) * 8, "ffffffff")])
def test_parts_of_one_launch(sizes, dtypes):
    from speculators_amd import _lib

    torch.manual_seed(len(sizes))
    parts = [torch.randn(n, device="cuda").to(torch.float32 if k == "f" else torch.bfloat16)
             for n, k in zip(sizes, dtypes, strict=True)]
    assert torch.equal(_lib.native().cat_bf16(*parts), torch.cat([p.bfloat16() for p in parts]))


# all fp32 and trained: one buffer; a bf16, frozen, strided or oddly sized weight among them: a copy each
@pytest.mark.parametrize("odd", ["", "bf16", "frozen", "strided", "size"])
def test_staged_weights_of_one_launch(odd):
    from speculators_amd.weights import WeightStager

    torch.manual_seed(3)
    new = lambda *s: torch.nn.Parameter(torch.randn(*s, device="cuda"))  # noqa: E731
    q, k, o, gate, up = new(64, 256), new(32, 256), new(128, 64), new(96, 128), new(96, 128)
    if odd == "bf16":
        o = torch.nn.Parameter(o.detach().bfloat16())
    elif odd == "frozen":
        o.requires_grad_(False)
    elif odd == "strided":
        o = torch.nn.Parameter(torch.randn(64, 128, device="cuda").t())
    elif odd == "size":
        o = new(9, 8)
    stager = WeightStager()
    stager.begin()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got = stager.get_all((q, k), None, (o,), (gate, up))
        again = stager.get_all((q, k), None, (o,), (gate, up))
    assert got[1] is None and all(a is b for a, b in zip(got, again, strict=True))
    qk, _, ow, gu = (s.w if s is not None else None for s in got)
    assert torch.equal(qk, torch.cat((q, k)).bfloat16()) and torch.equal(ow, o.bfloat16())
    assert torch.equal(gu, torch.cat((gate, up)).bfloat16())
    joint = qk.untyped_storage().data_ptr() == gu.untyped_storage().data_ptr()
    assert joint == (odd == "") and all(w.data_ptr() % 256 == 0 for w in (qk, gu))
