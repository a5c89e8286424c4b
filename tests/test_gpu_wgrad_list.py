"""Weight gradients of several products in one launch (spx_gemm_bf16_tn_list), and the node that stages a layer's weights together."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

LISTS = {
    "one tile of three slabs, the last of a row": [(129, 256, 256)],
    "ragged results, contractions that end inside a slab": [(200, 264, 520), (1000, 1032, 256), (130, 256, 1000)],
    "a last round in parts": [(4100, 512, 768)],
    "whole rounds, then one in parts of unlike contractions": [(2112, 4096, 4096), (2049, 264, 2048), (2304, 520, 256)],
    "a long tile first and a short last round": [(2665, 512, 512), (300, 4096, 4096), (200, 1032, 512)],
    "eight": [(130 + 64 * i, 256 + 8 * i, 520) for i in range(8)]}


def _operands(shapes, pad=0):
    g = torch.Generator(device="cuda").manual_seed(len(shapes))
    new = lambda t, n: torch.randn(t, n + pad, device="cuda", generator=g).bfloat16()[:, :n]  # noqa: E731
    return [(new(t, m), new(t, n)) for t, m, n in shapes]


@pytest.mark.parametrize("name", LISTS)
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("pad", [0, 8])
def test_list_against_float64(name, fp32, pad):
    """fp32 sums of t products, and one rounding to bf16; rows and columns beside a result are left alone."""
    from speculators_amd.gemm import _tn_list

    shapes = LISTS[name]
    pairs = _operands(shapes, pad)
    wide = [torch.full((m + 1, n + 8), 3.0, device="cuda", dtype=torch.float32 if fp32 else torch.bfloat16) for _, m, n in shapes]
    outs = [w[:m, :n] for w, (_, m, n) in zip(wide, shapes)]
    for _ in range(2):
        _tn_list(pairs, fp32, outs)
        for (a, b), out, w, (t, m, n) in zip(pairs, outs, wide, shapes):
            want = a.double().t() @ b.double()
            tol = (2e-6 * t ** 0.5 if fp32 else 2 ** -8) * want.abs().max().item() + 1e-4
            assert (out.double() - want).abs().max().item() <= tol
            assert (w[m:] == 3).all() and (w[:, n:] == 3).all()


def test_the_plan_cuts_where_the_tests_say_so():
    from speculators_amd.gemm import _tn_list_plan

    cut = {name: _tn_list_plan(tuple((*s, s[1], s[2], s[2]) for s in shapes), True)[1] > 0 for name, shapes in LISTS.items()}
    assert [name for name, is_cut in cut.items() if is_cut] == [name for name in LISTS if "in parts" in name]


@pytest.mark.parametrize("name", LISTS)
@pytest.mark.parametrize("fp32", [False, True])
def test_rows_of_whole_lines_and_others(name, fp32):
    """Results whose rows begin with lines of 128 bytes are stored past the caches, others through them: the same bits."""
    from speculators_amd.gemm import _tn_list

    pairs, dtype = _operands(LISTS[name]), torch.float32 if fp32 else torch.bfloat16
    got = []
    for beside, offset in ((8, 0), (8, 8), (0, 0)):
        lds = [-(-n // 64) * 64 + beside for _, _, n in LISTS[name]]
        wide = [torch.full((m * ld + 64,), 3.0, device="cuda", dtype=dtype) for (_, m, _), ld in zip(LISTS[name], lds)]
        outs = [w[offset:offset + m * ld].view(m, ld)[:, :n] for w, (_, m, n), ld in zip(wide, LISTS[name], lds)]
        assert any(out.data_ptr() % 128 or out.stride(0) * out.element_size() % 128 for out in outs) == (beside > 0)
        _tn_list(pairs, fp32, outs)
        assert all((w[offset + m * ld:] == 3).all() and (w[:offset] == 3).all() for w, (_, m, _), ld in zip(wide, LISTS[name], lds))
        got.append(outs)
    assert all(torch.equal(a, b) for others in got[1:] for a, b in zip(got[0], others))


@pytest.mark.parametrize("dtype,stride", [(torch.float32, 65544), (torch.float32, 1 << 21), (torch.bfloat16, 1 << 22)])
def test_results_in_rows_far_apart(dtype, stride):
    """A tile's 256 rows of the result span 2 GiB: not on the walking kernel, which offsets them in 32 bits, but as before it."""
    from speculators_amd.gemm import _tn_shape, _walks, gemm_tn

    (a, b), = _operands([(300, 8, 65528)], 256)
    out = torch.full((8 * stride,), 3.0, device="cuda", dtype=dtype).view(8, stride)[:, :65528]
    fp32 = dtype == torch.float32
    assert _walks(_tn_shape(a, b, None), fp32) and _walks(_tn_shape(a, b, out), fp32) == (stride == 65544)
    assert gemm_tn(a, b, out) is out
    want = a.double().t() @ b.double()
    tol = (2e-6 * 300 ** 0.5 if fp32 else 2 ** -8) * want.abs().max().item() + 1e-4
    assert (out.double() - want).abs().max().item() <= tol
    assert (torch.as_strided(out, (8, stride - 65528), (stride, 1), 65528) == 3).all()


@pytest.mark.parametrize("t,m,n,fp32,walks", [
    (1280, 3840, 5376, False, False), (1193, 768, 25088, False, False), (466, 5376, 3648, False, False),  # 1.18 - 1.23 of the smaller tiles
    (192, 5784, 29112, True, False), (384, 16688, 1816, False, False),  # 1.05
    (192, 11776, 9192, False, True), (2339, 14448, 3368, False, True), (697, 3520, 7608, True, True)])  # 0.82, 0.92, 0.71
def test_which_weight_gradients_walk(t, m, n, fp32, walks):
    from speculators_amd.gemm import _walks

    assert _walks((t, m, n, m, n, n), fp32) == walks


def test_rules():
    from speculators_amd import _lib, gemm

    x = torch.zeros(512, 512, dtype=torch.bfloat16, device="cuda")
    c = torch.zeros(512, 520, device="cuda")
    good = dict(a=x.data_ptr(), lda=512, b=x.data_ptr(), ldb=512, c=c.data_ptr(), ldc=520, M=512, N=512, T=512)
    lib, st = _lib.load(), ctypes.c_void_p(_lib.stream_ptr(x.device))

    def rc(n=1, **changes):
        items = (gemm._TnProduct * 9)(*[gemm._TnProduct(**{**good, **changes})] * 9)
        return lib.spx_gemm_bf16_tn_list(items, n, 1, None, 0, st)

    assert rc() == 0
    for changes in ({"T": 128}, {"T": 0}, {"lda": 248, "M": 248}, {"ldb": 516}, {"M": 516}, {"ldc": 504}, {"ldc": 516}, {"a": None},
                    {"c": c.data_ptr() + 4}, {"n": 0}, {"n": 9}):
        assert rc(**changes) != 0, changes


class _Into(torch.autograd.Function):
    """``x`` in a weight's input buffer."""

    @staticmethod
    def forward(ctx, x, slot):
        slot.data.copy_(x)  # (as a kernel writes it: the buffer of another use is not "modified")
        return slot

    @staticmethod
    def backward(ctx, g):
        return g, None


# one use; two of them in the weights' input buffers: one product a weight either way, and these are one launch for each type of result
# that several weights have; two uses outside the buffers: a product each, added up
@pytest.mark.parametrize("regime,lists", [("bf16", {False: 3}), ("autocast", {True: 3}), ("mixed", {False: 2})])
@pytest.mark.parametrize("uses,slots", [(1, False), (2, True), (2, False)])
def test_a_layer_staged_together(regime, lists, uses, slots, monkeypatch):
    """The gradients of weights that are staged by one node are those of a node each (the products' sums are the same up to the
    order of fp32 additions), whichever of them are asked for; nothing is kept alive once the graph is gone."""
    import gc

    from speculators_amd import gemm
    from speculators_amd.gemm import linear_staged
    from speculators_amd.weights import WeightStager

    torch.manual_seed(1)
    dt = torch.float32 if regime == "autocast" else torch.bfloat16
    new = lambda n, k, d=dt: torch.nn.Parameter((torch.randn(n, k, device="cuda") * k ** -0.5).to(d))  # noqa: E731
    q, k, o, up = new(1536, 1536, torch.float32 if regime == "mixed" else dt), new(768, 1536), new(1536, 2304), new(3072, 1536)
    x = torch.randn(600, 1536, device="cuda").bfloat16()
    launches = []
    plain = gemm._tn_list
    monkeypatch.setattr(gemm, "_tn_list", lambda pairs, fp32, outs: launches.append((fp32, len(pairs))) or plain(pairs, fp32, outs))

    def product(h, w):
        return linear_staged(_Into.apply(h, w.x_slot(600)) if slots else h, w)

    def loss(together):
        stager = WeightStager()
        stager.begin(uses=uses)
        with torch.autocast("cuda", torch.bfloat16, enabled=regime != "bf16"):
            if together:
                wqk, wo, wup = stager.get_all((q, k), (o,), (up,))
            else:
                wqk, wo, wup = stager.get(q, k), stager.get(o), stager.get(up)
            h = x
            for _ in range(uses):
                h = product(product(product(h, wqk), wo), wup)[:, :1536].contiguous()
        return h.float().square().mean()

    monkeypatch.setattr(torch.backends.cuda.matmul, "allow_bf16_reduced_precision_reduction", False)
    params = (q, k, o, up)
    want = torch.autograd.grad(loss(False), params)
    assert not any(n > 1 for _, n in launches)
    gc.collect()
    gc.disable()
    try:
        before = torch.cuda.memory_allocated()
        for _ in range(3):
            launches.clear()
            got = torch.autograd.grad(loss(True), params)
            assert {fp32: n for fp32, n in launches if n > 1} == ({} if uses == 2 and not slots else lists)
            assert sum(n > 1 for _, n in launches) == (uses == 1 or slots)
            for a, b, p in zip(got, want, params, strict=True):
                assert a.dtype == p.dtype and (a - b).norm() <= 2 ** -8 * b.norm()
            del got, a
        assert torch.cuda.memory_allocated() == before
        for i, p in enumerate(params):
            launches.clear()
            part, = torch.autograd.grad(loss(True), (p,))
            assert (part - want[i]).norm() <= 2 ** -8 * want[i].norm()
            assert not any(n > 1 for _, n in launches)  # (its own product alone)
    finally:
        gc.enable()
