"""Two sets of heads (queries; keys with the values) normed and rotated in one launch, against a launch each."""

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


class _Set(ctypes.Structure):  # spx_head_norm
    _fields_ = [("tok", ctypes.c_void_p), ("ld_tok", ctypes.c_int64), ("out", ctypes.c_void_p), ("out_hs", ctypes.c_int64),
                ("passed", ctypes.c_void_p), ("pass_hs", ctypes.c_int64), ("pos", ctypes.c_void_p), ("gain", ctypes.c_void_p),
                ("rstd", ctypes.c_void_p), ("T", ctypes.c_int64), ("n_heads", ctypes.c_int32), ("n_pass", ctypes.c_int32),
                ("eps", ctypes.c_float), ("accumulate", ctypes.c_int32), ("dtok", ctypes.c_void_p), ("ld_dtok", ctypes.c_int64),
                ("dw", ctypes.c_void_p)]


def _data(t, heads, n_pass, d, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    return {"tok": r(t, (heads + n_pass) * d), "out": r(heads, t, d), "passed": r(max(n_pass, 1), t, d), "gain": r(d),
            "pos": torch.randint(0, 5000, (t,), device="cuda", generator=g), "rstd": torch.empty(t, heads, device="cuda"),
            "dtok": torch.empty(t, (heads + n_pass) * d, device="cuda", dtype=torch.bfloat16), "shape": (t, heads, n_pass, d)}


def _set(x, dw=None, accumulate=0):
    t, heads, n_pass, d = x["shape"]
    p = lambda k: x[k].data_ptr()  # noqa: E731
    return _Set(p("tok"), x["tok"].stride(0), p("out"), t * d, p("passed") if n_pass else None, t * d, p("pos"), p("gain"),
                p("rstd"), t, heads, n_pass, 1e-6, accumulate, p("dtok"), x["dtok"].stride(0), dw.data_ptr() if dw is not None else None)


# one token, ragged last workgroups, both sides of the sizes from which a thread takes two and four heads
@pytest.mark.parametrize("tq,tk,hq,hkv", [(1, 1, 2, 1), (65, 129, 8, 2), (700, 1400, 32, 8), (3000, 6000, 32, 8)])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_two_sets_in_one_launch(tq, tk, hq, hkv, d):
    from speculators_amd import _lib

    freq = torch.rand(d // 2, device="cuda")
    st = _lib.stream_ptr(freq.device)
    q, k = _data(tq, hq, 0, d, 1), _data(tk, hkv, hkv, d, 2)
    want = []
    for x in (q, k):
        one = (_Set * 1)(_set(x))
        _lib.call("spx_head_norm_rope_sets", ctypes.addressof(one), 1, freq, d, 0, 1.25, st)
        want.append([x[n].clone() for n in ("out", "passed", "rstd")])
        x["out"].zero_(), x["rstd"].zero_()
    k["passed"].zero_()
    both = (_Set * 2)(_set(q), _set(k))
    _lib.call("spx_head_norm_rope_sets", ctypes.addressof(both), 2, freq, d, 0, 1.25, st)
    for x, w in zip((q, k), want, strict=True):
        assert all(torch.equal(x[n], v) for n, v in zip(("out", "passed", "rstd"), w, strict=True))
    # and back: out and passed serve as the gradients
    lib = _lib.load()
    slots = [int(lib.spx_rmsnorm_bwd_slots(t * h, d)) for t, h in ((tq, hq), (tk, hkv))]
    start = [torch.randn(n, d, device="cuda") for n in slots]
    want = []
    for x, w in zip((q, k), start, strict=True):
        dw = w.clone()
        one = (_Set * 1)(_set(x, dw, 1))
        _lib.call("spx_head_norm_rope_bwd_sets", ctypes.addressof(one), 1, freq, d, 0, 1.25, st)
        want.append((x["dtok"].clone(), dw))
        x["dtok"].zero_()
    got = [w.clone() for w in start]
    both = (_Set * 2)(_set(q, got[0], 1), _set(k, got[1], 1))
    _lib.call("spx_head_norm_rope_bwd_sets", ctypes.addressof(both), 2, freq, d, 0, 1.25, st)
    for x, g, (dtok, dw), n in zip((q, k), got, want, slots, strict=True):
        assert torch.equal(x["dtok"], dtok)
        # (which heads a thread takes, and so which partial sum a row is in, depends on the launch: the sums agree to the
        # order of some hundred thousand fp32 terms)
        scale = dw.double().abs().sum(0)
        assert ((g.double().sum(0) - dw.double().sum(0)).abs() <= 1e-5 * scale + 1e-6).all()


def test_refused():
    from speculators_amd import _lib

    freq = torch.rand(32, device="cuda")
    x = _data(4, 2, 0, 64, 1)
    st = _lib.stream_ptr(freq.device)
    for count in (0, 3):
        sets = (_Set * 3)(_set(x), _set(x), _set(x))
        with pytest.raises(_lib.SpxError):
            _lib.call("spx_head_norm_rope_sets", ctypes.addressof(sets), count, freq, 64, 0, 1.0, st)
    bad = (_Set * 2)(_set(x), _set(x))
    bad[1].rstd = None
    with pytest.raises(_lib.SpxError):
        _lib.call("spx_head_norm_rope_sets", ctypes.addressof(bad), 2, freq, 64, 0, 1.0, st)
