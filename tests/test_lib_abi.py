"""The C-ABI library loads on a machine without a GPU and exports every symbol
that include/spx.h declares (no compute calls here)."""

import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared_symbols():
    text = open(os.path.join(ROOT, "include", "spx.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(spx_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_entry_points():
    names = _declared_symbols()
    assert "spx_fused_vocab_loss_fwd" in names and "spx_version" in names


def test_library_exports_every_declared_symbol():
    from speculators_amd import _lib

    if not os.path.exists(_lib.LIB_PATH):
        pytest.fail("libspx_hip.so is not built; run __graft_entry__.build()")
    lib = _lib.load()
    assert lib.spx_version() >= 100
    for name in _declared_symbols():
        assert hasattr(lib, name), name
    # every bound signature is declared in the header and vice versa
    assert set(_lib.SIGNATURES) | {"spx_version", "spx_last_error"} == set(_declared_symbols())


def test_binding_module_has_every_entry_point():
    import torch

    from speculators_amd import _lib

    native = _lib.native()
    for name in _declared_symbols():
        assert hasattr(native, name), name
    with pytest.raises(_lib.SpxError, match="unknown loss op"):
        _lib.call("spx_fused_vocab_loss_fwd", 99, None, 0, None, 0, 1, 8, 0, None, None, None, None, None, None, 0,
                  None)
    with pytest.raises(_lib.SpxError, match="CPU tensor"):
        native.spx_rmsnorm_dweight(torch.zeros(8), 1, None, 8, None)
    with pytest.raises(TypeError):
        native.spx_rmsnorm_bwd_slots(1)
    assert native.spx_rmsnorm_bwd_slots(4096, 2048) == _lib.load().spx_rmsnorm_bwd_slots(4096, 2048)


def test_argument_errors_do_not_need_a_gpu():
    from speculators_amd import _lib

    lib = _lib.load()
    rc = lib.spx_fused_vocab_loss_fwd(99, None, 0, None, 0, 1, 8, 0, None, None, None, None, None,
                                      None, 0, None)
    assert rc == 1 and b"unknown loss op" in lib.spx_last_error()
    rc = lib.spx_fused_vocab_loss_fwd(0, None, 4, None, 4, 1, 8, 0, None, None, None, None, None,
                                      None, 0, None)
    assert rc == 1 and b"stride" in lib.spx_last_error()


def test_host_tensors_are_refused():
    import torch

    from speculators_amd import _lib, losses

    with pytest.raises(_lib.SpxError):
        losses.kl_div_loss(torch.randn(1, 2, 8), torch.randn(1, 2, 8))


def test_resolve_loss_config_mirrors_reference_errors():
    from speculators_amd import losses as L

    assert L.resolve_loss_config("kl_div")["kl_div"] == (L.kl_div_loss, 1.0)
    cfg = L.resolve_loss_config('{"ce": 0.1, "tv": 0.9}')
    assert cfg["ce"] == (L.ce_loss, 0.1) and cfg["tv"] == (L.tv_loss, 0.9)
    for name in ("kl_div", "rkl", "jsd", "ce", "tv", "nla", "lk_hybrid"):
        assert name in L.resolve_loss_config(name)
    with pytest.raises(ValueError, match="Unknown loss implementation"):
        L.resolve_loss_config("kl_div", "triton")
    with pytest.raises(ValueError, match="Unknown loss function"):
        L.resolve_loss_config("nope")
    with pytest.raises(ValueError, match="non-empty JSON dict"):
        L.resolve_loss_config("[]")
    with pytest.raises(ValueError, match="Unknown loss function 'zz'"):
        L.resolve_loss_config('{"zz": 1}')
    with pytest.raises(ValueError, match="must be a number"):
        L.resolve_loss_config('{"ce": "x"}')


def test_entry_points_run_without_the_interpreter_lock():
    """A call into the library lets other Python threads run (a launch may wait for queue space): with forced switches
    out of the picture a second thread gets its turn only where a call gives the lock up."""
    import sys
    import threading

    from speculators_amd import _lib

    native = _lib.native()
    gate, ran, attempts = threading.Lock(), [], 0
    gate.acquire()

    def other():
        with gate:
            ran.append(True)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    thread.start()
    try:
        sys.setswitchinterval(1000.0)
        gate.release()  # the other thread waits for the interpreter's lock from here on
        while not ran and attempts < 200000:
            attempts += 1
            try:  # (refused for its arguments: needs no GPU)
                native.spx_rmsnorm_dweight(None, 0, 0, None, None)
            except _lib.SpxError:
                pass
        got = bool(ran)
    finally:
        sys.setswitchinterval(interval)
    thread.join()
    assert got


def test_product_workspaces_belong_to_one_thread():
    """Two threads on one stream may interleave the launches of their products: each has a buffer of its own, kept while
    the thread lives."""
    import threading
    import weakref

    import torch

    from speculators_amd import gemm

    cpu = torch.device("cpu")
    mine = gemm._split_workspace(cpu, 64)
    assert gemm._split_workspace(cpu, 32) is mine
    other = []

    def work():
        ws = gemm._split_workspace(cpu, 64)
        assert ws is gemm._split_workspace(cpu, 64)
        other.append((ws.data_ptr() != mine.data_ptr(), weakref.ref(ws)))

    thread = threading.Thread(target=work)
    thread.start()
    thread.join()
    assert other[0][0] and other[0][1]() is None
    assert gemm._split_workspace(cpu, 64) is mine


@pytest.mark.parametrize("workspace,room", [(None, 1 << 30), (4100, 1 << 30), (4096, 1 << 20)])
def test_a_pair_product_cut_whole_needs_its_workspace(workspace, room):
    """Without one its size has another choice, whose kernels know no second half of the weight: refused before any launch."""
    from speculators_amd import _lib

    lib = _lib.load()
    m, n, k = 888, 2048, 16384
    assert lib.spx_gemm_pair_takes(1, m, n, k, n, 4) and lib.spx_gemm_auto_workspace_bytes(1, m, n, k, 4) > 1 << 20
    rc = lib.spx_gemm_bf16_pair(1, 4096, k, 4096, 4096, n, 4096, n, m, n, k, 4, workspace, room, None, None)
    assert rc == 1 and b"workspace" in lib.spx_last_error()


@pytest.mark.parametrize("rows,taken", [(128, False), (129, True), ((1 << 28) - 576, True), ((1 << 28) - 575, False), (1 << 28, False)])
def test_contractions_that_workgroups_walk(rows, taken):
    """Three slabs at least, and with eight parts fewer than 2^22: the kernel divides their number by a reciprocal good to there."""
    from speculators_amd import gemm

    assert (gemm._tn_list_plan(((rows, 4096, 4096, 4096, 4096, 4096),), True)[0] > 0) == taken
