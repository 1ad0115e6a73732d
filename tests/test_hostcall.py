"""The kept launchers of eager calls (hostcall), without a GPU: stub launchers
stand in for the compiled ones, CPU tensors for the device's."""

import contextlib
import copy
import pickle
import weakref

import numpy as np
import pytest
import torch

from ssalaad_amd import LRSLinearGroup, _lib, _runtime, addmm_inplace, ls_linear


class Stub:
    """A launcher that counts its calls and returns a given status."""

    def __init__(self, rc=0):
        self.rc, self.calls = rc, 0

    def launch(self, *args):
        self.calls += 1
        return self.rc


@pytest.fixture(autouse=True)
def no_device(monkeypatch):
    """The device queries of the call path, answered as for CPU tensors."""
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: None)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 0)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)


def kept_op_call(stub, nb=2, p=16):
    """Arguments of an op call whose launcher is kept."""
    crow = torch.arange(nb + 1, dtype=torch.int32)
    col = torch.zeros(nb, dtype=torch.int32)
    act = torch.arange(nb, dtype=torch.int32)
    vals = torch.zeros(nb, p, p)
    out, x = torch.zeros(3, nb * p), torch.zeros(3, p)
    sp = addmm_inplace._StructPlan(addmm_inplace._versions(crow, col, act, nb, 1), col, act, 1)
    sp.calls[(out.shape, x.shape, vals.shape, vals.dtype, 0)] = (_runtime.generation(), stub)
    setattr(crow, addmm_inplace._PLAN_ATTR, sp)
    return out, x, crow, col, vals, act


def kept_linear(stub, n=64, m=64, tokens=3):
    """A low-rank linear whose launcher for `tokens` rows is kept."""
    mod = ls_linear._LRSLinearLR(torch.randn(n, 16), torch.randn(16, m), in_features=m,
                                 out_features=n)
    st = mod._state = ls_linear._KernelState(mod, torch.device("cpu"))
    st._launchers[(tokens, 0, id(st))] = (_runtime.generation(), None, stub, (st,), (n,))
    return mod, torch.randn(tokens, m)


def kept_group(stub, n=64, m=64, tokens=3):
    mods = [kept_linear(None, n, m)[0] for _ in range(2)]
    sts = [mod._state for mod in mods]
    sts[0]._launchers[(tokens, 0, *map(id, sts))] = (_runtime.generation(), None, stub, tuple(sts),
                                                     (n, n))
    return LRSLinearGroup(*mods), torch.randn(tokens, m)


# Argument errors are found before any launch; a HIP error is read after it.
REFUSED = [-1, _lib.SSL_ERR_INVALID, _lib.SSL_ERR_UNSUPPORTED, _lib.SSL_ERR_WORKSPACE]


def test_op_call_with_a_hip_error_is_not_issued_again():
    """The kernel may be on the stream already (a stale error of the thread is
    reported too), and a second one would add x·Sᵀ twice."""
    stub = Stub(_lib.SSL_ERR_HIP)
    with pytest.raises(RuntimeError, match="ssl_bsr_addmm_inplace"):
        addmm_inplace._repeat(*kept_op_call(stub))
    assert stub.calls == 1


@pytest.mark.parametrize("rc", REFUSED)
def test_refused_op_call_takes_the_full_path(rc):
    stub = Stub(rc)
    assert addmm_inplace._repeat(*kept_op_call(stub)) is False
    assert stub.calls == 1
    stub = Stub(0)
    assert addmm_inplace._repeat(*kept_op_call(stub)) is True


@pytest.mark.parametrize("make", [kept_linear, kept_group])
def test_module_call_with_a_hip_error_raises(make, monkeypatch):
    stub = Stub(_lib.SSL_ERR_HIP)
    mod, x = make(stub)
    monkeypatch.setattr(ls_linear, "_launch", lambda *a: pytest.fail("issued again"))
    with pytest.raises(RuntimeError, match="ssl_slr_forward_group"):
        mod(x)
    assert stub.calls == 1


@pytest.mark.parametrize("make", [kept_linear, kept_group])
@pytest.mark.parametrize("rc", [0] + REFUSED)
def test_module_call_uses_the_kept_launcher_or_the_full_path(make, rc, monkeypatch):
    stub = Stub(rc)
    mod, x = make(stub)
    full = []
    monkeypatch.setattr(ls_linear, "_launch", lambda *a: full.append(1) or [x])
    monkeypatch.setattr(ls_linear._KernelState, "forward", lambda *a: full.append(1) or x)
    mod(x)
    assert stub.calls == 1 and len(full) == (0 if rc == 0 else 1)


def test_new_status_word_drops_the_launchers_made_without_it(monkeypatch):
    monkeypatch.setattr(_runtime, "_STATUS", {})
    monkeypatch.setattr(_runtime, "StatusWord", lambda: type("W", (), dict(host_ptr=64))())
    monkeypatch.setattr(torch.cuda, "device", lambda i: contextlib.nullcontext())
    dev = torch.device("cuda", 0)
    assert _runtime.status_address(dev) == 0
    stub = Stub()
    args = kept_op_call(stub)
    _runtime.status_word(dev)
    assert _runtime.status_address(dev) == 64
    assert addmm_inplace._repeat(*args) is False and stub.calls == 0


@pytest.mark.parametrize("member", [0, 1])
def test_reinterpreted_weights_are_refused_as_on_the_full_path(member, monkeypatch):
    """A view of A in another dtype keeps A's pointer and version."""
    stub = Stub()
    grp, x = kept_group(stub)
    monkeypatch.setattr(ls_linear, "_launch", lambda *a: pytest.fail("checks passed"))
    mod = grp.members[member]
    mod._kernel = lambda: pytest.fail("checks passed") if member == 0 else _lib.dtype_code(mod.A.dtype)
    mod.A = mod.A.view(torch.int32)
    with pytest.raises(TypeError):
        grp(x)
    assert stub.calls == 0

    mod, x = kept_linear(stub)
    mod.A = mod.A.view(torch.int32)
    with pytest.raises(TypeError, match="input dtype"):
        mod(x)
    assert stub.calls == 0


def test_modules_with_a_kernel_view_can_be_copied():
    """A copy has the same buffers and no kernel view of its own yet."""
    mod, _ = kept_linear(Stub())
    for twin in (copy.deepcopy(mod), pickle.loads(pickle.dumps(mod))):
        assert twin._state is None and mod._state is not None
        assert torch.equal(twin.A, mod.A) and twin.A.data_ptr() != mod.A.data_ptr()
    grp, _ = kept_group(Stub())
    assert [m._state for m in copy.deepcopy(grp).members] == [None, None]


def test_generation_counts_replaced_buffers_only(monkeypatch):
    """A first buffer of another stream, plan or device drops no launcher; a
    replaced one does, once the new one is in place."""
    cpu = torch.device("cpu")
    seen = []
    monkeypatch.setattr(_runtime, "_RETIRED", [])
    pool = {}
    real = _runtime._replaced
    monkeypatch.setattr(_runtime, "_replaced", lambda: (seen.append(pool[0].numel()), real()))
    before = _runtime.generation()
    small = _runtime._grown(pool, 0, 10, torch.int32, cpu, 16)
    assert small.numel() == 16 and _runtime.generation() == before
    assert _runtime._grown(pool, 0, 12, torch.int32, cpu, 16) is small
    assert _runtime._grown(pool, 0, 17, torch.int32, cpu, 16).numel() == 32
    assert seen == [32] and _runtime.generation() == before + 1 and _runtime._RETIRED == [small]

    plan = _runtime.DevicePlan(np.zeros((1, 8), np.int32), 1, 0, cpu)
    seen.clear()
    area = plan.exchange(512)
    assert not seen and plan.exchange(300) is area
    assert plan.exchange(1024) is not area and len(seen) == 1 and plan._retired == [area]


@pytest.mark.parametrize("which", [2, 3, 5], ids=["crow", "col", "active"])
def test_replaced_structure_takes_the_full_path(which):
    """A structure tensor given other data keeps its identity and version; the
    full path checks the new structure (a crow of other length is refused there)."""
    stub = Stub()
    args = kept_op_call(stub)
    assert addmm_inplace._repeat(*args) is True
    args[which].data = torch.cat([args[which], args[which][-1:]])
    assert addmm_inplace._repeat(*args) is False and stub.calls == 1
    stub = Stub()
    args = kept_op_call(stub)
    args[which].add_(0)
    assert addmm_inplace._repeat(*args) is False and stub.calls == 0


def test_watch_keeps_what_it_reads():
    """A buffer's own methods may drop it from the dict that is being watched."""

    class Buffer:
        _version = 3

        def __init__(self, buffers):
            self.buffers = buffers

        def data_ptr(self):
            self.buffers.pop("a", None)
            self.buffers["c"] = None
            return 64

    buffers = {}
    buffers["a"], buffers["b"] = Buffer(buffers), Buffer(buffers)
    last = weakref.ref(buffers["a"])
    watch = _lib.hostcall().Watch(buffers)
    assert last() is None and not watch.unchanged(buffers)
    assert _lib.hostcall().Watch({"b": buffers["b"]}).unchanged({"b": buffers["b"]})
    with pytest.raises(AttributeError):
        _lib.hostcall().Watch({"a": 1})


def test_op_builds_a_launcher_for_repeated_calls_only(monkeypatch):
    """A call's second time builds its launcher, a replaced buffer builds it
    anew, and more token counts in turn than are kept build none at all."""
    crow = torch.zeros(2, dtype=torch.int32)
    sp = addmm_inplace._StructPlan((), crow, crow, 1)
    most = addmm_inplace._MAX_CALLS
    assert not any(addmm_inplace._keeps(sp, (M,)) for M in range(most))
    assert all(addmm_inplace._keeps(sp, (M,)) for M in range(most))
    sp.calls[(1,)] = (_runtime.generation(), Stub())
    assert not addmm_inplace._keeps(sp, (1,))
    _runtime._replaced()
    assert addmm_inplace._keeps(sp, (1,))
    sp = addmm_inplace._StructPlan((), crow, crow, 1)
    assert not any(addmm_inplace._keeps(sp, (M,)) for M in list(range(most + 1)) * 3)


def test_op_calls_without_a_launcher_are_left_at_once():
    """Tiled token counts (no launcher is kept for them) and an x that is to be
    refused for its dimensions."""
    stub = Stub()
    out, x, *rest = kept_op_call(stub)
    assert addmm_inplace._repeat(out, x[0], *rest) is False
    assert addmm_inplace._repeat(out, x[0, 0], *rest) is False
    getattr(rest[0], addmm_inplace._PLAN_ATTR).tiled.add(3)
    assert addmm_inplace._repeat(out, x, *rest) is False and stub.calls == 0


def test_full_path_of_unchanged_weights_reads_the_buffers_once(monkeypatch):
    mod, x = kept_linear(Stub(_lib.SSL_ERR_INVALID))
    grp, gx = kept_group(Stub(_lib.SSL_ERR_INVALID))
    monkeypatch.setattr(ls_linear, "_launch", lambda states, x, outf: [x] * len(states))
    monkeypatch.setattr(ls_linear._LRSLinearBase, "_weights_key", lambda mod: pytest.fail("again"))
    assert mod(x) is x and grp(gx) == (gx, gx)
