"""The kept launchers of eager calls (hostcall): a repeated call equals the first
one, and whatever differs from it — weights, shapes, strides, streams, a refused
status — takes the full path again with the full path's results and errors."""

import sys
from concurrent.futures import ThreadPoolExecutor

import pytest
import torch

from ssalaad_amd import LRSLinear, LRSLinearGroup, _lib, _runtime, addmm_inplace, clear_wait_status, prepare_bsr_addmm

pytestmark = pytest.mark.gpu


def _linear(seed, n=192, m=160, r=24, p=32, dtype=torch.bfloat16, bias=True):
    g = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *s: (torch.randn(*s, generator=g, device="cuda") * 0.1).to(dtype)  # noqa: E731
    nb, nbk = -(-n // p), -(-m // p)
    S = rnd(nb * p, nbk * p)
    S[n:], S[:, m:] = 0, 0
    keep = torch.rand(nb, 1, nbk, 1, generator=g, device="cuda") < 0.6
    S = (S.view(nb, p, nbk, p) * keep).view(nb * p, nbk * p)
    mod = LRSLinear(rnd(n, r), rnd(r, m), S.to_sparse_bsr((p, p)), in_features=m, out_features=n,
                    bias=rnd(n) if bias else None, block_p=p, block_q=p)
    return mod, S[:n, :m]


def _expect(mod, S, x):
    y = (x.double() @ mod.B.double().T) @ mod.A.double().T + x.double() @ S.double().T
    return y if mod.bias is None else y + mod.bias.double()


def _close(y, ref):
    # t and y are each rounded once to the 16-bit dtype (2^-9): at most 1e-2 of the largest value
    assert float((y.double() - ref).abs().max()) <= 1e-2 * float(ref.abs().max())


@pytest.mark.parametrize("n,m,tokens", [(192, 160, 1), (150, 160, 5), (192, 150, 16), (64, 32, 129),
                                        (192, 160, 200)])
def test_repeated_linear_calls(n, m, tokens, gpu_device):
    mod, S = _linear(0, n, m)
    x = torch.randn(tokens, m, device="cuda").to(torch.bfloat16)
    first = mod(x).clone()
    _close(first, _expect(mod, S, x))
    for _ in range(3):
        assert torch.equal(mod(x), first)
    x2 = torch.randn_like(x)
    _close(mod(x2), _expect(mod, S, x2))
    # leading dimensions, a row-strided x, an unaligned x
    assert torch.equal(mod(x.view(tokens, 1, m)), first.view(tokens, 1, n))
    if tokens == 1:
        assert mod(x[0]).shape == (n,) and torch.equal(mod(x[0]), first[0])
    wide = torch.empty(tokens, m + 24, device="cuda", dtype=x.dtype)
    wide[:, 3:m + 3] = x
    assert torch.equal(mod(wide[:, 3:m + 3]), first)
    assert mod(x[:0]).shape == (0, n)


class Counting:
    """A kept launcher that counts the calls issued through it."""

    def __init__(self, launcher):
        self.launcher, self.calls = launcher, 0

    def launch(self, *args):
        self.calls += 1
        return self.launcher.launch(*args)


def _live(kept, call):
    """Repeat `call` until its launcher is in the dict that `kept()` returns;
    then count what goes through it, one call among others."""
    for _ in range(4):
        call()
        if kept():
            break
    (key, entry), = list(kept().items())
    at, = [i for i, v in enumerate(entry) if type(v).__name__ in ("GroupCall", "OpCall")]
    counting = Counting(entry[at])
    kept()[key] = entry[:at] + (counting,) + entry[at + 1:]
    call()
    assert counting.calls == 1
    return counting


def _replace_b(mod):
    mod.B = mod.B * 3


def _new_bias_storage(mod):
    mod.bias.data = mod.bias * 0 + 1


def _drop_bias(mod):
    mod.bias = None


@pytest.mark.parametrize("change", [lambda mod: mod.A.mul_(2), _replace_b, _new_bias_storage,
                                    _drop_bias, lambda mod: mod.S_values.mul_(1)],
                         ids=["in-place", "replaced", "new-storage", "dropped", "S-in-place"])
def test_changed_weights_leave_the_launcher(change, gpu_device):
    mod, S = _linear(1)
    x = torch.randn(4, 160, device="cuda").to(torch.bfloat16)
    counting = _live(lambda: mod._state._launchers, lambda: mod(x))
    change(mod)
    _close(mod(x), _expect(mod, S, x))
    assert counting.calls == 1


def test_changed_weights_and_refusals(gpu_device):
    mod, S = _linear(1)
    x = torch.randn(4, 160, device="cuda").to(torch.bfloat16)
    counting = _live(lambda: mod._state._launchers, lambda: mod(x))
    with pytest.raises(TypeError):
        mod(x.half())
    with pytest.raises(ValueError):
        mod(x[:, :128])
    with pytest.raises(ValueError):
        mod(x.cpu())
    word = _runtime.status_word(x.device)
    word._word.value = 1
    assert counting.launcher.launch(x.data_ptr(), x.data_ptr()) == -1  # nothing is launched
    try:
        with pytest.raises(RuntimeError):
            mod(x)
    finally:
        clear_wait_status()
    assert counting.calls == 2  # the refused call asked it, and no other did
    _close(mod(x), _expect(mod, S, x))
    assert counting.calls == 3
    mod.half()
    _close(mod(x.half()), _expect(mod, S, x.half()))
    assert counting.calls == 3


def test_a_kept_launcher_is_not_built_again(gpu_device, monkeypatch):
    """Calls that cannot use it (an x that is copied first) leave it as it is."""
    mod, S = _linear(9)
    x = torch.randn(4, 160, device="cuda").to(torch.bfloat16)
    wide = torch.empty(4, 184, device="cuda", dtype=x.dtype)
    wide[:, 3:163] = x
    counting = _live(lambda: mod._state._launchers, lambda: mod(x))
    monkeypatch.setattr(_lib, "hostcall", lambda **kw: pytest.fail("built again"))
    for _ in range(3):
        _close(mod(wide[:, 3:163]), _expect(mod, S, x))
    mod(x)
    assert counting.calls == 2


def test_threads_share_a_launcher(gpu_device):
    """Each call fills in a copy of the descriptors: threads that use one module
    (on one stream, so that its scratch is ordered) get their own outputs."""
    mod, S = _linear(8)
    xs = [torch.randn(4, 160, device="cuda").to(torch.bfloat16) for _ in range(4)]
    want = [mod(x) for x in xs]
    counting = _live(lambda: mod._state._launchers, lambda: mod(xs[0]))
    torch.cuda.synchronize()
    with ThreadPoolExecutor(4) as pool:
        got = list(pool.map(lambda x: [mod(x) for _ in range(50)], xs))
    torch.cuda.synchronize()
    assert counting.calls == 201
    for ys, w in zip(got, want):
        assert all(torch.equal(y, w) for y in ys)


def test_groups_streams_and_grown_pools(gpu_device):
    a, Sa = _linear(2, bias=False)
    b, Sb = _linear(3, n=96)
    grp = LRSLinearGroup(a, b)
    x = torch.randn(3, 160, device="cuda").to(torch.bfloat16)
    first = [y.clone() for y in grp(x)]
    counting = _live(lambda: a._state._launchers, lambda: grp(x))
    for y, (mod, S) in zip(first, ((a, Sa), (b, Sb))):
        _close(y, _expect(mod, S, x))
    assert all(torch.equal(u, v) for u, v in zip(grp(x), first))
    assert counting.calls == 2
    word = _runtime.status_word(x.device)
    word._word.value = 1
    assert counting.launcher.launch(*[x.data_ptr()] * 3) == -1
    with pytest.raises(RuntimeError):
        grp(x)
    word.clear()
    calls = counting.calls
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            assert all(torch.equal(u, v) for u, v in zip(grp(x), first))
    side.synchronize()
    before = _runtime.generation()
    big = torch.randn(400, 160, device="cuda").to(torch.bfloat16)
    _close(grp(big)[0], _expect(a, Sa, big))
    _runtime.workspace(x.device, _runtime.workspace(x.device, 1).numel() + 1)  # a grown pool
    assert _runtime.generation() > before
    for _ in range(2):
        assert all(torch.equal(u, v) for u, v in zip(grp(x), first))
    assert counting.calls == calls  # bound to the first stream and the outgrown pool
    a._state._launchers.clear()
    counting = _live(lambda: a._state._launchers, lambda: grp(x))
    b.A.add_(1)
    _close(grp(x)[1], _expect(b, Sb, x))
    assert counting.calls == 1


@pytest.mark.parametrize("tokens", [1, 7, 100])
def test_repeated_op_calls(tokens, gpu_device):
    mod, S = _linear(4, bias=False)
    crow, col, vals = mod.S_crow, mod.S_col, mod.S_values
    act = mod.S_active_rows
    op = torch.ops.ssalaad.tilelang_bsr_addmm_inplace_dense_
    x = torch.randn(tokens, 160, device="cuda").to(torch.bfloat16)
    out0 = torch.randn(tokens, 192, device="cuda").to(torch.bfloat16)

    def run(x_, out_, v_):
        out_ = out_.clone()
        op(out_, x_, crow, col, v_, act)
        return out_

    first = run(x, out0, vals)
    kept = lambda: getattr(crow, addmm_inplace._PLAN_ATTR).calls  # noqa: E731
    assert _lib.prefill_choice() == (0, 0)
    counting = _live(kept, lambda: run(x, out0, vals))
    _close(first, out0.double() + x.double() @ S.double().T)
    for _ in range(2):
        assert torch.equal(run(x, out0, vals), first)
    _close(run(x, out0, vals * 2), out0.double() + 2 * (x.double() @ S.double().T))
    vals.mul_(0.5)
    _close(run(x, out0, vals), out0.double() + 0.5 * (x.double() @ S.double().T))
    vals.mul_(2)
    assert counting.calls == 5  # other values too: they are read anew
    wide = torch.empty(tokens, 168, device="cuda", dtype=x.dtype)
    wide[:, 1:161] = x
    assert torch.equal(run(wide[:, 1:161], out0, vals), first)
    with pytest.raises(TypeError):
        run(x.half(), out0, vals)
    assert counting.calls == 5
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(3):
            assert torch.equal(run(x, out0, vals), first)
    side.synchronize()
    assert counting.calls == 5 and len(kept()) == 2
    word = _runtime.status_word(x.device)
    word._word.value = 1
    assert counting.launcher.launch(*[x.data_ptr()] * 3) == -1
    with pytest.raises(RuntimeError):
        run(x, out0, vals)
    word.clear()
    calls = counting.calls
    _runtime.workspace(x.device, _runtime.workspace(x.device, 1).numel() + 1)  # a grown pool
    for _ in range(3):
        assert torch.equal(run(x, out0, vals), first)
    assert counting.calls == calls
    act2 = act[:-1].clone()  # fewer active rows: the last block-row keeps its bits
    out = out0.clone()
    op(out, x, crow, col, vals, act2)
    assert torch.equal(out[:, -32:], out0[:, -32:]) and torch.equal(out[:, :-32], first[:, :-32])


def test_op_does_without_the_host_call_path(gpu_device, monkeypatch):
    """Where the extension is not built every call of the op takes the full path;
    none raises after the kernel has added to out."""
    mod, S = _linear(5, bias=False)
    args = [t.clone() for t in (mod.S_crow, mod.S_col, mod.S_values, mod.S_active_rows)]
    x = torch.randn(3, 160, device="cuda").to(torch.bfloat16)
    out0 = torch.randn(3, 192, device="cuda").to(torch.bfloat16)
    monkeypatch.setattr(_lib, "_hostcall", None)
    monkeypatch.setitem(sys.modules, "ssalaad_amd.hostcall", None)  # its import fails
    monkeypatch.delattr("ssalaad_amd.hostcall")
    with pytest.raises(RuntimeError, match="not built"):
        _lib.hostcall()
    for _ in range(4):
        out = out0.clone()
        torch.ops.ssalaad.tilelang_bsr_addmm_inplace_dense_(out, x, *args)
        _close(out, out0.double() + x.double() @ S.double().T)
    assert not getattr(args[0], addmm_inplace._PLAN_ATTR).calls


def test_first_op_call_under_capture_allocates_no_pinned_memory(gpu_device, monkeypatch):
    """On a device without a status word (no fused call so far) the op makes
    none: pinned memory may not be allocated while a stream is capturing. Once
    there is one, repeated calls check it."""
    mod, _ = _linear(6, bias=False)
    args = [t.clone() for t in (mod.S_crow, mod.S_col, mod.S_values, mod.S_active_rows)]
    prepare_bsr_addmm(*args, 160)
    op = torch.ops.ssalaad.tilelang_bsr_addmm_inplace_dense_
    x = torch.randn(3, 160, device="cuda").to(torch.bfloat16)
    out0 = torch.randn(3, 192, device="cuda").to(torch.bfloat16)
    want = out0.clone()
    op(want, x, *args)
    args[0] = args[0].clone()  # no kept launchers
    prepare_bsr_addmm(*args, 160)
    monkeypatch.setattr(_runtime, "_STATUS", {})
    real = _runtime.StatusWord
    monkeypatch.setattr(_runtime, "StatusWord", lambda: pytest.fail("allocated"))
    out = out0.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        op(out, x, *args)
    for _ in range(3):
        out.copy_(out0)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    op(out.copy_(out0), x, *args)
    monkeypatch.setattr(_runtime, "StatusWord", real)
    word = _runtime.status_word(x.device)
    word._word.value = 1
    with pytest.raises(RuntimeError, match="gave up"):
        op(out, x, *args)
    word.clear()
    op(out.copy_(out0), x, *args)
    assert torch.equal(out, want)


def test_streaming_op_calls_reserve_no_part_tiles(gpu_device, monkeypatch):
    """fp32 calls of any token count stream: they ask for no room for the tiled
    kernel's parts; a 16-bit call of the same size does."""
    asked = []
    real = _runtime.workspace
    monkeypatch.setattr(_runtime, "workspace", lambda dev, n: (asked.append(n), real(dev, n))[1])
    for dtype in (torch.float32, torch.bfloat16):
        mod, _ = _linear(7, dtype=dtype, bias=False)
        x, out = (torch.zeros(300, n, device="cuda", dtype=dtype) for n in (160, 192))
        torch.ops.ssalaad.tilelang_bsr_addmm_inplace_dense_(out, x, mod.S_crow, mod.S_col,
                                                            mod.S_values, mod.S_active_rows)
        assert (_lib.prefill_choice()[0] > 0) == (dtype == torch.bfloat16)
    assert asked[0] == 0 and asked[1] == _lib.load().ssl_bsr_addmm_workspace_size(300, 6, 32, 0) > 0


def test_launchers_check_their_arguments():
    h = _lib.hostcall()
    with pytest.raises(ValueError):
        h.GroupCall(0, 0, 1, 1, 1, 64, 16, 16, 1, 0, 1, 0)
    with pytest.raises(ValueError):
        h.OpCall(0, 0, *[0] * 19)
    w = h.Watch({"a": torch.zeros(2), "b": None})
    assert not w.unchanged({"a": torch.zeros(2)})
