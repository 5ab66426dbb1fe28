"""The native host side of the hip backend (``csrc/kr_host.cpp``) classifies tensors as the Python side does, and
leaves what it does not take to it."""

import sys
import threading
import time

import pytest
import torch

from kareus_amd.backend.hip import HipBackend, load_native


def _slices():
    whole = torch.empty(40, 8, 64, dtype=torch.bfloat16)
    wide = torch.empty(16, 128, dtype=torch.bfloat16)
    deep = torch.empty(5, 3, 4, 2, 16, dtype=torch.bfloat16)
    return [whole, whole[:, 0:1], whole[:, 2:4], whole[:, 4:8], whole[:, 1:4], whole[:1, 2:4], whole[3:4, 5:6], wide,
            wide[:, :64], wide.t(), wide[:1], deep, deep[:, :, 1], deep[:, :1], deep[..., :8],
            torch.empty(4, 64, 64, dtype=torch.bfloat16)[:, :32], torch.empty(40, 8, 60, dtype=torch.bfloat16)[:, 0:2],
            torch.empty(1, 60, dtype=torch.bfloat16)]


@pytest.mark.parametrize("i", range(len(_slices())))
@pytest.mark.parametrize("max_run_rows", [16, 1])
def test_rows_view_equals_the_python_side(i, max_run_rows):
    t = _slices()[i]
    be = HipBackend.__new__(HipBackend)          # without the native side
    be.MAX_RUN_ROWS = max_run_rows
    got, want = load_native().rows_view(t, max_run_rows), be.rows_view(t)
    if want is not None and max_run_rows == 1 and want.dim() == 3:
        want = None                              # (the Python side reads the class's limit, not the instance's)
    assert (got is None) == (want is None)
    if got is not None:
        assert got.shape == want.shape and got.data_ptr() == want.data_ptr()
        assert all(n == 1 or a == b for n, a, b in zip(got.shape, got.stride(), want.stride()))


def test_split_qkv_is_the_grouped_view():
    s, b, ng, per, hd = 6, 2, 3, 4, 16
    mixed = torch.arange(s * b * ng * (per + 2) * hd, dtype=torch.float32).view(s, b, -1)
    q, k, v, fused = load_native().split_qkv(mixed, ng, per, hd)
    want = mixed.view(s, b, ng, per + 2, hd)
    assert torch.equal(fused, want) and torch.equal(q, want[:, :, :, :per])
    assert torch.equal(k, want[:, :, :, per]) and torch.equal(v, want[:, :, :, per + 1])
    assert load_native().split_qkv(mixed[:, :1], ng, per, hd) is None and load_native().split_qkv(mixed, ng + 1, per, hd) is None


def test_calls_leave_other_tensors_to_the_python_side():
    n, x = load_native(), torch.zeros(8, 8, dtype=torch.bfloat16)          # on the host: not the device's business
    assert n.gemm(0, x, x, 8, 8, 8, None, False, 1, None, None, None, 0) is None
    assert n.rmsnorm_fwd(x, x[0], 1e-5) is None and n.attn_fwd(x, x, x, 1.0, 0) is None
    assert n.dropout_bwd(x, x, 1.0) is None and n.wgrad_segments([x], [x], None, False, 1, 0) is None


@pytest.mark.parametrize("mode", ["real", "fake", "symbolic"])
def test_views_can_be_traced(mode):
    """A trace of the split and of ``rows_view`` holds for tensors that lie elsewhere in their storage."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from kareus_amd.operators import QKVPostProcessOp
    from kareus_amd.backend import hip

    s, b, ng, per, hd = 6, 2, 3, 4, 16
    x = torch.randn(4, s, b, ng * (per + 2) * hd)
    be = HipBackend.__new__(HipBackend)
    be._n = hip.load_native()
    op = QKVPostProcessOp(ng, ng * per, hd, grouped_query_view=True, backend="hip")

    def split(m):
        q, k, v = op.split(m)
        return q + 0, k + 0, v + 0, be.rows_view(m) + 0

    traced = make_fx(split, tracing_mode=mode)(x[1])
    for part in (x[0], x[2], x[3].clone()):
        f = part.view(s, b, ng, per + 2, hd)
        want = f[..., :per, :], f[..., per, :], f[..., per + 1, :], part.view(s * b, -1)
        assert all(torch.equal(a, c) for a, c in zip(traced(part), want))


# ------------------------------------------------- what the Python side refuses, the native side leaves to it
def _on_device(*shape, dtype=torch.bfloat16, device="cuda"):
    """A tensor of the device in all but its memory: a call that takes it ends before any launch."""
    from torch._subclasses.fake_tensor import FakeTensorMode

    with FakeTensorMode():
        return torch.empty(*shape, dtype=dtype, device=device)


def _backend():
    be = HipBackend.__new__(HipBackend)          # without the kernel library: nothing here may get as far
    be._n = load_native()
    return be


def test_a_rotary_call_with_the_wrong_group_size_or_table_is_refused():
    fused, table = _on_device(6, 2, 3, 6, 16), _on_device(6, 1, 1, 16, dtype=torch.float32)
    be = _backend()
    with pytest.raises(RuntimeError, match=r"contiguous \[s, b, ng, per\+2, hd\]"):
        be.rope_fused_inplace(fused, 3, table, False)
    with pytest.raises(RuntimeError, match="shape|size"):        # two rows of angles per position
        be.rope_fused_inplace(fused, 4, _on_device(6, 1, 2, 16, dtype=torch.float32), False)
    # (the right ones are taken: with no device here, that shows as the runtime's error)
    if not torch.cuda.is_available():
        with pytest.raises(RuntimeError, match="HIP"):
            be._n.rope_fused(fused, 4, table, False)


def _refused():
    d, f = _on_device, torch.float32
    a, b, deep = d(16, 64), d(32, 64), lambda n: d(2, 2, n // 4, 64)
    return {
        "gemm: B of three dimensions": lambda n: n.gemm(0, a, d(2, 16, 64), 16, 32, 64, None, False, 1, None, None, None, 0),
        "gemm: A of four": lambda n: n.gemm(0, deep(16), b, 16, 32, 64, None, False, 1, None, None, None, 0),
        "gemm: residual of four": lambda n: n.gemm(0, a, d(64, 64), 16, 64, 64, None, False, 1, deep(16), None, None, 0),
        "gemm: output of four": lambda n: n.gemm(0, a, d(64, 64), 16, 64, 64, deep(16), False, 1, None, None, None, 0),
        "gemm: one row without a row stride": lambda n: n.gemm(0, d(64).expand(1, 64).as_strided((1, 64), (0, 1)), b, 1, 32, 64,
                                                               None, False, 1, None, None, None, 0),
        "wgrad: output of three": lambda n: n.wgrad_segments([d(64, 16)], [d(64, 32)], d(1, 16, 32), False, 1, 0),
        "wgrad: pieces of four": lambda n: n.wgrad_segments([d(2, 2, 16, 16)], [d(64, 32)], None, False, 1, 0),
        "wgrad: a pair on two devices": lambda n: n.wgrad_segments([d(64, 16)], [d(64, 32, device="cuda:1")], None, False, 1, 0),
        "rmsnorm: dy of three": lambda n: n.rmsnorm_bwd(d(4, 4, 64), a, d(16, dtype=f), d(64), None, None, None),
        "rmsnorm: dx of four": lambda n: n.rmsnorm_bwd(a, a, d(16, dtype=f), d(64), None, deep(16), None),
    }


@pytest.mark.parametrize("what", sorted(_refused()))
def test_operands_the_python_side_refuses_are_left_to_it(what):
    """(What the Python side copies or views, tensors of more dimensions among it, the native side may take.)"""
    assert _refused()[what](load_native()) is None


def _bad_outs():
    d = _on_device
    return [(d(4, 2, 64), d(4, 2, 32)), (d(4, 2, 64), d(2, 4, 64).transpose(0, 1)), (d(4, 2, 64), d(4, 2, 72)[..., :64]),
            (d(4, 64), d(4, 68)[:, :64]), (d(3, 4), None), (d(4, 64), torch.empty(4, 64))]


@pytest.mark.parametrize("i", range(len(_bad_outs())))
def test_a_refused_dropout_draws_no_seed(i):
    """Shapes and strides of ``out`` that cannot be addressed: the CPU generator stays where it was, so the masks of the
    calls that follow are those of a run without the refused one."""
    x, out = _bad_outs()[i]
    before = torch.get_rng_state()
    with pytest.raises(RuntimeError, match="dropout_add|hip backend"):
        _backend().dropout_add(x, x, 0.5, out=out)
    assert torch.equal(torch.get_rng_state(), before)


def test_a_number_python_cannot_convert_ends_the_call_with_its_error():
    n, x = load_native(), torch.zeros(4, 2, 16)
    for call in (lambda: n.rows_view(x, "16"), lambda: n.split_qkv(x, None, 2, 4),
                 lambda: n.gemm(0, _on_device(8, 8), _on_device(8, 8), None, 8, 8, None, False, 1, None, None, None, 0)):
        with pytest.raises(TypeError):
            call()


def test_split_and_budget_may_be_any_truth_value_and_any_number():
    class Seen:
        def gemm(self, *args):
            self.args = args
            return "done"

    be, x = _backend(), torch.zeros(8, 8)
    be._n = Seen()
    for split, code in ((None, 0), (True, 1), (2, 1), (False, 2), (0, 2)):
        assert be.gemm(0, x, x, 8, 8, 8, split_k=split, max_cus=16.0) == "done"
        assert be._n.args[8] == code and type(be._n.args[12]) is int


def test_a_reservation_does_not_get_in_front_of_the_checks():
    from kareus_amd.backend import reserve_compute_units

    be, x = _backend(), torch.zeros(64, 64, dtype=torch.bfloat16)
    with reserve_compute_units(16):
        with pytest.raises(RuntimeError, match="needs tensors on the HIP device"):
            be.gemm(0, x, x, 64, 64, 64)
        for dys, xs in (([x], [x]), ([], [])):
            with pytest.raises(RuntimeError, match="operand pairs must be"):
                be.linear_wgrad_segments(dys, xs)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_running_out_of_memory_is_torchs_own_error():
    """(A limit on this process's share, so that nothing really runs out.)"""
    n, x = load_native(), torch.ones(8192, 8192, device="cuda", dtype=torch.bfloat16)
    gamma = torch.ones(8192, device="cuda", dtype=torch.bfloat16)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (32 << 20)) / total)
    try:
        with pytest.raises(torch.OutOfMemoryError):
            n.rmsnorm_fwd(x, gamma, 1e-5)                              # a result of 128 MiB
        with pytest.raises(torch.OutOfMemoryError):
            n.gemm(0, x, x, 8192, 8192, 8192, None, False, 0, None, None, None, 0)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
@pytest.mark.parametrize("what", ["gemm", "wgrad", "rotary"])
def test_other_threads_run_during_a_launch(what):
    """With a switch interval that never ends, another thread gets the interpreter only where the launching thread lets
    go of it: inside the native calls.  (Calls into given outputs: the end of a tensor's life lets go of it too.)  The
    launches go on until the other thread has had three turns, at most for four seconds."""
    n = load_native()
    x, out = (torch.ones(256, 256, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    fused, table = torch.ones(128, 1, 1, 3, 128, device="cuda", dtype=torch.bfloat16), torch.zeros(128, 1, 1, 128, device="cuda")
    call = {"gemm": lambda: n.gemm(0, x, x, 256, 256, 256, out, False, 0, None, None, None, 0),
            "wgrad": lambda: n.wgrad_segments([x], [x], out, False, 0, 0),
            "rotary": lambda: n.rope_fused(fused, 1, table, False)}[what]
    call()
    torch.cuda.synchronize()
    turns, stop, old = [0], [False], sys.getswitchinterval()

    def other():
        while not stop[0]:
            turns[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=other)
    sys.setswitchinterval(1000.0)
    try:
        thread.start()
        seen, end, launched = turns[0], time.perf_counter() + 4.0, 0
        while turns[0] - seen < 3 and time.perf_counter() < end and launched < 20000:
            call()
            launched += 1
    finally:
        got = turns[0] - seen
        stop[0] = True
        sys.setswitchinterval(old)
        thread.join()
    torch.cuda.synchronize()
    assert got >= 3, f"{launched} launches, {got} turns of the other thread"


# ------------------------------------------------- both sides give the same bits
class _Off:
    def __getattr__(self, name):
        return lambda *args: None


def _forms(be, dev="cuda"):
    """(name, function of the native side, call): every form a layer uses, and the odd ones beside them."""
    g = torch.Generator().manual_seed(3)
    rnd = lambda *shape: torch.randn(*shape, generator=g).to(dev, torch.bfloat16)
    new = lambda *shape: torch.zeros(*shape, device=dev, dtype=torch.bfloat16)
    m, n, k = 264, 320, 136
    x, w, dy = rnd(m, k), rnd(n, k), rnd(m, n)
    wide, runs, deep = rnd(m, 2 * k), rnd(132, 4, k)[:, 1:3], rnd(2, 2, 66, k)
    res, res_runs, add_runs = rnd(m, n), rnd(132, 4, n)[:, 2:4], rnd(132, 4, k)[:, 0:2]
    long_dy, long_x = rnd(4096, 128), rnd(4096, 136)   # cut
    for split in (True, False, None):
        yield f"forward {split}", "gemm", lambda s=split: be.linear_fwd(x, w, split_k=s)
        yield f"input gradient {split}", "gemm", lambda s=split: be.linear_dgrad(dy, w, split_k=s)
        yield f"weight gradient {split}", "gemm", lambda s=split: be.linear_wgrad(dy, x, split_k=s)
        yield f"cut weight gradient {split}", "gemm", lambda s=split: be.linear_wgrad(long_dy, long_x, split_k=s)
        yield f"pieces {split}", "wgrad_segments", lambda s=split: be.linear_wgrad_segments(
            [long_dy[:1024], long_dy[1024:2048]], [long_x[:1024], long_x[1024:2048]], split_k=s)
    yield "row stride", "gemm", lambda: be.linear_fwd(wide[:, k:], w)
    yield "budget", "gemm", lambda: be.linear_fwd(x, w, max_cus=9)
    yield "residual", "gemm", lambda: be.linear_fwd(x, w, residual=res)
    yield "residual in runs", "gemm", lambda: be.linear_fwd(x, w, residual=res_runs)
    yield "output in runs", "gemm", lambda: be.linear_fwd(x, w, residual=res, out=new(132, 4, n)[:, 0:2])
    yield "output with a row stride", "gemm", lambda: be.linear_fwd(x, w, out=new(m, n + 8)[:, :n])
    yield "accumulated", "gemm", lambda: be.linear_wgrad(dy, x, out=torch.ones(n, k, device=dev, dtype=torch.bfloat16), accumulate=True)
    yield "gradient in runs", "gemm", lambda: be.linear_dgrad(res_runs, w)
    yield "weight gradient of runs", "gemm", lambda: be.linear_wgrad(res_runs, x)
    y1 = new(m, n // 2)
    yield "swiglu", "gemm", lambda: (be.linear_fwd(x, w, swiglu_out=y1), y1)
    pre = rnd(m, 2 * k)
    yield "swiglu backward", "gemm", lambda: be.linear_dgrad(dy, w, swiglu_bwd_x=pre)
    gamma = rnd(k)
    for name, t in (("dense", x), ("row stride", wide[:, k:]), ("runs", runs), ("four dimensions", deep)):
        yield f"norm {name}", "rmsnorm_fwd", lambda t=t: be.rmsnorm_fwd(t, gamma, 1e-5)
        rstd = be.rmsnorm_fwd(t, gamma, 1e-5)[1]
        yield f"norm backward {name}", "rmsnorm_bwd", lambda t=t, r=rstd: be.rmsnorm_bwd(x, t, r, gamma)
    rstd = be.rmsnorm_fwd(runs, gamma, 1e-5)[1]
    part = torch.zeros(be.rmsnorm_partial_rows(m, k), k, device=dev)
    yield "norm backward, all in runs", "rmsnorm_bwd", lambda: (
        be.rmsnorm_bwd(x, runs, rstd, gamma, residual_grad=add_runs, out=new(132, 4, k)[:, 2:4], partials_out=part)[0], part)
    for hd, s in ((64, 200), (128, 128), (128, 72), (96, 40)):
        table = torch.randn(s + 8, 1, 1, hd, generator=g).to(dev)
        buf = rnd(s, 2, 2, 6, hd)
        q, kk, v = buf[:, :, :, :4], buf[:, :, :, 4], buf[:, :, :, 5]
        do = rnd(s, 2, 8, hd)
        for back in (False, True):
            def rope(buf=buf, table=table, back=back):
                t = buf.clone()
                be.rope_fused_inplace(t, 4, table, back)
                return t
            yield f"rotary {hd} {s} {back}", "rope_fused", rope
        for kw in ({}, dict(beside_other_streams=True), dict(general_kernels=True)):
            yield f"attention {hd} {s} {kw}", "attn_fwd", lambda a=(q, kk, v), kw=kw: be.attn_fwd(*a, 0.1, **kw)
            dense = (q.flatten(2, 3).contiguous(), kk.contiguous(), v)
            yield f"attention, dense {hd} {s} {kw}", "attn_fwd", lambda a=dense, kw=kw: be.attn_fwd(*a, 0.1, **kw)
            o, lse = be.attn_fwd(q, kk, v, 0.1, **kw)
            yield f"attention backward {hd} {s} {kw}", "attn_bwd", lambda a=(do, q, kk, v, o, lse), kw=kw: be.attn_bwd(*a, 0.1, **kw)
    x3, r3 = rnd(33, 8, k), rnd(33, 8, k)
    def dropped(out=None):
        torch.manual_seed(5)
        return be.dropout_add(x3, r3, 0.3, out=out)
    yield "dropout", "dropout_add", dropped
    yield "dropout into a tensor", "dropout_add", lambda: dropped(new(33, 8, k))
    mask = dropped()[1]
    yield "dropout backward", "dropout_bwd", lambda: be.dropout_bwd(x3, mask, 1.5)


def _flat(got):
    return [t for part in got for t in _flat(part)] if isinstance(got, (tuple, list)) else [got] if torch.is_tensor(got) else []


@pytest.mark.gpu
@pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")
def test_the_native_side_gives_the_bits_of_the_python_side():
    """Every form that the native side takes, against the same call through the Python side: the same kernels on the same
    operands, so the same bits, shapes and strides."""
    native, python = HipBackend(), HipBackend()
    python._n = _Off()
    taken = []

    class Watch:
        def __getattr__(self, name):
            fn = getattr(load_native(), name)

            def call(*args):
                got = fn(*args)
                if got is not None:
                    taken.append(name)
                return got
            return call

    native._n = Watch()
    for (name, fn, a), (_, _, b) in zip(_forms(native), _forms(python)):
        taken.clear()
        got = _flat(a())
        assert fn in taken, f"{name}: left to the Python side"
        want = _flat(b())
        assert len(got) == len(want) and got, name
        for t, u in zip(got, want):
            assert t.shape == u.shape and t.stride() == u.stride() and t.dtype == u.dtype, name
            assert torch.equal(t, u), name
