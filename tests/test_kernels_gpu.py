"""Parity of every HIP kernel with the CPU oracle, called through the C ABI (ctypes) on the same
seeded inputs.  Integer-exact where the arithmetic is exact (residual add, index maps), otherwise
bf16 tolerance: max |err| / max |ref| <= 2e-2 against the fp32 oracle evaluated on the bf16-rounded
inputs (the stated bf16 tolerance of the benchmark); observed errors are ~3e-3, one bf16 ulp."""

import ctypes
import math

import pytest
import torch

from oracle import llama_layer_ref as R

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a HIP device")]
TOL = 2e-2
DEV = "cuda"


@pytest.fixture(scope="module")
def be():
    from kareus_amd.backend import get_backend

    return get_backend("hip")


def rel(got, want):
    got, want = got.float().cpu(), want.float().cpu()
    return ((got - want).abs().max() / want.abs().max().clamp_min(1e-30)).item()


def rnd(*shape, scale=1.0, seed=0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(DEV, torch.bfloat16)


# ------------------------------------------------------------------ elementwise
@pytest.mark.parametrize("shape,p", [((64, 2, 512), 0.1), ((257, 3, 1024), 0.5), ((16, 8), 0.0), ((1000, 4096), 0.25)])
def test_dropout_add_and_its_backward(be, shape, p):
    """out = residual + dropout(x) (bias_dropout_add.py:15-45): with the mask the kernel wrote, the reference's
    arithmetic gives the same bits (dropout output rounded to bf16, then the add); about 1 - p of the elements
    are kept; the mask follows from PyTorch's CPU generator alone; the backward is dy * mask / (1 - p)."""
    x, r = rnd(*shape, seed=3), rnd(*shape, seed=4)
    torch.manual_seed(11)
    out, mask = be.dropout_add(x, r, p)
    assert mask.dtype == torch.uint8 and mask.shape == x.shape and int(mask.max()) <= 1
    keep = mask.float().mean().item()
    n = mask.numel()
    assert abs(keep - (1 - p)) <= 5 * (p * (1 - p) / n) ** 0.5 + 1e-9
    want = (r.float() + (x.float() * mask / (1 - p)).to(torch.bfloat16).float()).to(torch.bfloat16)
    assert torch.equal(out, want)
    torch.manual_seed(11)
    out2, mask2 = be.dropout_add(x, r, p)
    assert torch.equal(mask, mask2) and torch.equal(out, out2)
    if p > 0:
        torch.manual_seed(12)
        assert not torch.equal(be.dropout_add(x, r, p)[1], mask)
        # no structure along rows or between neighbours: the kept fraction of every column and of the
        # products of neighbouring mask bits is what independent draws give
        m2 = mask.view(-1, mask.shape[-1]).float()
        if m2.shape[0] >= 64:
            col = m2.mean(0)
            assert (col - (1 - p)).abs().max() <= 6 * (p * (1 - p) / m2.shape[0]) ** 0.5
        pair = (m2[:, 1:] * m2[:, :-1]).mean().item()
        assert abs(pair - (1 - p) ** 2) <= 0.02
    dy = rnd(*shape, seed=5)
    dx = be.dropout_bwd(dy, mask, 1 / (1 - p))
    assert torch.equal(dx, (dy.float() * mask / (1 - p)).to(torch.bfloat16))
    # a strided nanobatch slice as operand and as output
    if len(shape) == 3 and shape[1] >= 2:
        big_x, big_r, big_o = rnd(shape[0], 2 * shape[1], shape[2], seed=6), rnd(shape[0], 2 * shape[1], shape[2], seed=7), \
            torch.zeros(shape[0], 2 * shape[1], shape[2], device=DEV, dtype=torch.bfloat16)
        xs, rs, os_ = big_x[:, :shape[1]], big_r[:, shape[1]:], big_o[:, shape[1]:]
        torch.manual_seed(13)
        o3, m3 = be.dropout_add(xs, rs, p, out=os_)
        torch.manual_seed(13)
        o4, m4 = be.dropout_add(xs.contiguous(), rs.contiguous(), p)
        assert o3.data_ptr() == os_.data_ptr() and torch.equal(os_, o4) and torch.equal(m3, m4)
        assert not big_o[:, :shape[1]].any()


@pytest.mark.parametrize("s,b,ng,per,hd", [(64, 2, 2, 4, 128), (333, 1, 1, 1, 64), (50, 3, 3, 2, 256),
                                           (4096, 2, 2, 4, 128)])
def test_query_key_norm_and_its_backward(be, s, b, ng, per, hd):
    """The q / k layernorm of the QKV split on the fused buffer (qkv_postprocess.py:115-118, 150-157): query and
    key heads against the oracle's RMSNorm over the head dimension and its backward formula, value heads carried
    along bit for bit, weight gradients summed over all heads of the kind.  (The last case has more rows than
    the launch has row slots, so every workgroup walks several.)"""
    eps = 1e-5
    mixed = rnd(s, b, ng, per + 2, hd, seed=1)
    gq = (1 + 0.3 * torch.randn(hd, generator=torch.Generator().manual_seed(2))).to(DEV, torch.bfloat16)
    gk = (1 + 0.3 * torch.randn(hd, generator=torch.Generator().manual_seed(3))).to(DEV, torch.bfloat16)
    before = mixed.clone()
    out, rstd = be.qk_norm_fwd(mixed, gq, gk, eps)
    assert torch.equal(mixed, before) and out.shape == mixed.shape and rstd.shape == (s, b, ng, per + 1)
    xq, xk = mixed[..., :per, :].float(), mixed[..., per, :].float()
    assert rel(out[..., :per, :], R.rmsnorm(xq, gq.float(), eps)) <= TOL
    assert rel(out[..., per, :], R.rmsnorm(xk, gk.float(), eps)) <= TOL
    assert torch.equal(out[..., per + 1, :], mixed[..., per + 1, :])
    assert rel(rstd, torch.rsqrt(mixed[..., :per + 1, :].float().pow(2).mean(-1) + eps)) <= 1e-5
    dy = rnd(s, b, ng, per + 2, hd, seed=4)
    rdq, rdgq = R.rmsnorm_bwd_formula(dy[..., :per, :].float(), xq, gq.float(), eps)
    rdk, rdgk = R.rmsnorm_bwd_formula(dy[..., per, :].float(), xk, gk.float(), eps)
    dvalue = dy[..., per + 1, :].clone()
    dx, dgq, dgk = be.qk_norm_bwd(dy, mixed, rstd, gq, gk)
    assert dx.data_ptr() == dy.data_ptr()                                   # in place
    assert rel(dx[..., :per, :], rdq) <= TOL and rel(dx[..., per, :], rdk) <= TOL
    assert torch.equal(dx[..., per + 1, :], dvalue)
    assert rel(dgq, rdgq) <= TOL and rel(dgk, rdgk) <= TOL
    # the same call again gives the same bits (fixed summation order, no atomics)
    dy2 = rnd(s, b, ng, per + 2, hd, seed=4)
    dx2, dgq2, dgk2 = be.qk_norm_bwd(dy2, mixed, rstd, gq, gk)
    assert torch.equal(dx2, dx) and torch.equal(dgq2, dgq) and torch.equal(dgk2, dgk)
    with pytest.raises(RuntimeError, match="dense fused buffer"):
        be.qk_norm_fwd(mixed[:, :, :, :per + 1], gq, gk, eps)
    with pytest.raises(RuntimeError, match="head dimension"):
        be.qk_norm_fwd(mixed, gq[: hd // 2], gk, eps)


@pytest.mark.parametrize("n", [8, 1000 * 512, 4096 * 4096, 13 * 8 + 5])
def test_add_is_exact(be, n):
    a, b = rnd(n, seed=1), rnd(n, seed=2)
    assert torch.equal(be.add(a, b), a + b)
    assert torch.equal(be.add(a, a), a + a)  # aliasing inputs (ResidualFork with identical grads)


@pytest.mark.parametrize("rows,f", [(512, 1376), (64, 8), (1000, 1024), (2048, 3584)])
def test_swiglu(be, rows, f):
    x, dy = rnd(rows, 2 * f, seed=3), rnd(rows, f, seed=4)
    assert rel(be.swiglu_fwd(x), R.swiglu(x.float())) <= TOL
    assert rel(be.swiglu_bwd(dy, x), R.swiglu_bwd_formula(dy.float(), x.float())) <= TOL
    big = torch.full((8, 16), 30.0, device=DEV, dtype=torch.bfloat16)  # saturated gate: y = x1*x2, finite
    big[:, :8] *= -1
    assert torch.isfinite(be.swiglu_fwd(big)).all() and be.swiglu_fwd(big).abs().max() < 1e-8


def test_swiglu_gradient_of_a_gate_is_finite_where_that_of_its_up_value_is_not(be):
    """gy gate sigmoid(gate) above the largest float, gy sigmoid(gate) (1 + ..) up below it: on its own and in the epilogue of the
    input gradient (one row of the weight holds gy, so the product is gy exactly)."""
    gy, f = 3.0e38, 64
    gate = torch.tensor([4.0, 16.0, 20.0, 88.0]).repeat(f // 4)
    x = torch.cat([gate, torch.full((f,), 0.5)]).repeat(8, 1).to(DEV, torch.bfloat16)
    dy = torch.full((8, f), gy, device=DEV, dtype=torch.bfloat16)
    g, top = gate.double(), dy[0].double().cpu()
    want = top * torch.sigmoid(g) * (1.0 + g * (1.0 - torch.sigmoid(g))) * 0.5
    one, w = torch.zeros(8, 8, device=DEV, dtype=torch.bfloat16), torch.zeros(8, f, device=DEV, dtype=torch.bfloat16)
    one[:, 0], w[0] = 1.0, gy
    for dx in (be.swiglu_bwd(dy, x), be.linear_dgrad(one, w, swiglu_bwd_x=x)):
        d_gate, d_up = dx[:, :f].double().cpu(), dx[:, f:].double().cpu()
        assert ((d_gate - want).abs() <= 2.0 ** -8 * want).all()   # one rounding to bf16, and fp32's
        assert (d_up == math.inf).all()


@pytest.mark.parametrize("s,b,heads,hd", [(256, 2, 8, 128), (64, 1, 3, 64), (4096, 1, 2, 128)])
def test_rope(be, s, b, heads, hd):
    t = rnd(s, b, heads, hd, seed=5)
    f = R.rope_table(s, hd, 500000.0).to(DEV)
    y = be.rope_fwd(t, f)
    assert rel(y, R.rope(t.float().cpu(), f.cpu())) <= TOL
    assert rel(be.rope_bwd(t, f), R.rope(t.float().cpu(), -f.cpu())) <= TOL
    assert torch.equal(y[0], t[0])  # position 0 is the identity, exactly
    # strided input (a view into a wider buffer) gives the same result as its contiguous copy
    wide = rnd(s, b, heads + 2, hd, seed=6)
    assert torch.equal(be.rope_fwd(wide[:, :, 1:-1], f), be.rope_fwd(wide[:, :, 1:-1].contiguous(), f))


def test_rope_fused_in_place_leaves_value_heads(be):
    s, b, ng, per, hd = 128, 2, 2, 3, 128
    fused = rnd(s, b, ng, per + 2, hd, seed=7)
    before = fused.clone()
    f = R.rope_table(s, hd, 500000.0).to(DEV)
    be.rope_fused_inplace(fused, per, f, False)
    ref = R.rope(before[:, :, :, : per + 1].flatten(2, 3).float().cpu(), f.cpu()).view(s, b, ng, per + 1, hd)
    assert rel(fused[:, :, :, : per + 1], ref) <= TOL
    assert torch.equal(fused[:, :, :, per + 1], before[:, :, :, per + 1])
    be.rope_fused_inplace(fused, per, f, True)  # backward rotation undoes it up to rounding
    assert rel(fused, before) <= TOL


# ------------------------------------------------------------------ rmsnorm
@pytest.mark.parametrize("rows,cols", [(1024, 512), (130, 1024), (67, 1536), (129, 2048), (4096, 3072), (1000, 4096),
                                       (3, 8), (70, 8192), (257, 1376), (33, 2560), (40, 3584), (45, 5120), (31, 6144), (9, 4104)])
def test_rmsnorm(be, rows, cols):
    x, dy = rnd(rows, cols, seed=8), rnd(rows, cols, seed=9)
    g = (1 + 0.1 * torch.randn(cols, generator=torch.Generator().manual_seed(10))).to(DEV, torch.bfloat16)
    y, rstd = be.rmsnorm_fwd(x, g, 1e-5)
    assert rel(y, R.rmsnorm(x.float(), g.float(), 1e-5)) <= TOL
    assert rel(rstd, torch.rsqrt(x.float().pow(2).mean(-1) + 1e-5)) <= 1e-5
    dx, dg = be.rmsnorm_bwd(dy, x, rstd, g)
    rdx, rdg = R.rmsnorm_bwd_formula(dy.float(), x.float(), g.float(), 1e-5)
    assert rel(dx, rdx) <= TOL and rel(dg, rdg) <= TOL
    const = torch.full((4, cols), 3.0, device=DEV, dtype=torch.bfloat16)  # closed form for a constant row
    yc, _ = be.rmsnorm_fwd(const, torch.ones(cols, device=DEV, dtype=torch.bfloat16), 1e-5)
    assert (yc.float() - 3.0 / math.sqrt(9.0 + 1e-5)).abs().max() < 1e-2


@pytest.mark.parametrize("cols", [512, 1376, 2560, 3072, 4096, 5000, 6144, 8192])
def test_rmsnorm_backward_fused_with_residual_add_is_bit_identical(be, cols):
    """RMSNorm backward + the residual fork's gradient sum in one kernel: same bits as the two
    kernels one after the other, also when the residual gradient is a row-strided slice and the
    result goes into a slice of a larger tensor; the weight gradient is untouched."""
    rows, batch = 300, 3
    x, dy = rnd(rows, cols, seed=40), rnd(rows, cols, seed=41)
    res_full = rnd(rows, batch, cols, seed=42)
    g = (1 + 0.1 * torch.randn(cols, generator=torch.Generator().manual_seed(43))).to(DEV, torch.bfloat16)
    _, rstd = be.rmsnorm_fwd(x, g, 1e-5)
    dx_plain, dg_plain = be.rmsnorm_bwd(dy, x, rstd, g)
    res = res_full[:, 1, :]
    want = be.add(dx_plain, res)
    got, dg = be.rmsnorm_bwd(dy, x, rstd, g, residual_grad=res)
    assert torch.equal(got, want) and torch.equal(dg, dg_plain)
    whole = torch.zeros(rows, batch, cols, device=DEV, dtype=torch.bfloat16)
    sink = whole[:, 2, :]
    back, _ = be.rmsnorm_bwd(dy, x, rstd, g, residual_grad=res.contiguous(), out=sink)
    assert back.data_ptr() == sink.data_ptr() and torch.equal(whole[:, 2, :], want)
    assert not whole[:, :2, :].any()
    oracle = R.rmsnorm_bwd_formula(dy.float(), x.float(), g.float(), 1e-5)[0] + res.float()
    assert rel(got, oracle) <= TOL


def test_add_writes_into_a_batch_slice(be):
    """The residual add can put its sum into a [seq, nb, hidden] slice of a [seq, batch, hidden]
    tensor (one row stride addresses seq rows of nb*hidden elements)."""
    seq, batch, hidden = 96, 4, 512
    for nb in (1, 2):
        a, b = rnd(seq, nb, hidden, seed=50 + nb), rnd(seq, nb, hidden, seed=60 + nb)
        whole = torch.zeros(seq, batch, hidden, device=DEV, dtype=torch.bfloat16)
        out = be.add(a, b, out=whole[:, nb:2 * nb])
        assert out.data_ptr() == whole[:, nb:2 * nb].data_ptr()
        assert torch.equal(whole[:, nb:2 * nb], a + b) and not whole[:, :nb].any() and not whole[:, 2 * nb:].any()
    with pytest.raises(RuntimeError):
        be.add(a, b, out=torch.zeros(seq, hidden, 2 * nb, device=DEV, dtype=torch.bfloat16).transpose(1, 2)[:, :nb])


def test_row_strided_nanobatch_slices_need_no_copy(be):
    """One sequence out of a [seq, batch, hidden] tensor is a matrix with row stride batch*hidden:
    RMSNorm (forward and backward) and the residual add must read it in place and give exactly
    what they give on a dense copy."""
    seq, batch, hidden = 384, 4, 1024
    full, gfull = rnd(seq, batch, hidden, seed=30), rnd(seq, batch, hidden, seed=31)
    g = (1 + 0.1 * torch.randn(hidden, generator=torch.Generator().manual_seed(32))).to(DEV, torch.bfloat16)
    xs, dys = full[:, 2, :], gfull[:, 1, :]
    assert not xs.is_contiguous() and xs.stride(0) == batch * hidden
    y, rstd = be.rmsnorm_fwd(xs, g, 1e-5)
    yd, rstdd = be.rmsnorm_fwd(xs.contiguous(), g, 1e-5)
    assert torch.equal(y, yd) and torch.equal(rstd, rstdd) and y.is_contiguous()
    dx, dg = be.rmsnorm_bwd(dys, xs, rstd, g)
    dxd, dgd = be.rmsnorm_bwd(dys.contiguous(), xs.contiguous(), rstd, g)
    assert torch.equal(dx, dxd) and torch.equal(dg, dgd)
    dense = rnd(seq, 1, hidden, seed=33)
    out = be.add(full[:, 2:3, :], dense)                      # strided + dense, 3-D as the engine passes them
    assert out.shape == dense.shape and out.is_contiguous()
    assert torch.equal(out, full[:, 2:3, :] + dense)
    assert torch.equal(be.add(dense, gfull[:, 0:1, :]), dense + gfull[:, 0:1, :])
    assert torch.equal(be.add(full[:, 0:1, :], gfull[:, 3:4, :]), full[:, 0:1, :] + gfull[:, 3:4, :])
    wide = be.add(full[:, 0:2, :], gfull[:, 2:4, :])           # two sequences: no single row stride, copied
    assert torch.equal(wide, full[:, 0:2, :] + gfull[:, 2:4, :])


# ------------------------------------------------------------------ GEMM
SHAPES = [(256, 256, 64), (512, 768, 512), (264, 520, 200), (1024, 2752, 512), (2048, 512, 1376),
          (8, 8, 8), (4096, 640, 384), (40, 1536, 4096),
          # outputs of 192 tiles or more, where the library picks narrower tiles than 256 columns:
          (4096, 3584, 128),    # 224 columns (16 x 16 tiles fill one round of workgroups)
          (16384, 768, 64),     # 192 columns
          (16384, 640, 72),     # 160 columns, and a contraction tail
          # outputs of fewer than 192 full tiles, where narrower tiles and cuts of the contraction compete:
          (4096, 1536, 4096),   # forward: 128-column tiles uncut; the other two layouts take other plans
          (4088, 1000, 2056),   # the same with ragged edges in all three dimensions
          (1536, 4096, 1024)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_three_layouts(be, m, n, k):
    x, w, dy = rnd(m, k, seed=11), rnd(n, k, scale=0.05, seed=12), rnd(m, n, seed=13)
    assert rel(be.linear_fwd(x, w), x.float() @ w.float().t()) <= TOL
    assert rel(be.linear_dgrad(dy, w), dy.float() @ w.float()) <= TOL
    assert rel(be.linear_wgrad(dy, x), dy.float().t() @ x.float()) <= TOL


def test_gemm_plan_does_not_change_the_sums_much(be):
    """The library picks tile width and cuts of the contraction by a cost model that depends on the
    workspace it is given (alone on the GPU: cuts allowed; beside other streams: fewer or none; never:
    no workspace).  All plans compute the same sums, up to the rounding of a cut's fp32 partial tiles."""
    for (m, n, k) in [(4096, 1536, 4096), (4096, 1024, 4096), (1536, 4096, 4096), (520, 264, 8192)]:
        x, w, dy, xx = rnd(m, k, seed=31), rnd(n, k, scale=0.05, seed=32), rnd(k, m, scale=0.1, seed=33), rnd(k, n, seed=34)
        for layout, a, b, ref in ((0, x, w, x.float() @ w.float().t()), (1, x, w.t().contiguous(), x.float() @ w.float().t()),
                                  (2, dy, xx, dy.float().t() @ xx.float())):
            outs = [be.gemm(layout, a, b, m, n, k, split_k=mode) for mode in (True, False, None)]
            for o in outs:
                assert rel(o, ref) <= TOL
            assert rel(outs[0], outs[2]) <= 1e-2 and rel(outs[1], outs[2]) <= 1e-2
            c0 = rnd(m, n, seed=35)
            acc = be.gemm(layout, a, b, m, n, k, out=c0.clone(), accumulate=True, split_k=None)
            assert rel(acc, ref + c0.float()) <= TOL


def _gemm_plan(be, m, n, k, epilogue=0, workspace=0):
    rows, splits = ctypes.c_int(), ctypes.c_int()
    assert be.lib.kr_gemm_plan(m, n, k, epilogue, 0, workspace, ctypes.byref(rows), ctypes.byref(splits)) == 0
    return rows.value, splits.value


def _gemm_tile(be, layout, m, n, k, epilogue=0, accumulate=0, max_cus=0, workspace=0):
    rows, cols, pieces = ctypes.c_int(), ctypes.c_int(), ctypes.c_int()
    assert be.lib.kr_gemm_plan_tile(layout, m, n, k, epilogue, accumulate, max_cus, workspace, ctypes.byref(rows), ctypes.byref(cols),
                                    ctypes.byref(pieces)) == 0
    return rows.value, cols.value, pieces.value


@pytest.mark.parametrize("m,n,k", [(8, 8, 8), (128, 128, 64), (136, 264, 72), (120, 128, 128), (520, 1024, 200),
                                   (264, 136, 584), (136, 640, 720), (256, 1000, 1096),   # the deep ring, contraction tails
                                   (512, 3584, 1024),     # one round of small tiles, more than one per compute unit
                                   (2048, 3456, 136)])    # 432 small tiles
def test_gemm_small_tiles_have_the_bits_of_the_large_ones(be, m, n, k):
    """Outputs of few tiles are computed in tiles of 128 rows or 64.  The same rows and columns as a corner of an output of 192
    and more large tiles, which is computed in them: every element is the same chain of matrix instructions in both, so
    the bits are the same.  (Both plans are asserted.)"""
    def embed(t, rows=None, cols=None):
        r, c = max(rows or t.shape[0], t.shape[0]), max(cols or t.shape[1], t.shape[1])
        big = rnd(r, c, scale=0.05, seed=67)
        big[:t.shape[0], :t.shape[1]] = t
        return big

    R_, C_ = 4096, 3072   # 16 x 12 large tiles at the least
    x, w, dy = rnd(m, k, seed=61), rnd(n, k, scale=0.05, seed=62), rnd(m, n, seed=63)
    for layout, a, b, (p, q, c) in ((0, x, w, (m, n, k)), (1, dy, w, (m, k, n)), (2, dy, x, (n, k, m))):
        big = (max(p, R_), max(q, C_), c)
        rows, cols, pieces = _gemm_tile(be, layout, p, q, c)
        assert rows <= 128 and cols <= 128 and pieces == 1 and max(_gemm_tile(be, layout, *big)[:2]) == 256
        big_a = embed(a, cols=R_) if layout == 2 else embed(a, rows=R_)
        big_b = embed(b, rows=C_) if layout == 0 else embed(b, cols=C_)
        got = be.gemm(layout, a, b, p, q, c, split_k=None)
        assert torch.equal(got, be.gemm(layout, big_a, big_b, *big, split_k=None)[:p, :q])
        base = rnd(p, q, seed=64)
        assert torch.equal(be.gemm(layout, a, b, p, q, c, out=base.clone(), accumulate=True, split_k=None),
                           be.gemm(layout, big_a, big_b, *big, out=embed(base, R_, C_), accumulate=True, split_k=None)[:p, :q])
        wide = torch.zeros(p, q + 8, device=DEV, dtype=torch.bfloat16)
        be.gemm(layout, a, b, p, q, c, out=wide[:, :q], split_k=None)
        assert torch.equal(wide[:, :q], got) and not wide[:, q:].any()
    assert rel(be.linear_fwd(x, w), x.float() @ w.float().t()) <= TOL
    big_x, big_w, big = embed(x, rows=R_), embed(w, rows=C_), (max(m, R_), max(n, C_), k)
    res = rnd(m, n, seed=65)
    assert _gemm_plan(be, m, n, k, 1)[0] <= 128 and _gemm_plan(be, *big, 1)[0] == 256
    assert torch.equal(be.linear_fwd(x, w, residual=res), be.linear_fwd(big_x, big_w, residual=embed(res, R_, C_))[:m, :n])


@pytest.mark.parametrize("m,n,k,tile", [(8, 8, 8, (64, 64)), (64, 64, 64, (64, 64)), (72, 136, 1096, (64, 64)), (200, 328, 264, (64, 64)),
                                        (128, 4096, 200, (64, 64)), (520, 3208, 584, (128, 64)), (1000, 512, 2752, (64, 64)),
                                        (264, 1376, 256, (64, 64)),
                                        # more tiles than compute units, or one per unit and short or deep rings of K-steps
                                        (2008, 3456, 200, (128, 128)), (1000, 5000, 1096, (128, 128)), (520, 5000, 72, (128, 128)),
                                        (776, 4096, 584, (128, 128)), (776, 2952, 1096, (128, 128)), (904, 4096, 2056, (128, 128))])
def test_gemm_smallest_tiles_have_the_bits_of_the_large_ones(be, m, n, k, tile):
    """Outputs of few tiles are computed in 128 x 128 tiles, those that would leave compute units without one in 128 x 64 or
    64 x 64: every layout and kind of output against a corner of an output of 192 large tiles, at contractions shorter than the
    ring and longer.  (What runs is asserted.)"""
    M, N = 4096, 3072 if n <= 3072 else 4096 if n <= 4096 else 5120
    a, b, old, res = rnd(M, k, seed=61), rnd(N, k, scale=0.05, seed=62), rnd(M, N, seed=63), rnd(M, N, seed=64)

    def asserted(layout, epilogue=0, accumulate=0):
        assert _gemm_tile(be, layout, m, n, k, epilogue, accumulate) == (*tile, 1)
        assert max(_gemm_tile(be, layout, M, N, k, epilogue, accumulate)[:2]) == 256

    for layout, f, g in ((0, lambda t: t, lambda t: t), (1, lambda t: t, lambda t: t.t().contiguous()),
                         (2, lambda t: t.t().contiguous(), lambda t: t.t().contiguous())):
        big, few = (layout, f(a), g(b), M, N, k), (layout, f(a[:m]), g(b[:n]), m, n, k)
        asserted(layout)
        assert torch.equal(be.gemm(*few, split_k=None), be.gemm(*big, split_k=None)[:m, :n])
        asserted(layout, accumulate=1)
        acc = [be.gemm(*c, out=o.clone(), accumulate=True, split_k=None) for c, o in ((few, old[:m, :n]), (big, old))]
        assert torch.equal(acc[0], acc[1][:m, :n])
    assert rel(be.linear_fwd(a[:m], b[:n]), a[:m].float() @ b[:n].float().t()) <= TOL
    asserted(0, 1)
    assert torch.equal(be.linear_fwd(a[:m], b[:n], residual=res[:m, :n]), be.linear_fwd(a, b, residual=res)[:m, :n])
    wt = b.t().contiguous()
    pre = rnd(M, 2 * N, seed=65)
    few_pre = torch.cat([pre[:m, :n], pre[:m, N:N + n]], dim=1)
    asserted(1, 4)
    dx, big_dx = (be.linear_dgrad(x, w, swiglu_bwd_x=p) for x, w, p in ((a[:m], wt[:, :n].contiguous(), few_pre), (a, wt, pre)))
    assert torch.equal(dx[:, :n], big_dx[:m, :n]) and torch.equal(dx[:, n:], big_dx[:m, N:N + n])


@pytest.mark.parametrize("m,n,k,cus", [(1024, 512, 2048, 120), (1000, 504, 1992, 116), (1000, 1000, 2056, 196), (256, 512, 1376, 12), (256, 512, 1376, 28), (504, 2040, 4104, 88),
                                       (512, 2048, 4104, 248)])
def test_gemm_smallest_tiles_add_up_the_pieces_that_larger_ones_are_cut_into(be, m, n, k, cus):
    """A contraction that larger tiles would be cut into: the 128 x 64 and 64 x 64 tiles walk it whole and add it up in the same
    pieces, in the same order.  Against the cut launch on fewer compute units (both plans are asserted), in every layout, stored,
    accumulated and with the operands in pieces of their own."""
    a, b, old = rnd(m, k, seed=61), rnd(n, k, scale=0.05, seed=62), rnd(m, n, seed=64)
    ws = be.lib.kr_gemm_workspace_bytes(0, m, n, k)
    for layout, x, w in ((0, a, b), (1, a, b.t().contiguous()), (2, a.t().contiguous(), b.t().contiguous())):
        for acc in (False, True):
            whole, cut = (_gemm_tile(be, layout, m, n, k, 0, acc, c, ws) for c in (0, cus))
            assert whole[:2] == (64, 64) and cut[0] * cut[1] > 64 * 64 and whole[2] == cut[2] > 1
            got = [be.gemm(layout, x, w, m, n, k, max_cus=c, **(dict(out=old.clone(), accumulate=True) if acc else {})) for c in (0, cus)]
            assert torch.equal(*got)
            assert rel(got[0], a.float() @ b.float().t() + (old.float() if acc else 0.0)) <= TOL
    if k % 64 == 0:
        x, w = a.t().contiguous(), b.t().contiguous()
        half = k // 128 * 64
        if 2 * half == k:
            assert torch.equal(be.linear_wgrad_segments([x[:half], x[half:]], [w[:half], w[half:]]), be.gemm(2, x, w, m, n, k))


@pytest.mark.parametrize("m,M,n,k,rows", [(536, 1024, 16384, 72, 192), (776, 1024, 16384, 200, 224), (1600, 2048, 8192, 64, 224),
                                          (3000, 4096, 4096, 136, 192), (6024, 7424, 4096, 136, 192),
                                          # a partial last column of tiles, many K-steps with a partial last one
                                          (776, 1024, 16360, 1096, 224), (1600, 2048, 8136, 1096, 224), (536, 1024, 16328, 1096, 192),
                                          (3000, 4096, 4088, 1096, 192)])
def test_gemm_tiles_of_fewer_rows_have_the_bits_of_the_large_ones(be, m, M, n, k, rows):
    """Outputs whose rows or rounds 224 or 192 rows divide better than 256: the first rows of an output of M, which takes 256,
    plain and with a residual, with one K-step, two, three and many of them, the last one whole or partial.  (What runs is
    asserted.)"""
    for layout, epilogue in ((0, 0), (1, 0), (0, 1)):
        assert _gemm_tile(be, layout, m, n, k, epilogue) == (rows, 256, 1) and _gemm_tile(be, layout, M, n, k, epilogue) == (256, 256, 1)
    a, b, res = rnd(M, k, seed=61), rnd(n, k, scale=0.05, seed=62), rnd(M, n, seed=64)
    wt, few = b.t().contiguous(), a[:m]
    got = be.linear_fwd(few, b)
    assert torch.equal(got, be.linear_fwd(a, b)[:m]) and rel(got, few.float() @ b.float().t()) <= TOL
    assert torch.equal(be.linear_dgrad(few, wt), be.linear_dgrad(a, wt)[:m])
    assert torch.equal(be.linear_fwd(few, b, residual=res[:m]), be.linear_fwd(a, b, residual=res)[:m])


@pytest.mark.parametrize("m,n,k,rows", [(3000, 4088, 1096, 192), (3000, 4088, 136, 192), (1600, 8136, 1096, 224), (1600, 8136, 72, 224)])
def test_gemm_tiles_of_fewer_rows_several_to_a_workgroup(be, m, n, k, rows):
    """On half the compute units a workgroup has two such tiles, on all of them one: the same bits."""
    a, b, res = rnd(m, k, seed=61), rnd(n, k, scale=0.05, seed=62), rnd(m, n, seed=64)
    for layout, w, what in ((0, b, {}), (1, b.t().contiguous(), {}), (0, b, dict(residual=res))):
        got = []
        for cus in (0, 128):
            assert _gemm_tile(be, layout, m, n, k, 1 if what else 0, max_cus=cus) == (rows, 256, 1)
            got.append(be.gemm(layout, a, w, m, n, k, split_k=None, max_cus=cus, **what))
        assert torch.equal(*got)


@pytest.mark.parametrize("m,n,k", [(3080, 2008, 2056), (1544, 4072, 2104), (6024, 1000, 1032), (5000, 1160, 4096), (4104, 1032, 1992)])
def test_gemm_narrow_tiles_have_the_bits_of_wide_ones(be, m, n, k):
    """Outputs of fewer large tiles than compute units take narrower ones, down to 128 columns, whose transposed operand has a
    layout of its own: the corner of an output of 192 tiles and more, with remainders in rows, columns and contraction."""
    M, N = 6144, 4096
    a, b = rnd(M, k, seed=61), rnd(N, k, scale=0.05, seed=62)
    for layout, f, g in ((0, lambda t: t, lambda t: t), (1, lambda t: t, lambda t: t.t().contiguous()),
                         (2, lambda t: t.t().contiguous(), lambda t: t.t().contiguous())):
        big = be.gemm(layout, f(a), g(b), M, N, k, split_k=None)
        got = be.gemm(layout, f(a[:m]), g(b[:n]), m, n, k, split_k=None)
        assert torch.equal(got, big[:m, :n])
    assert rel(got, a[:m].float() @ b[:n].float().t()) <= TOL


@pytest.mark.parametrize("tile", [128, 256])
@pytest.mark.parametrize("k", [8, 64, 72, 128, 136, 192, 200, 1096])
def test_gemm_items_of_one_workgroup_have_the_bits_of_items_of_their_own(be, k, tile):
    """A workgroup that has further items requests their first K-steps in the last two of the one it is at.  On eight
    compute units every workgroup has several items, on the whole device one at most: the same bits, in every layout, with
    every kind of output, at contractions of one K-step, two, three and many, with and without a partial last one."""
    m, n = (520, 640) if tile == 128 else (4104, 3080)
    x, w, dy = rnd(m, k, seed=61), rnd(n, k, scale=0.05, seed=62), rnd(m, n, seed=63)
    for layout, a, b, (p, q, c) in ((0, x, w, (m, n, k)), (1, x, w.t().contiguous(), (m, n, k)),
                                    (2, x.t().contiguous(), w.t().contiguous(), (m, n, k))):
        alone, few = (dict(split_k=None, max_cus=cus) for cus in (0, 8))
        got = be.gemm(layout, a, b, p, q, c, **few)
        assert torch.equal(got, be.gemm(layout, a, b, p, q, c, **alone))
        base = rnd(p, q, seed=64)
        assert torch.equal(be.gemm(layout, a, b, p, q, c, out=base.clone(), accumulate=True, **few),
                           be.gemm(layout, a, b, p, q, c, out=base.clone(), accumulate=True, **alone))
    assert rel(got, x.float() @ w.float().t()) <= TOL
    pre = rnd(m, 2 * n, seed=65)
    assert torch.equal(be.gemm(0, x, w, m, n, k, residual=dy, **few), be.gemm(0, x, w, m, n, k, residual=dy, **alone))
    wt = w.t().contiguous()
    assert torch.equal(be.gemm(1, x, wt, m, n, k, swiglu_bwd_x=pre, **few), be.gemm(1, x, wt, m, n, k, swiglu_bwd_x=pre, **alone))
    f = 1280 if tile == 256 else 320
    ys = [torch.empty(m, f, device=DEV, dtype=torch.bfloat16) for _ in range(2)]
    x2 = [be.gemm(0, x, w[:2 * f].contiguous(), m, 2 * f, k, swiglu_out=y, **how) for y, how in zip(ys, (few, alone))]
    assert torch.equal(*x2) and torch.equal(*ys)


@pytest.mark.parametrize("m,f,k,forward,backward", [(8, 64, 64, (64, 64), (64, 64)), (128, 320, 128, (64, 64), (64, 64)),
                                                    (136, 448, 200, (64, 64), (64, 64)), (520, 512, 1096, (64, 64), (64, 64)),
                                                    (512, 1792, 1024, (128, 64), (64, 64)), (776, 2048, 584, (128, 128), (128, 64)),
                                                    (1000, 1728, 1096, (128, 128), (128, 64)), (520, 2048, 2056, (128, 128), (128, 64)),
                                                    (2008, 1536, 72, (128, 128), (128, 128))])
def test_gemm_small_tiles_with_swiglu_have_the_bits_of_the_large_ones(be, m, f, k, forward, backward):
    """The SwiGLU epilogues, forward (gate and up columns of a tile side by side) and backward, in the same way."""
    M, F = max(m, 4096), max(3584, f)      # 16 x 28 large tiles: gate and up
    x, gate, up = rnd(M, k, seed=61), rnd(F, k, scale=0.05, seed=62), rnd(F, k, scale=0.05, seed=63)
    xs, ws = x[:m].contiguous(), torch.cat([gate[:f], up[:f]])
    if be.can_fuse_swiglu(2 * f):
        assert _gemm_tile(be, 0, m, 2 * f, k, 2) == (*forward, 1) and _gemm_plan(be, M, 2 * F, k, 2)[0] == 256
        y, big_y = (torch.empty(r, c, device=DEV, dtype=torch.bfloat16) for r, c in ((m, f), (M, F)))
        got, big = be.linear_fwd(xs, ws, swiglu_out=y), be.linear_fwd(x, torch.cat([gate, up]), swiglu_out=big_y)
        assert torch.equal(got[:, :f], big[:m, :f]) and torch.equal(got[:, f:], big[:m, F:F + f]) and torch.equal(y, big_y[:m, :f])
    # backward: the gradient of the activation, [m, f] = dy [m, k] . W [k, f], never stored; out [m, 2 f]
    dy, w, pre = rnd(M, k, seed=66), rnd(k, F, scale=0.05, seed=67), rnd(M, 2 * F, seed=68)
    assert _gemm_tile(be, 1, m, f, k, 4) == (*backward, 1) and _gemm_plan(be, M, F, k, 4)[0] == 256
    pre_s = torch.cat([pre[:m, :f], pre[:m, F:F + f]], dim=1)
    got = be.linear_dgrad(dy[:m].contiguous(), w[:, :f].contiguous(), swiglu_bwd_x=pre_s)
    big = be.linear_dgrad(dy, w, swiglu_bwd_x=pre)
    assert torch.equal(got[:, :f], big[:m, :f]) and torch.equal(got[:, f:], big[:m, F:F + f])


@pytest.mark.parametrize("m,n,k", [(776, 7168, 2560), (1000, 5120, 2568), (2040, 4096, 1544), (1160, 4352, 2632)])
def test_gemm_one_round_of_narrow_tiles_with_an_epilogue_has_the_bits_of_wide_ones(be, m, n, k):
    """More 128 x 128 tiles than compute units, whose 256 x 128 tiles are one round: the residual and both SwiGLU epilogues against
    a corner of an output of 192 tiles and more, with remainders in rows, columns (backward) and contraction, and with the
    residual in row runs."""
    M, f = 4096, n // 2
    F = max(3584, f)
    x, gate, up = rnd(M, k, seed=61), rnd(F, k, scale=0.05, seed=62), rnd(F, k, scale=0.05, seed=63)
    xs, ws = x[:m].contiguous(), torch.cat([gate[:f], up[:f]])
    assert _gemm_tile(be, 0, m, n, k, 2) == (256, 128, 1)
    y, big_y = (torch.empty(r, c, device=DEV, dtype=torch.bfloat16) for r, c in ((m, f), (M, F)))
    got, big = be.linear_fwd(xs, ws, swiglu_out=y), be.linear_fwd(x, torch.cat([gate, up]), swiglu_out=big_y)
    assert torch.equal(got[:, :f], big[:m, :f]) and torch.equal(got[:, f:], big[:m, F:F + f]) and torch.equal(y, big_y[:m, :f])
    c = n - 8  # a remainder in columns
    res, w = rnd(M, 2 * F, seed=65), torch.cat([gate, up])
    assert _gemm_tile(be, 0, m, c, k, 1)[:2] == (256, 128) and max(_gemm_tile(be, 0, M, 2 * F, k, 1)[:2]) == 256
    want = be.linear_fwd(x, w, residual=res)[:m, :c]
    assert torch.equal(be.linear_fwd(xs, w[:c].contiguous(), residual=res[:m, :c].contiguous()), want)
    runs = torch.zeros(m // 4, 8, c, device=DEV, dtype=torch.bfloat16)[:, 2:6]
    runs.copy_(res[:m, :c].reshape(m // 4, 4, c))
    assert torch.equal(be.linear_fwd(xs, w[:c].contiguous(), residual=runs), want)
    dy, wb, pre = rnd(M, k, seed=66), rnd(k, 2 * F, scale=0.05, seed=67), rnd(M, 4 * F, seed=68)
    assert _gemm_tile(be, 1, m, c, k, 4) == (256, 128, 1) and _gemm_plan(be, M, 2 * F, k, 4)[0] == 256
    pre_s = torch.cat([pre[:m, :c], pre[:m, 2 * F:2 * F + c]], dim=1)
    got = be.linear_dgrad(dy[:m].contiguous(), wb[:, :c].contiguous(), swiglu_bwd_x=pre_s)
    big = be.linear_dgrad(dy, wb, swiglu_bwd_x=pre)
    assert torch.equal(got[:, :c], big[:m, :c]) and torch.equal(got[:, c:], big[:m, 2 * F:2 * F + c])


@pytest.mark.parametrize("layout", [0, 1, 2])
@pytest.mark.parametrize("steps,tail", [(151, 64), (151, 8), (152, 40), (153, 64), (153, 24), (154, 8), (155, 64), (159, 56)])
def test_gemm_deep_ring_cut_into_short_last_ranges(be, layout, steps, tail):
    """Small tiles alone on their compute units request four K-steps ahead; cut sixteen ways, ``steps`` K-steps leave 1, 2, 3,
    4, 5 and 9 for the last range (10 for the others), the last one of ``tail`` rows.  Operands of -1, 0 and 1: every
    sum is a small whole number, exact in fp32 in any order, so the result is the exact product rounded to bf16 once."""
    m, n, k = 128, 120, (steps - 1) * 64 + tail
    ws = be.lib.kr_gemm_workspace_bytes(layout, m, n, k)
    assert ws == 16 * m * n * 4 and _gemm_plan(be, m, n, k, workspace=ws) == (128, 16)
    assert k // 64 // 16 > 8                                  # the deep ring's condition
    g = torch.Generator().manual_seed(steps)
    a, b = (torch.randint(-1, 2, s, generator=g).to(DEV, torch.bfloat16) for s in (((k, m) if layout == 2 else (m, k)),
                                                                                   ((n, k) if layout == 0 else (k, n))))
    want = (a.double().t() if layout == 2 else a.double()) @ (b.double().t() if layout == 0 else b.double())
    assert torch.equal(be.gemm(layout, a, b, m, n, k), want.to(torch.bfloat16))
    base = torch.randint(-3, 4, (m, n), generator=g).to(DEV, torch.bfloat16)
    assert torch.equal(be.gemm(layout, a, b, m, n, k, out=base.clone(), accumulate=True), (want + base.double()).to(torch.bfloat16))


def test_gemm_is_reproducible(be):
    """No atomics and a fixed order of accumulation: repeated launches give the same bits (a
    race on an LDS tile between the waves of a workgroup would show up here)."""
    m, n, k = 4096, 3584, 1088
    x, w, dy = rnd(m, k, seed=14), rnd(n, k, scale=0.05, seed=15), rnd(m, n, seed=16)
    first = (be.linear_fwd(x, w).clone(), be.linear_dgrad(dy, w).clone(), be.linear_wgrad(dy, x).clone())
    for _ in range(5):
        again = (be.linear_fwd(x, w), be.linear_dgrad(dy, w), be.linear_wgrad(dy, x))
        assert all(torch.equal(a, b) for a, b in zip(again, first))


def test_gemm_closed_forms(be):
    eye = torch.eye(512, device=DEV, dtype=torch.bfloat16)
    x = rnd(264, 512, seed=14)
    assert torch.equal(be.linear_fwd(x, eye), x) and torch.equal(be.linear_dgrad(x, eye), x)  # identity weight
    ones = torch.ones(128, 512, device=DEV, dtype=torch.bfloat16)
    small = (torch.arange(264 * 512) % 7 - 3).reshape(264, 512).to(DEV, torch.bfloat16)  # exact small ints
    assert torch.equal(be.linear_fwd(small, ones).float(), small.float().sum(1, keepdim=True).expand(264, 128))
    onehot = torch.zeros(264, 8, device=DEV, dtype=torch.bfloat16)  # dW = dy^T x with one-hot dy picks rows of x
    onehot[5, 3] = 1
    dw = be.linear_wgrad(onehot, x)
    assert torch.equal(dw[3], x[5]) and dw.abs().sum() == x[5].abs().sum()


def test_gemm_split_k_accumulate_and_strides(be):
    for (m, n, k) in [(512, 768, 4096), (264, 520, 2440)]:
        dy, x = rnd(k, m, scale=0.1, seed=15), rnd(k, n, seed=16)
        assert be.lib.kr_gemm_workspace_bytes(2, m, n, k) > 0  # this shape is computed split-K
        ref = dy.float().t() @ x.float()
        assert rel(be.linear_wgrad(dy, x), ref) <= TOL
        c0 = rnd(m, n, seed=17)
        assert rel(be.gemm(2, dy, x, m, n, k, out=c0.clone(), accumulate=True), ref + c0.float()) <= TOL
    a, w, c0 = rnd(296, 512, seed=18), rnd(264, 512, seed=19), rnd(296, 264, seed=20)
    assert rel(be.gemm(0, a, w, 296, 264, 512, out=c0.clone(), accumulate=True), a.float() @ w.float().t() + c0.float()) <= TOL
    wide = rnd(296, 1024, seed=21)  # lda > K: operand is a column slice of a wider matrix
    assert torch.equal(be.gemm(0, wide[:, 256:768], w, 296, 264, 512), be.gemm(0, wide[:, 256:768].contiguous(), w, 296, 264, 512))
    with pytest.raises(RuntimeError, match="not supported"):
        be.gemm(0, a[:295], w, 295, 264, 512)


# ------------------------------------------------------------------ attention
def _grouped(s, b, nq, nkv, hd, seed):
    per = nq // nkv
    fused = rnd(s, b, nkv, per + 2, hd, seed=seed)
    return fused, fused[:, :, :, :per], fused[:, :, :, per], fused[:, :, :, per + 1]


@pytest.mark.parametrize("s,b,nq,nkv", [(128, 1, 1, 1), (256, 2, 4, 2), (512, 1, 3, 1), (384, 1, 8, 8), (1024, 1, 4, 1),
                                        (2048, 1, 2, 1),    # 32 query tiles per key tile: the steady state of the pipelines
                                        (512, 17, 8, 8),    # 544 workgroups, one query head per KV head: dK/dV written directly
                                        (640, 3, 6, 2),     # odd tile count, three query heads per KV head
                                        (256, 1, 24, 8),    # the head map of benchmark configuration 3 (Llama-3.2-3B)
                                        (256, 2, 32, 8),    # ... and of configuration 5 (Llama-3.1-8B), four query heads per KV head
                                        # enough 256-query tiles for every compute unit: the forward kernel whose halves share K / V tiles
                                        (1024, 8, 8, 2),    # 4 tiles x 64 (batch, head) pairs, eight pairs start together on an XCD
                                        (768, 11, 8, 8),    # 3 tiles per pair: plain longest-first order
                                        (512, 33, 8, 2),    # 2 tiles per pair, 264 pairs: the last group of 16 pairs is incomplete
                                        (2304, 4, 8, 2),    # 9 tiles per pair: an odd tile count, half 0 idles through two steps of 36
                                        (512, 6, 24, 8),    # three query heads per KV head in the shared-tile kernels
                                        # enough key tiles that a dK/dV workgroup serves several query heads of its KV group:
                                        (512, 32, 8, 4),    # both heads of a group: dK/dV stored directly, no partial results
                                        (512, 64, 8, 2),    # all four heads of a group
                                        (256, 128, 6, 2)])  # all three heads of a group
def test_attention_forward_backward(be, s, b, nq, nkv):
    hd = 128
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=22)
    do = rnd(s, b, nq, hd, seed=23)
    o, lse = be.attn_fwd(q, k, v, hd ** -0.5)
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
    ro.backward(do.float().cpu())
    dq, dk, dv = be.attn_bwd(do, q, k, v, o, lse, hd ** -0.5)
    assert rel(dq.flatten(2, 3), qf.grad) <= TOL and rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL
    assert dq._kr_mixed.shape == (s, b, (nq + 2 * nkv) * hd)  # gradients share one fused buffer
    again = be.attn_bwd(do, q, k, v, o, lse, hd ** -0.5)       # no atomics, fixed reduction order: same bits
    assert all(torch.equal(x, y) for x, y in zip(again, (dq, dk, dv)))
    # dense [s, b, nq, hd] tensors go through the same kernels
    qd = q.flatten(2, 3).contiguous()
    od, lsed = be.attn_fwd(qd, k.contiguous(), v.contiguous(), hd ** -0.5)
    assert torch.equal(od, o) and torch.equal(lsed, lse)
    dqd, dkd, dvd = be.attn_bwd(do, qd, k.contiguous(), v.contiguous(), od, lsed, hd ** -0.5)
    assert torch.equal(dqd, dq.flatten(2, 3)) and torch.equal(dkd, dk) and torch.equal(dvd, dv)


def test_attention_at_sequence_8192(be):
    """The sequence length of benchmark configuration 5, against the brute-force oracle (two query heads on
    one KV head keep the oracle's 8192 x 8192 score matrices within a few seconds of CPU time)."""
    s, b, nq, nkv, hd = 8192, 1, 2, 1, 128
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=70)
    do = rnd(s, b, nq, hd, seed=71)
    o, lse = be.attn_fwd(q, k, v, hd ** -0.5)
    dq, dk, dv = be.attn_bwd(do, q, k, v, o, lse, hd ** -0.5)
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
    ro.backward(do.float().cpu())
    assert rel(dq.flatten(2, 3), qf.grad) <= TOL and rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL
    # the whole forms (256-query workgroups: the query gradient with one wave per SIMD walks 128 key tiles here)
    o2, lse2 = be.attn_fwd(q, k, v, hd ** -0.5, beside_other_streams=True)
    assert rel(o2, ro) <= TOL and rel(lse2, rlse) <= 1e-4
    dq2, dk2, dv2 = be.attn_bwd(do, q, k, v, o2, lse2, hd ** -0.5, beside_other_streams=True)
    assert rel(dq2.flatten(2, 3), qf.grad) <= TOL and rel(dk2, kf.grad) <= TOL and rel(dv2, vf.grad) <= TOL


def test_attention_does_not_depend_on_the_launch_size(be):
    """Forward and query-gradient kernels come in two variants chosen by workgroup count (forward:
    halves of a workgroup share K / V tiles once there is a 256-query tile for every compute unit;
    query gradient: up to 1024 workgroups each row's keys are split between two halves of a
    workgroup).  Within a variant a sequence gives the same bits whatever the batch around it;
    across variants the results agree to rounding."""
    s, nq, nkv, hd, b = 1024, 8, 2, 128, 17                   # 4 x 8 x 17 = 544 tiles of 256 queries
    q, k, v = rnd(s, b, nq, hd, seed=40), rnd(s, b, nkv, hd, seed=41), rnd(s, b, nkv, hd, seed=42)
    o_all, lse_all = be.attn_fwd(q, k, v, hd ** -0.5)
    o_9, lse_9 = be.attn_fwd(q[:, 4:13].contiguous(), k[:, 4:13].contiguous(), v[:, 4:13].contiguous(), hd ** -0.5)  # 288 tiles
    assert torch.equal(o_all[:, 4:13], o_9) and torch.equal(lse_all[4:13], lse_9)
    for bi in (0, 9, 16):
        o1, lse1 = be.attn_fwd(q[:, bi:bi + 1].contiguous(), k[:, bi:bi + 1].contiguous(),
                               v[:, bi:bi + 1].contiguous(), hd ** -0.5)   # 64 workgroups of 128 queries
        assert rel(o_all[:, bi:bi + 1], o1) <= 1e-2 and rel(lse_all[bi], lse1[0]) <= 1e-5
        o2, lse2 = be.attn_fwd(q[:, bi:bi + 2].contiguous(), k[:, bi:bi + 2].contiguous(),
                               v[:, bi:bi + 2].contiguous(), hd ** -0.5)   # 128 workgroups, same variant
        assert torch.equal(o2[:, :1], o1) and torch.equal(lse2[0], lse1[0])
    ro, rlse = R.causal_gqa_attention(q[:, 3:4].float(), k[:, 3:4].float(), v[:, 3:4].float(), return_lse=True)
    assert rel(o_all[:, 3:4], ro) <= TOL and rel(lse_all[3:4], rlse) <= 1e-4
    # the query-gradient kernel: unsplit variant for the whole batch, split variant for one sequence
    do = rnd(s, b, nq, hd, seed=43)
    dq_all, dk_all, dv_all = be.attn_bwd(do, q, k, v, o_all, lse_all, hd ** -0.5)
    for bi in (0, 16):
        sl = slice(bi, bi + 1)
        one = [t[:, sl].contiguous() for t in (do, q, k, v, o_all)]
        dq1, dk1, dv1 = be.attn_bwd(one[0], one[1], one[2], one[3], one[4], lse_all[sl].contiguous(), hd ** -0.5)
        assert rel(dq_all[:, sl], dq1) <= 1e-2 and rel(dk_all[:, sl], dk1) <= 1e-2 and rel(dv_all[:, sl], dv1) <= 1e-2


@pytest.mark.parametrize("s,b,nq,nkv", [(512, 1, 8, 2), (768, 2, 4, 4), (256, 1, 6, 2), (384, 1, 2, 1), (1024, 1, 24, 8)])
def test_attention_beside_other_streams(be, s, b, nq, nkv):
    """The forms the engine launches on its nanobatch streams (KR_ATTN_BESIDE_OTHER_STREAMS: whole rows and whole
    key tiles per workgroup whatever their number; a length that is not a multiple of 256 keeps the 128-query
    forms): against the fp32 oracle like the default forms, the same bits on every call, and — unlike the default
    forms, which pick a variant by workgroup count — the same bits for a sequence whatever the batch around it."""
    hd = 128
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=222)
    do = rnd(s, b, nq, hd, seed=223)
    o, lse = be.attn_fwd(q, k, v, hd ** -0.5, beside_other_streams=True)
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
    ro.backward(do.float().cpu())
    dq, dk, dv = be.attn_bwd(do, q, k, v, o, lse, hd ** -0.5, beside_other_streams=True)
    assert rel(dq.flatten(2, 3), qf.grad) <= TOL and rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL
    again = be.attn_bwd(do, q, k, v, o, lse, hd ** -0.5, beside_other_streams=True)
    assert all(torch.equal(x, y) for x, y in zip(again, (dq, dk, dv)))
    # against the default forms: equal to rounding
    o0, lse0 = be.attn_fwd(q, k, v, hd ** -0.5)
    assert rel(o, o0) <= 1e-2 and rel(lse, lse0) <= 1e-5
    # a batch of 40 such sequences (enough tiles for every compute unit) gives each of them the same bits
    if s % 256 == 0 and nq == 8:
        big = 40
        qb, kb, vb = (t.repeat_interleave(big, dim=1) for t in (q, k, v))
        ob, lseb = be.attn_fwd(qb, kb, vb, hd ** -0.5, beside_other_streams=True)
        assert torch.equal(ob[:, 7:8], o) and torch.equal(lseb[7:8], lse)
        ob2, _ = be.attn_fwd(qb, kb, vb, hd ** -0.5)            # alone on the GPU it takes the same form
        assert torch.equal(ob2, ob)
        dob = do.repeat_interleave(big, dim=1)
        dqb, dkb, dvb = be.attn_bwd(dob, qb, kb, vb, ob, lseb, hd ** -0.5, beside_other_streams=True)
        assert torch.equal(dqb[:, 7:8], dq)


def test_attention_special_cases(be):
    hd, s = 128, 256
    # all keys equal -> output row i is the mean of v[0..i]
    q = rnd(s, 1, 1, hd, seed=24)
    k = rnd(1, 1, 1, hd, seed=25).expand(s, 1, 1, hd).contiguous()
    v = rnd(s, 1, 1, hd, seed=26)
    o, lse = be.attn_fwd(q, k, v, hd ** -0.5)
    want = torch.cumsum(v.float(), 0) / torch.arange(1, s + 1, device=DEV).view(s, 1, 1, 1)
    assert rel(o, want) <= TOL
    assert torch.equal(o[0], v[0])  # a single visible key: o = v exactly
    # causality: changing later keys/values leaves earlier rows bit-identical
    k2, v2 = k.clone(), v.clone()
    k2[200:] += 1
    v2[200:] -= 3
    o2, _ = be.attn_fwd(q, k2, v2, hd ** -0.5)
    assert torch.equal(o2[:200], o[:200])
    with pytest.raises(RuntimeError, match="not supported"):
        be.attn_fwd(rnd(128, 1, 1, 136), rnd(128, 1, 1, 136), rnd(128, 1, 1, 136), 1.0)  # head_dim above 128


@pytest.mark.parametrize("s,b,nq,nkv", [(512, 2, 4, 2),       # split-key forward (few 256-query tiles)
                                         (512, 64, 8, 2)])     # forward over shared tiles
@pytest.mark.parametrize("kind", ["wide", "rising", "falling"])
def test_attention_when_the_row_maximum_keeps_moving(be, s, b, nq, nkv, kind):
    """The forward kernels move the reference point of a row's exponents only when its maximum has grown
    by more than 2^8.  Scores N(0,1) never do that after the first tile, so: scores spread over +-40
    (jumps of every size), scores that rise along the keys (a new maximum in every tile, by a little or
    by a lot depending on the row) and scores that fall (the first reference stays for good, later
    probabilities underflow).  Checked against the fp32 oracle like every other shape, lse included."""
    hd = 128
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=300)
    q, k = q.clone(), k.clone()
    if kind == "wide":
        k *= 12.0                                         # scores ~ N(0, 12^2): jumps of many powers of two
    else:
        # one shared direction u: score(i, j) = (q_i . u)(k_j . u) + noise, |k_j . u| growing with j
        u = torch.nn.functional.normalize(rnd(hd, seed=301).float(), dim=0).bfloat16()
        ramp = torch.linspace(0.0, 30.0, s, device=DEV).view(s, 1, 1, 1)
        if kind == "falling":
            ramp = -ramp
        k += (ramp * u.float()).bfloat16()
        q += (torch.linspace(0.2, 4.0, s, device=DEV).view(s, 1, 1, 1, 1) * u.float()).bfloat16()
    scale = hd ** -0.5
    o, lse = be.attn_fwd(q, k, v, scale)
    qf, kf, vf = (t.float().cpu() for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    assert torch.isfinite(o.float()).all() and torch.isfinite(lse).all()
    assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
    assert torch.equal(o[0], v[0].repeat_interleave(nq // nkv, dim=1))     # one visible key: o = v exactly


@pytest.mark.parametrize("s,b,nq,nkv,hd", [(100, 1, 1, 1, 128),    # ragged length at the fast kernels' head dimension
                                            (256, 2, 8, 8, 64),     # benchmark configuration 1: 8 heads of 64
                                            (77, 3, 6, 2, 64),      # ragged, grouped queries
                                            (200, 1, 4, 1, 96), (1, 1, 1, 1, 64), (130, 2, 4, 2, 128), (33, 1, 2, 2, 8),
                                            (1000, 2, 8, 2, 128),   # a ragged length at a training width
                                            (640, 2, 8, 8, 64)])    # whole tiles, half the head dimension
@pytest.mark.parametrize("general", [False, True])
def test_attention_general_shapes(be, s, b, nq, nkv, hd, general):
    """Head dimensions other than 128 and sequence lengths that are not whole 128-row tiles: padded into the MFMA
    kernels through the workspace (``general=False``, what the engine runs) or on the general fp32 kernels — same
    interface and layouts (fused QKV views, dense tensors), checked like the fast path."""
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=100)
    do = rnd(s, b, nq, hd, seed=101)
    scale = hd ** -0.5
    attn_fwd = lambda *a: be.attn_fwd(*a, general_kernels=general)
    attn_bwd = lambda *a: be.attn_bwd(*a, general_kernels=general)
    o, lse = attn_fwd(q, k, v, scale)
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
    assert torch.equal(o[0], v[0].repeat_interleave(nq // nkv, dim=1))     # one visible key: o = v exactly
    ro.backward(do.float().cpu())
    dq, dk, dv = attn_bwd(do, q, k, v, o, lse, scale)
    assert all(torch.isfinite(t.float()).all() for t in (o, dq, dk, dv))
    assert rel(dq.flatten(2, 3), qf.grad) <= TOL and rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL
    again = attn_bwd(do, q, k, v, o, lse, scale)                            # fixed order of every sum: same bits
    assert all(torch.equal(x, y) for x, y in zip(again, (dq, dk, dv)))
    qd = q.flatten(2, 3).contiguous()
    od, lsed = attn_fwd(qd, k.contiguous(), v.contiguous(), scale)
    assert torch.equal(od, o) and torch.equal(lsed, lse)


@pytest.mark.parametrize("s,hd", [(256, 64), (200, 64), (200, 128), (64, 96)])
@pytest.mark.parametrize("flags", [None, 0, 0x100])
def test_attention_forward_without_a_workspace_keeps_fp32_probabilities(be, s, hd, flags):
    """``kr_attn_fwd`` and ``kr_attn_fwd_flags`` have no workspace: shapes other than hd = 128 with whole 128-row tiles run
    on the general kernels, bit for bit, also those that the MFMA kernels could take as they lie.  Their only rounding is
    the output's: with V of one sign, so that no sum cancels, o is within half a bf16 step (eight significant bits: at most
    2^-8 of the value) of the exact result, plus what fp32 sums over at most 256 keys and the fast exponential
    leave (1e-4)."""
    _, q, k, v = _grouped(s, 1, 4, 2, hd, seed=130)
    q, k, v = q.flatten(2, 3).contiguous(), k.contiguous(), v.abs().contiguous()
    scale = hd ** -0.5
    o, lse = torch.empty_like(q), torch.empty(1, 4, s, device=DEV)
    strides = (*be._q_strides(q, 2), *be._k_strides(k), *be._k_strides(v), *be._q_strides(o, 2))
    args = (q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(), s, 1, 4, 2, hd, scale, *strides)
    rc = be.lib.kr_attn_fwd(*args, be._stream()) if flags is None else be.lib.kr_attn_fwd_flags(*args, flags, be._stream())
    assert rc == 0
    want_o, want_lse = be.attn_fwd(q, k, v, scale, general_kernels=True)
    assert torch.equal(o, want_o) and torch.equal(lse, want_lse)
    exact = R.causal_gqa_attention(q.double().cpu(), k.double().cpu(), v.double().cpu())
    assert ((o.double().cpu() - exact).abs() / exact).max() <= 2.0 ** -8 + 1e-4


@pytest.mark.parametrize("s,b,nq,nkv,hd", [(1024, 2, 8, 2, 64), (1000, 2, 8, 2, 64), (300, 1, 4, 4, 64), (1000, 1, 8, 2, 128)])
def test_attention_in_place_reserves_and_touches_no_copies(be, s, b, nq, nkv, hd):
    """Shapes that run as they lie: a call allocates its results and the statistics and partial sums of the backward,
    no padded copies (2 MiB: the allocator's rounding); and the backward, in a workspace of just that size, leaves
    what lies behind it alone."""
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=140)
    do, scale = rnd(s, b, nq, hd, seed=141), hd ** -0.5
    w = be.lib.kr_attn_bwd_workspace_bytes_strided(s, b, nq, nkv, hd, max(t.stride(0) for t in (q, k, v, do)))

    def peak(fn):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        got = fn()
        return got, torch.cuda.max_memory_allocated() - before

    (o, lse), used = peak(lambda: be.attn_fwd(q, k, v, scale))
    assert used <= o.numel() * 2 + lse.numel() * 4 + (2 << 20)
    (dq, dk, dv), used = peak(lambda: be.attn_bwd(do, q, k, v, o, lse, scale))
    assert used <= (dq.numel() + dk.numel() + dv.numel()) * 2 + w + (2 << 20)

    ws = torch.full((w + 4096,), 0xA5, dtype=torch.uint8, device=DEV)
    got = [torch.empty(t.shape, dtype=t.dtype, device=DEV) for t in (dq, dk, dv)]
    per = nq // nkv
    rc = be.lib.kr_attn_bwd(do.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr(), lse.data_ptr(),
                            *(t.data_ptr() for t in got), ws.data_ptr(), s, b, nq, nkv, hd, scale, *be._q_strides(q, per),
                            *be._k_strides(k), *be._k_strides(v), *be._q_strides(o, per), *be._q_strides(do, per),
                            *be._q_strides(got[0], per), *be._k_strides(got[1]), *be._k_strides(got[2]), be._stream())
    assert rc == 0 and bool((ws[w:] == 0xA5).all())
    assert all(torch.equal(x, y) for x, y in zip(got, (dq, dk, dv)))


def test_attention_padded_into_the_mfma_kernels_equals_the_whole_tile_call(be):
    """A ragged length is the whole-tile problem with rows taken away: queries below s see the same keys, so the
    padded call must give the bits of the MFMA kernels on the next multiple of 128 restricted to the first s
    rows (forward), and gradients that ignore the rows beyond s."""
    s, sp, b, nq, nkv, hd = 300, 384, 2, 4, 2, 128
    _, q, k, v = _grouped(sp, b, nq, nkv, hd, seed=110)
    scale = hd ** -0.5
    o_full, lse_full = be.attn_fwd(q, k, v, scale)
    o, lse = be.attn_fwd(q[:s], k[:s], v[:s], scale)
    assert torch.equal(o, o_full[:s]) and torch.equal(lse, lse_full[..., :s])
    # backward: the whole-tile call with zero upstream gradient beyond s gives the same dq, dk, dv rows below s
    do_full = rnd(sp, b, nq, hd, seed=111)
    do_full[s:] = 0
    dq_f, dk_f, dv_f = be.attn_bwd(do_full, q, k, v, o_full, lse_full, scale)
    dq, dk, dv = be.attn_bwd(do_full[:s], q[:s], k[:s], v[:s], o, lse, scale)
    assert torch.equal(dq, dq_f[:s]) and torch.equal(dk, dk_f[:s]) and torch.equal(dv, dv_f[:s])


@pytest.mark.parametrize("s,b,nq,nkv,hd", [(8, 1, 2, 1, 64), (127, 1, 2, 2, 64), (128, 1, 2, 1, 64), (129, 2, 4, 1, 64),
                                            (136, 1, 3, 1, 128), (200, 1, 4, 2, 64), (248, 2, 2, 1, 128),
                                            (320, 1, 4, 4, 64), (520, 1, 3, 1, 128), (1000, 2, 32, 8, 64),
                                            (1000, 8, 8, 2, 128), (1024, 2, 32, 8, 64),
                                            # an odd number of 128-row tiles, more than 1024 of them over all heads: dQ
                                            # unsplit in 128-query tiles
                                            (128, 33, 32, 8, 64), (100, 33, 32, 8, 64), (300, 11, 32, 8, 64),
                                            (100, 33, 32, 8, 128), (300, 11, 32, 8, 128), (128, 33, 32, 8, 128)])
@pytest.mark.parametrize("beside", [False, True])
def test_attention_in_place_at_head_dimension_64_and_ragged_lengths(be, s, b, nq, nkv, hd, beside):
    """The MFMA kernels on tensors as they lie: tiles of 128 rows of 64 channels (an odd number of them for the split
    forms, none at all for a part), last tiles that the sequence ends in, every form of every kernel: ``beside`` takes
    the unsplit forward and dK/dV and, at whole 256-query tiles, the dQ kernel of 64 rows per wave, and so do the three
    shapes of 1000 and 1024 without it; dQ in 128-query tiles is split in two at few workgroups and unsplit in
    the last six shapes.  What lies behind the sequence in memory is
    infinite: it must not be read into a result.  Tolerances as for every attention shape (bf16 operands, fp32 sums)."""
    base, q, k, v = _grouped(s + 3, b, nq, nkv, hd, seed=120)
    base[s:] = float("inf")
    q, k, v = q[:s], k[:s], v[:s]
    do_all = rnd(s + 3, b, nq, hd, seed=121)
    do_all[s:] = float("inf")
    do = do_all[:s]
    scale = hd ** -0.5
    o, lse = be.attn_fwd(q, k, v, scale, beside_other_streams=beside)
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
    ro.backward(do.float().cpu())
    dq, dk, dv = be.attn_bwd(do, q, k, v, o, lse, scale, beside_other_streams=beside)
    assert all(torch.isfinite(t.float()).all() for t in (o, lse, dq, dk, dv))
    assert rel(dq.flatten(2, 3), qf.grad) <= TOL and rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL


@pytest.mark.parametrize("s,b,nq,nkv,hd", [(1152, 5, 3, 1, 128),     # 15 pairs of 9 tiles: an XCD's range starts and ends inside a pair
                                           (1152, 5, 3, 1, 64), (904, 7, 2, 2, 128), (136, 1, 2, 1, 128),
                                           (2048, 5, 8, 2, 128),     # more than 64 workgroups per XCD, of at most 16 pairs
                                           (256, 70, 8, 2, 128),     # ... of more pairs
                                           (768, 5, 6, 2, 128), (640, 5, 6, 6, 128),  # few short rows: two workgroups a key tile in groups, one without
                                           (1024, 43, 3, 1, 128),    # 516 workgroups: 65 on four XCDs, 64 on the others, one order on all
                                           (512, 129, 2, 1, 128), (256, 129, 8, 2, 128), (256, 129, 8, 2, 64),
                                           (2048, 4, 8, 2, 128)])    # a 256-query tile for every unit: split forms, two heads per workgroup
def test_attention_over_orders_of_workgroups(be, s, b, nq, nkv, hd):
    """Every tile of every (batch, head) pair is computed once, whatever part of the pairs an XCD has: a tile left out or taken
    twice for another is far outside the tolerance (every tensor is filled before it is written)."""
    _, q, k, v = _grouped(s, b, nq, nkv, hd, seed=140)
    do = rnd(s, b, nq, hd, seed=141)
    scale = hd ** -0.5
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    ro, rlse = R.causal_gqa_attention(qf, kf, vf, return_lse=True)
    ro.backward(do.float().cpu())
    for beside in (False, True):
        trash = [torch.full((s * b * nq * hd * 4,), float("nan"), device=DEV, dtype=torch.bfloat16) for _ in range(2)]
        del trash     # (what the allocator hands out next held NaN)
        o, lse = be.attn_fwd(q, k, v, scale, beside_other_streams=beside)
        assert rel(o, ro) <= TOL and rel(lse, rlse) <= 1e-4
        dq, dk, dv = be.attn_bwd(do, q, k, v, o, lse, scale, beside_other_streams=beside)
        assert rel(dq.flatten(2, 3), qf.grad) <= TOL and rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL


@pytest.mark.parametrize("s,b,nq,nkv", [(256, 1, 2, 1), (384, 1, 2, 2),          # two and three query tiles: the ring of four stages starts
                                        (640, 2, 4, 2), (2048, 8, 2, 1),         # ... and turns over
                                        (1536, 1, 6, 2), (1536, 1, 6, 6),        # few workgroups: two a key tile in groups, one without
                                        (2056, 1, 4, 2), (2304, 1, 2, 2),        # few key tiles, long rows: two workgroups a key tile
                                        (512, 64, 8, 2), (500, 64, 8, 2),        # four heads of a group in one workgroup, whole and ragged
                                        (256, 128, 6, 2)])                       # three
def test_key_value_gradients_at_head_dimension_64(be, s, b, nq, nkv):
    """Each half of a workgroup takes 64 of every 128 queries and the halves' sums are exchanged at the end: every length of the
    loop, several heads per workgroup, partial results and direct ones, against fp32 autograd; the same bits again."""
    _, q, k, v = _grouped(s, b, nq, nkv, 64, seed=130)
    do = rnd(s, b, nq, 64, seed=131)
    o, lse = be.attn_fwd(q, k, v, 0.125)
    qf, kf, vf = (t.float().cpu().clone().requires_grad_(True) for t in (q.flatten(2, 3), k, v))
    R.causal_gqa_attention(qf, kf, vf).backward(do.float().cpu())
    _, dk, dv = be.attn_bwd(do, q, k, v, o, lse, 0.125)
    assert rel(dk, kf.grad) <= TOL and rel(dv, vf.grad) <= TOL
    _, dk2, dv2 = be.attn_bwd(do, q, k, v, o, lse, 0.125)
    assert torch.equal(dk, dk2) and torch.equal(dv, dv2)


# ------------------------------------------------------------------ fused GEMM epilogues
@pytest.mark.parametrize("m,n,k", [(512, 768, 512), (264, 520, 200), (4096, 4096, 1024), (1000, 3072, 640),
                                   (16384, 640, 72)])
def test_gemm_with_fused_residual_equals_gemm_then_add(be, m, n, k):
    """C = bf16(bf16(A.B) + R) in the GEMM's epilogue: the same bits as the GEMM followed by the residual add,
    also with a row-strided residual and a row-strided output (a nanobatch slice of the block's output).
    (The unfused reference runs without split-K, as a fused launch always does: splitting the contraction
    changes the order of the sum.)"""
    x, w = rnd(m, k, seed=80), rnd(n, k, scale=0.05, seed=81)
    res_wide = rnd(m, 2 * n, seed=82)
    res = res_wide[:, n // 2: n // 2 + n] if (n // 2) % 8 == 0 else res_wide[:, :n]
    want = be.add(res.contiguous(), be.linear_fwd(x, w, split_k=None))
    got = be.linear_fwd(x, w, residual=res)
    assert torch.equal(got, want)
    whole = torch.zeros(m, 3 * n, device=DEV, dtype=torch.bfloat16)
    be.linear_fwd(x, w, residual=res, out=whole[:, n:2 * n])
    assert torch.equal(whole[:, n:2 * n], want) and not whole[:, :n].any() and not whole[:, 2 * n:].any()
    assert rel(got, x.float() @ w.float().t() + res.float()) <= TOL
    with pytest.raises(RuntimeError, match="not supported"):   # fused epilogues exist for the forward layout only
        be.gemm(1, rnd(m, n, seed=83), w, m, k, n, residual=rnd(m, k, seed=84))


@pytest.mark.parametrize("m,f,k", [(512, 128, 256), (264, 384, 200), (4096, 3584, 4096), (1000, 1024, 3072),
                                   (16384, 320, 72), (8192, 672, 136), (304, 14336, 64)])
def test_gemm_with_fused_swiglu_equals_gemm_then_swiglu(be, m, f, k):
    """fc1 with the activation in its epilogue: x = A.W^T [m, 2f] and y = silu(x[:, :f]) * x[:, f:] from one
    launch, the same bits as the GEMM followed by the SwiGLU kernel."""
    a, w = rnd(m, k, seed=85), rnd(2 * f, k, scale=0.05, seed=86)
    x_want = be.linear_fwd(a, w, split_k=None)
    y_want = be.swiglu_fwd(x_want)
    y = torch.empty(m, f, device=DEV, dtype=torch.bfloat16)
    x = be.linear_fwd(a, w, swiglu_out=y)
    assert torch.equal(x, x_want) and torch.equal(y, y_want)
    assert rel(y, R.swiglu(a.float() @ w.float().t())) <= TOL
    assert be.can_fuse_swiglu(2 * f)
    with pytest.raises(RuntimeError, match="not supported"):   # no tile width divides 2f = 144: the caller keeps the two launches
        be.linear_fwd(a[:, :k], rnd(2 * 72, k, seed=87), swiglu_out=torch.empty(m, 72, device=DEV, dtype=torch.bfloat16))


def test_gemm_compute_unit_budget_changes_nothing_but_the_launch(be):
    m, n, k = 4096, 3584, 1088
    x, w = rnd(m, k, seed=88), rnd(n, k, scale=0.05, seed=89)
    full = be.linear_fwd(x, w, split_k=None)
    for cus in (1, 64, 200, 256, 1000):
        assert torch.equal(be.linear_fwd(x, w, split_k=False, max_cus=cus), full)


@pytest.mark.parametrize("m,n,k", [(7168, 4096, 256), (7160, 4088, 200), (4096, 7168, 128), (3584, 8192, 72)])
def test_weight_gradient_with_transposed_store(be, m, n, k):
    """A weight gradient whose tile grid fits the device better the other way round (fc1 of workload c4:
    7168 x 4096) is computed as the transposed product with a transposing store; results are those of the
    direct form (which a call that accumulates still takes) and do not depend on the form bit for bit."""
    dy, x = rnd(k, m, scale=0.1, seed=90), rnd(k, n, seed=91)
    ref = dy.float().t() @ x.float()
    got = be.linear_wgrad(dy, x, split_k=None)
    assert rel(got, ref) <= TOL
    direct = be.gemm(2, dy, x, m, n, k, out=torch.zeros(m, n, device=DEV, dtype=torch.bfloat16), accumulate=True,
                     split_k=None)
    assert torch.equal(got, direct)
    wide = torch.zeros(m, n + 64, device=DEV, dtype=torch.bfloat16)        # row-strided output
    be.gemm(2, dy, x, m, n, k, out=wide[:, :n], split_k=None)
    assert torch.equal(wide[:, :n], got) and not wide[:, n:].any()
    assert torch.equal(be.linear_wgrad(dy, x, split_k=None), got)


@pytest.mark.parametrize("m,f,h", [(512, 128, 256), (264, 520, 200), (4096, 3584, 1024), (1000, 1024, 640), (16384, 72, 3072)])
def test_input_gradient_with_fused_swiglu_backward_equals_the_two_kernels(be, m, f, h):
    """fc2's input-gradient GEMM with the SwiGLU backward in its epilogue: dy . W is never written, the
    gradient of the activation's input comes out of the one launch with the bits of the GEMM followed by
    kr_swiglu_bwd."""
    dy, w = rnd(m, h, seed=110), rnd(h, f, scale=0.05, seed=111)        # W_fc2 [hidden, ffn]
    x = rnd(m, 2 * f, seed=112)                                         # the activation's input (fc1's output)
    want = be.swiglu_bwd(be.linear_dgrad(dy, w, split_k=None), x)
    got = be.linear_dgrad(dy, w, swiglu_bwd_x=x)
    assert got.shape == (m, 2 * f) and torch.equal(got, want)
    assert rel(got, R.swiglu_bwd_formula(dy.float() @ w.float(), x.float())) <= TOL
    wide = rnd(m, 2 * f + 16, seed=113)                                 # row-strided activation input
    assert torch.equal(be.linear_dgrad(dy, w, swiglu_bwd_x=wide[:, :2 * f]),
                       be.swiglu_bwd(be.linear_dgrad(dy, w, split_k=None), wide[:, :2 * f].contiguous()))
