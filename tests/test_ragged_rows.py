"""Row kernels on rows whose length or start no 16-byte chunk divides: lengths around every edge at which the
dispatch takes another instantiation, and rows that start at odd elements (column slices of a wider buffer),
with guard elements behind every row that must not change."""
import pytest
import torch

from oracle import ref_torch as R
from tritonformer_amd import _lib
from tritonformer_amd import kernels as K

from tests.util import assert_close, rel_l2

pytestmark = pytest.mark.gpu




def odd_rows(t, dev, fill=7.0):
    """`t` (rows, n) as a view that starts at element 3 of each row of a wider buffer of odd pitch."""
    rows, n = t.shape
    pitch = (n + 5) | 1
    buf = torch.full((rows, pitch), fill, dtype=t.dtype, device=dev)
    view = buf[:, 3:3 + n]
    view.copy_(t)
    return buf, view


def untouched(buf, n, fill=7.0):
    return bool((buf[:, :3] == fill).all() and (buf[:, 3 + n:] == fill).all())


# 64 / 128 / 256 chunks of one wave, 512 / 1024 of a workgroup: one element either side of each edge
@pytest.mark.parametrize("d", [1, 9, 511, 513, 1023, 1025, 2047, 2048, 2049, 4095, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("add", [False, True])
def test_layernorm_rows(d, dtype, add, dev):
    rows = 37
    g = torch.Generator().manual_seed(d)
    x, res, dy, ds = (torch.randn(rows, d, generator=g).to(dtype) for _ in range(4))
    gamma, beta = torch.randn(d, generator=g).to(dtype), torch.randn(d, generator=g).to(dtype)
    lib, st, dt = _lib.load(), _lib.stream_ptr(), _lib.dtype_code(dtype)
    xb, xv = odd_rows(x, dev)
    rb, rv = odd_rows(res, dev)
    gb, gv = odd_rows(dy, dev)
    sb, sv = odd_rows(ds, dev)
    yb, yv = odd_rows(torch.zeros_like(x), dev)
    tb, tv = odd_rows(torch.zeros_like(x), dev)
    ob, ov = odd_rows(torch.zeros_like(x), dev)
    pb, pv = odd_rows(torch.stack([gamma, beta]), dev)
    mean, rstd = torch.empty(rows, device=dev), torch.empty(rows, device=dev)
    dg, db = torch.empty(d, dtype=dtype, device=dev), torch.empty(d, dtype=dtype, device=dev)
    nb = lib.tf_layernorm_bwd_partial_bytes(rows, d)
    part = torch.empty(nb, dtype=torch.uint8, device=dev)
    ptr = lambda t: t.data_ptr()  # noqa: E731
    if add:
        _lib.check(lib.tf_add_layernorm_fwd(st, dt, dt, rows, d, ptr(xv), xv.stride(0), ptr(rv), rv.stride(0), ptr(tv),
                                            tv.stride(0), ptr(pv[0]), ptr(pv[1]), 1e-5, ptr(yv), yv.stride(0), ptr(mean), ptr(rstd)))
        total = (x.float() + res.float()).to(dtype)
        assert torch.equal(tv.cpu(), total) and untouched(tb, d)
        _lib.check(lib.tf_add_layernorm_bwd(st, dt, dt, rows, d, ptr(gv), gv.stride(0), ptr(sv), sv.stride(0), ptr(tv),
                                            tv.stride(0), ptr(pv[0]), ptr(mean), ptr(rstd), ptr(ov), ov.stride(0), ptr(dg),
                                            ptr(db), ptr(part), nb))
    else:
        total = x
        _lib.check(lib.tf_layernorm_fwd(st, dt, dt, rows, d, ptr(xv), xv.stride(0), ptr(pv[0]), ptr(pv[1]), 1e-5, ptr(yv),
                                        yv.stride(0), ptr(mean), ptr(rstd)))
        _lib.check(lib.tf_layernorm_bwd(st, dt, dt, rows, d, ptr(gv), gv.stride(0), ptr(xv), xv.stride(0), ptr(pv[0]), ptr(mean),
                                        ptr(rstd), ptr(ov), ov.stride(0), ptr(dg), ptr(db), ptr(part), nb))
    assert untouched(yb, d) and untouched(ob, d)
    assert_close(yv, R.layer_norm(total, gamma, beta, 1e-5), dtype, "y")
    dx, dgr, dbr = R.layer_norm_bwd(total, gamma, dy, 1e-5)
    # one rounding of a result of order 1 (2^-11, 2^-8); d = 1 and 9 divide by a small variance
    scale = max(1.0, dx.abs().max().item())
    assert_close(ov, dx + ds.float() if add else dx, dtype, "dx", atol=(2e-2 if dtype == torch.float16 else 1.5e-1) * scale)
    lim = 1e-3 if dtype == torch.float16 else 8e-3
    assert rel_l2(db, dbr) < lim and (d == 1 or rel_l2(dg, dgr) < lim)


# edges of the wave-per-row kernels (4096 16-bit, 2048 fp32 elements) and of the workgroup-per-row ones
@pytest.mark.parametrize("n", [1, 7, 513, 2047, 2049, 4097, 32767, 32769, 65535, 65537])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_softmax_rows(n, dtype, dev):
    rows = 9
    g = torch.Generator().manual_seed(n)
    x = (2 * torch.randn(rows, n, generator=g)).to(dtype)
    dy = torch.randn(rows, n, generator=g).to(dtype)
    lib, st, dt = _lib.load(), _lib.stream_ptr(), _lib.dtype_code(dtype)
    xb, xv = odd_rows(x, dev)
    gb, gv = odd_rows(dy, dev)
    yb, yv = odd_rows(torch.zeros_like(x), dev)
    ob, ov = odd_rows(torch.zeros_like(x), dev)
    _lib.check(lib.tf_softmax_fwd(st, dt, rows, n, xv.data_ptr(), xv.stride(0), yv.data_ptr(), yv.stride(0)))
    _lib.check(lib.tf_softmax_bwd(st, dt, rows, n, gv.data_ptr(), gv.stride(0), yv.data_ptr(), yv.stride(0), ov.data_ptr(),
                                  ov.stride(0)))
    assert untouched(yb, n) and untouched(ob, n)
    tol = {torch.float32: dict(atol=1e-6, rtol=1e-4), torch.float16: dict(atol=1e-5, rtol=4e-3),
           torch.bfloat16: dict(atol=1e-5, rtol=2e-2)}[dtype]
    assert_close(yv, R.softmax(x.float()), dtype, "y", **tol)
    assert_close(ov, R.softmax_bwd(yv.detach().float().cpu(), dy.float()), dtype, "dx", atol=tol["atol"] * 10, rtol=tol["rtol"])


def masked_rows(n, dtype, seed):
    """Rows as masking leaves them, and rows whose maximum is of large magnitude."""
    g = torch.Generator().manual_seed(seed)
    lowest = torch.finfo(dtype).min
    rows = [torch.full((n,), lowest)]                                   # masked throughout: uniform
    for fill in (lowest, float("-inf")):
        head, few, most = (2 * torch.randn(n, generator=g) for _ in range(3))
        head[: n // 2] = fill
        few[n // 3 : n // 3 + 24] = fill
        most[torch.arange(n) != n // 3] = fill
        rows += [head, few, most]
    for big in (6e4, -6e4) if dtype == torch.float16 else (1e10, -1e10, 3e38, -3e38):
        one = 2 * torch.randn(n, generator=g)
        one[n // 2] = big
        rows += [torch.full((n,), big), one]
    return torch.stack(rows).to(dtype)


# either side of the wave-per-row kernels' end (4096 16-bit, 2048 fp32 elements), the longest rows of the
# workgroup-per-row ones and those beyond; ragged and whole
@pytest.mark.parametrize("n", [513, 2048, 2049, 4096, 4097, 4104, 32769, 65535, 65536, 65537])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_softmax_of_masked_rows(n, dtype, dev):
    x = masked_rows(n, dtype, n)
    y = K.softmax_fwd(x.to(dev)[None])[0]
    want = torch.softmax(x.double(), -1)
    # fp32 exponentials (relative error below 1e-5 down to exp(-100)) and sums, one rounding of the result
    ulp, least = {torch.float32: (2.0 ** -24, 2.0 ** -126), torch.float16: (2.0 ** -11, 2.0 ** -25),
                  torch.bfloat16: (2.0 ** -8, 2.0 ** -126)}[dtype]
    assert ((y.double().cpu() - want).abs() <= want * (ulp + 1e-5) + least).all()
    dx = K.softmax_bwd(torch.ones_like(y)[None], y[None])
    assert torch.isfinite(dx).all()


# ragged rows whose small probabilities are subnormal numbers
@pytest.mark.parametrize("n", [777, 2049, 4097, 32769, 65537])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_softmax_of_ragged_rows_keeps_subnormal_numbers(n, dtype, dev):
    x = torch.linspace(-100, 0, n).to(dtype).repeat(2, 1)
    y = K.softmax_fwd(x.to(dev)[None])[0].double().cpu()
    want = torch.softmax(x.double(), -1)
    # as in the test above, with two units of the smallest number: those of the exponential and of the quotient
    ulp, least = (2.0 ** -24, 2.0 ** -149) if dtype == torch.float32 else (2.0 ** -8, 2.0 ** -133)
    assert ((want < 2.0 ** -126) & (want > 4 * least)).sum() > n // 50
    assert ((y - want).abs() <= want * (ulp + 1e-5) + 2 * least).all()


# ... and where the upstream gradient, a loss scale, lifts them into the normal numbers of the type
@pytest.mark.parametrize("v", [1001, 50257, 70001])
def test_cross_entropy_gradient_of_ragged_rows_keeps_subnormal_numbers(v, dev):
    x = torch.linspace(-100, 0, v).bfloat16().repeat(2, 1)
    lab, gout = torch.full((2,), v - 1), torch.full((2,), 1024.0, dtype=torch.bfloat16)
    loss, lse, _, _ = K.cross_entropy_fwd(x.to(dev), lab.to(dev))
    grad = K.cross_entropy_bwd(gout.to(dev), x.to(dev), lab.to(dev), lse).double().cpu()
    want = torch.softmax(x.double(), -1)
    assert ((want < 2.0 ** -126) & (want > 2.0 ** -140)).any()
    want[:, v - 1] -= 1.0
    # one rounding of the result, of half the smallest bf16 number (2^-133, over 1024) at least; logarithm and argument of
    # the exponential in fp32; a unit of the subnormal exponential
    assert ((grad / 1024 - want).abs() <= want.abs() * (2.0 ** -8 + 1e-4) + 2.0 ** -144 + 2.0 ** -149).all()


# fp32 results against 64 bits, and against what fp32 operands and results alone cost: the argument of the exponential in
# fp32, exponential and sum exactly rounded.  A fifth above that is left for an exponential of one unit in the last place
# and a sum in pairs (measured 1.07 to 1.13; with serial sums and x * log2e - m * log2e in one step 1.24 to 1.33).
@pytest.mark.parametrize("n", [2051, 4097, 20001, 65535])
def test_softmax_of_long_ragged_rows_loses_nothing_to_its_sums(n, dev):
    x = 2 * torch.randn(1000, n, generator=torch.Generator().manual_seed(n))
    want = torch.softmax(x.double(), -1)
    t = (x - x.amax(-1, keepdim=True)) * torch.tensor(1.4426950408889634)
    e = torch.exp2(t.double()).float()
    least = ((e * (1 / e.double().sum(-1, keepdim=True).float())).double() - want).norm()
    assert (K.softmax_fwd(x.to(dev)[None])[0].cpu().double() - want).norm() < 1.2 * least


# every length of the last chunk of rows that a workgroup holds (4, 8 and 16 chunks per thread; backward operands of the last
# read twice): padded to whole chunks with -inf and zeros, the rows have the same terms
@pytest.mark.parametrize("dtype,n0", [(torch.float16, 4096), (torch.float16, 40000), (torch.bfloat16, 65528), (torch.float32, 2048),
                                      (torch.float32, 16384), (torch.float32, 20000), (torch.float32, 65528)])
def test_softmax_of_long_rows_takes_every_end(dtype, n0, dev):
    lib, st, dt = _lib.load(), _lib.stream_ptr(), _lib.dtype_code(dtype)
    for n in range(n0 + 1, n0 + 8):
        x = torch.randn(3, n, generator=torch.Generator().manual_seed(n)).to(dtype)
        got = []
        for pad in (0, -n % 8):
            wide = torch.cat([x, torch.full((3, pad), float("-inf"), dtype=dtype)], 1)
            dy = torch.cat([x, torch.zeros(3, pad, dtype=dtype)], 1)
            put = (lambda t: t.to(dev)) if pad else (lambda t: odd_rows(t, dev)[1])
            wide, dy, y, dx = put(wide), put(dy), put(torch.zeros_like(wide)), put(torch.zeros_like(wide))
            _lib.check(lib.tf_softmax_fwd(st, dt, 3, n + pad, wide.data_ptr(), wide.stride(0), y.data_ptr(), y.stride(0)))
            if pad:  # the backward of one forward
                got[0] = (got[0][0], y[:, :n].clone(), got[0][1])
                y[:, :n] = got[0][0]
            _lib.check(lib.tf_softmax_bwd(st, dt, 3, n + pad, dy.data_ptr(), dy.stride(0), y.data_ptr(), y.stride(0),
                                          dx.data_ptr(), dx.stride(0)))
            got.append((y[:, :n], dx[:, :n]))
        # the compiler may contract the terms of a sum otherwise in the two kernels: 128 terms of a thread and 10 steps between
        # threads in fp32, twice, sum |y dy| < 6 in the backward, and one rounding of a result (2^-24: a subnormal one of fp16)
        sums, eps = 2 * 138 * 2.0 ** -24, torch.finfo(dtype).eps
        y0, y1, dx0, dx1 = [t.double() for t in (*got[0], got[1][1])]
        assert ((y0 - y1).abs() <= y1 * (sums + eps) + 2.0 ** -24).all(), n
        assert ((dx0 - dx1).abs() <= y0 * 6 * sums + dx1.abs() * eps + 2.0 ** -24).all(), n


# 8 / 16 / 25 chunks of 256 threads in registers (16384, 32768, 51200 entries), then the streaming forward
@pytest.mark.parametrize("v", [1, 9, 16383, 16385, 32769, 50257, 51199, 51201, 70001])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_cross_entropy_rows(v, dtype, dev):
    rows = 11
    g = torch.Generator().manual_seed(v)
    x = torch.randn(rows, v, generator=g).to(dtype)
    lab = torch.randint(0, v, (rows,), generator=g)
    lab[0], lab[1] = 0, v - 1
    lib, st, dt = _lib.load(), _lib.stream_ptr(), _lib.dtype_code(dtype)
    xb, xv = odd_rows(x, dev)
    ob, ov = odd_rows(torch.zeros_like(x), dev)
    fb, fv = odd_rows(torch.zeros_like(x), dev)
    labels = lab.to(dev)
    loss, lse = torch.empty(rows, dtype=dtype, device=dev), torch.empty(rows, device=dev)
    gout = torch.full((rows,), 4.0, dtype=dtype, device=dev)
    _lib.check(lib.tf_cross_entropy_fwd(st, dt, rows, v, xv.data_ptr(), xv.stride(0), 0, 0, labels.data_ptr(), loss.data_ptr(),
                                        lse.data_ptr()))
    _lib.check(lib.tf_cross_entropy_bwd(st, dt, rows, v, xv.data_ptr(), xv.stride(0), 0, 0, labels.data_ptr(), lse.data_ptr(),
                                        gout.data_ptr(), 1, ov.data_ptr(), ov.stride(0), 0))
    assert untouched(ob, v)
    assert_close(loss, R.cross_entropy(x, lab), dtype, "loss", atol=1e-2 if dtype == torch.float16 else 6e-2)
    assert_close(ov, R.cross_entropy_bwd(x, lab, gout.cpu()), dtype, "grad", atol=1e-3, rtol=1e-2)
    # the forward that also writes the gradient: the same bits
    loss2, lse2 = torch.empty_like(loss), torch.empty_like(lse)
    _lib.check(lib.tf_cross_entropy_fwd_grad(st, dt, rows, v, xv.data_ptr(), xv.stride(0), 0, 0, labels.data_ptr(),
                                             loss2.data_ptr(), lse2.data_ptr(), fv.data_ptr(), fv.stride(0), 0, 4.0,
                                             gout.data_ptr()))
    assert torch.equal(fv, ov) and torch.equal(loss, loss2) and torch.equal(lse, lse2) and untouched(fb, v)


@pytest.mark.parametrize("v", [2047, 2048, 2049, 2055, 2112, 50257])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_cross_entropy_gradient_is_the_same_bits_wherever_its_rows_start(v, dtype, dev):
    """The gradient kernel counts its chunks from the line in which a row starts, from the row's start (short rows, in place)
    or over aligned rows: 70 rows of odd pitch start at every element of a line, labels at the ends of the row and of its
    first and last chunks.  The same rows padded with -inf to aligned ones have the same sums and so the same bits."""
    g = torch.Generator().manual_seed(v)
    rows = 70
    x = (2 * torch.randn(rows, v, generator=g)).to(dtype).to(dev)
    at = [0, 1, 7, 8, 63, 64, v - 1, v - 2, v - 8, v - 9]
    labels = torch.tensor([at[i % len(at)] for i in range(rows)], device=dev)
    gout = torch.randn(rows, generator=g).to(dtype).to(dev)
    lse = torch.logsumexp(x.float(), 1)
    wide = (v + 7) // 8 * 8
    aligned = torch.full((rows, wide), float("-inf"), dtype=dtype, device=dev)
    aligned[:, :v] = x

    def run(logits, out):
        _lib.check(_lib.load().tf_cross_entropy_bwd(
            torch.cuda.current_stream().cuda_stream, _lib.dtype_code(dtype), rows, logits.shape[1], logits.data_ptr(), logits.stride(0),
            0, 0, labels.data_ptr(), lse.data_ptr(), gout.data_ptr(), 1, out.data_ptr(), out.stride(0), 0))
        return out

    want = run(aligned, torch.empty_like(aligned))[:, :v]
    buf, view = odd_rows(x, dev)
    out_buf, out = odd_rows(torch.zeros_like(x), dev)
    assert torch.equal(run(view, out), want) and untouched(out_buf, v)
    assert torch.equal(run(x, torch.empty_like(x)), want)
    assert torch.equal(run(view, view), want) and untouched(buf, v)


@pytest.mark.parametrize("v", [2048, 2051, 50257])
def test_cross_entropy_gradient_of_subnormal_probabilities_is_the_same_bits_in_both_ragged_forms(v, dev):
    """Chunks from the line (results of their own) and from the row's start (in place) cut a row differently, and a chunk takes
    the library exponential if one of its elements is subnormal: probabilities on both sides of 2^-126, which two lanes write
    at the ends of a row, lifted into bf16's numbers by the upstream gradient."""
    g = torch.Generator().manual_seed(v)
    rows = 70
    x = -80 - 20 * torch.rand(rows, v, generator=g)
    x[:, v // 2] = 0
    x = x.bfloat16().to(dev)
    labels = torch.tensor([[0, 7, v // 2, v - 8, v - 1][i % 5] for i in range(rows)], device=dev)
    lse = torch.logsumexp(x.float(), 1)
    gout = torch.full((rows,), 2.0 ** 20, dtype=torch.bfloat16, device=dev)

    def run(logits, out):
        _lib.check(_lib.load().tf_cross_entropy_bwd(
            torch.cuda.current_stream().cuda_stream, _lib.dtype_code(torch.bfloat16), rows, v, logits.data_ptr(),
            logits.stride(0), 0, 0, labels.data_ptr(), lse.data_ptr(), gout.data_ptr(), 1, out.data_ptr(), out.stride(0), 0))
        return out

    buf, view = odd_rows(x, dev)
    out_buf, out = odd_rows(torch.zeros_like(x), dev)
    lines = run(view, out).clone()
    want = torch.softmax(x.cpu().double(), 1)
    for end in (slice(0, 8), slice(v - 8, v)):
        assert (want[:, end] < 2.0 ** -126).any() and (want[:, end] > 2.0 ** -126).any()
    assert untouched(out_buf, v) and torch.equal(run(view, view), lines) and untouched(buf, v)
    want[torch.arange(rows), labels.cpu()] -= 1
    # as in the test of subnormal numbers above
    assert ((lines.cpu().double() / 2.0 ** 20 - want).abs() <= want.abs() * (2.0 ** -8 + 1e-4) + 2.0 ** -148).all()


# every length of the last chunk, in the first, an inner and the last of a thread's chunks: the rows padded with -inf to
# whole chunks add zeros to the same sums
@pytest.mark.parametrize("v0", [0, 8, 2040, 4096, 16376, 30000, 51192])
def test_cross_entropy_forward_takes_every_end_of_a_row(v0, dev):
    for v in range(v0 + 1, v0 + 9):
        g = torch.Generator().manual_seed(v)
        x = (2 * torch.randn(3, v, generator=g)).half()
        wide = torch.full((3, (v + 7) // 8 * 8), float("-inf"), dtype=x.dtype)
        wide[:, :v] = x
        labels = torch.tensor([0, v - 1, v // 2], device=dev)
        got = []
        for t in (odd_rows(x, dev)[1], wide.to(dev)):
            loss, lse = torch.empty(3, dtype=x.dtype, device=dev), torch.empty(3, device=dev)
            _lib.check(_lib.load().tf_cross_entropy_fwd(_lib.stream_ptr(), _lib.dtype_code(x.dtype), 3, t.shape[1], t.data_ptr(),
                                                        t.stride(0), 0, 0, labels.data_ptr(), loss.data_ptr(), lse.data_ptr()))
            got.append((loss, lse))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), v


# vocabularies held in registers and streamed (beyond 51200), ragged and whole; the masked tokens fill whole chunks of
# the first ones of a thread, with -inf and with the type's lowest value
@pytest.mark.parametrize("v", [257, 16385, 51199, 51201, 51208, 70001, 128257])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_cross_entropy_of_masked_rows(v, dtype, dev):
    g = torch.Generator().manual_seed(v)
    x = torch.randn(6, v, generator=g)
    for r, fill in enumerate((float("-inf"), torch.finfo(dtype).min)):
        x[3 * r, 64:80] = fill
        x[3 * r + 1, : v - 40] = fill
        x[3 * r + 2, torch.arange(v) % 16 >= 8] = fill
    x = x.to(dtype)
    lab = torch.full((6,), v - 1 - (v - 1) % 16, dtype=torch.int64)
    gout = torch.full((6,), 4.0, dtype=dtype)
    loss, lse, _, _ = K.cross_entropy_fwd(x.to(dev), lab.to(dev))
    grad = K.cross_entropy_bwd(gout.to(dev), x.to(dev), lab.to(dev), lse)
    assert torch.isfinite(loss).all() and torch.isfinite(grad).all()
    assert_close(loss, R.cross_entropy(x, lab), dtype, "loss", atol=1e-2 if dtype == torch.float16 else 6e-2)
    assert_close(grad, R.cross_entropy_bwd(x, lab, gout), dtype, "grad", atol=1e-3, rtol=1e-2)
    _, _, both = K.shifted_cross_entropy_fwd_grad(x.to(dev).repeat_interleave(2, 0).view(6, 2, v), lab.to(dev)[:, None].expand(6, 2), 4.0)
    assert torch.equal(both[:, 0], grad)


@pytest.mark.parametrize("rows,cols", [(1, 1), (33, 7), (100, 255), (70, 257), (513, 1733), (97, 512)])
def test_column_sums_and_relu_mask_rows(rows, cols, dev):
    g = torch.Generator().manual_seed(cols)
    x, act = torch.randn(rows, cols, generator=g).half(), torch.randn(rows, cols, generator=g).half()
    lib, st, dt = _lib.load(), _lib.stream_ptr(), _lib.dtype_code(torch.float16)
    xb, xv = odd_rows(x, dev)
    ab, av = odd_rows(act, dev)
    ob, ov = odd_rows(torch.zeros_like(x), dev)
    out = torch.empty(cols, device=dev)
    nb = lib.tf_colsum_partial_bytes(rows, cols)
    part = torch.empty(nb, dtype=torch.uint8, device=dev)
    _lib.check(lib.tf_colsum(st, dt, _lib.TF_F32, rows, cols, xv.data_ptr(), xv.stride(0), out.data_ptr(), part.data_ptr(), nb))
    # sums of `rows` values of order 1 in fp32, in another order
    assert (out.cpu() - x.double().sum(0)).abs().max() < 1e-6 * rows + 1e-6
    _lib.check(lib.tf_relu_mask(st, dt, rows, cols, xv.data_ptr(), xv.stride(0), av.data_ptr(), av.stride(0), ov.data_ptr(),
                                ov.stride(0)))
    assert torch.equal(ov.cpu(), torch.where(act > 0, x, torch.zeros_like(x))) and untouched(ob, cols)
    assert torch.equal(K.mask_grad(xv, av), ov)
    # mask and sums in one pass: the bits of the two passes, from odd and from whole rows
    _lib.check(lib.tf_colsum(st, dt, _lib.TF_F32, rows, cols, ov.data_ptr(), ov.stride(0), out.data_ptr(), part.data_ptr(), nb))
    fb, fv = odd_rows(torch.zeros_like(x), dev)
    sums = torch.empty(cols, device=dev)
    _lib.check(lib.tf_relu_mask_colsum(st, dt, _lib.TF_F32, rows, cols, xv.data_ptr(), xv.stride(0), av.data_ptr(),
                                       av.stride(0), fv.data_ptr(), fv.stride(0), sums.data_ptr(), part.data_ptr(), nb))
    assert torch.equal(fv, ov) and torch.equal(sums, out) and untouched(fb, cols)
    for a, b in [(xv, av), (xv.contiguous(), av.contiguous())]:
        masked, s = K.mask_grad_sums(a, b, torch.float32)
        assert torch.equal(masked, ov) and torch.equal(s, out)


# either side of the tile edges (128, 256) and of one, two and three 64-wide stages, alone and in slices; rows shorter
# than a chunk; operands and result start at odd elements, what lies behind the operands' rows is NaN
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (5, 3, 63), (3, 9, 130), (129, 257, 64), (255, 130, 65), (257, 127, 129),
                                   (130, 260, 200), (33, 300, 385)])
@pytest.mark.parametrize("cfg,splits", [(0, 1), (1, 1), (0, 2), (1, 3)])
@pytest.mark.parametrize("la,lb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_register_staged_gemm(m, n, k, cfg, splits, la, lb, dev):
    dtype = torch.float16 if (m + n + k) % 2 else torch.bfloat16
    g = torch.Generator().manual_seed(m * 1000 + n * 10 + k)
    a, b = torch.randn(m, k, generator=g).to(dtype), torch.randn(k, n, generator=g).to(dtype)
    bias = torch.randn(1, n, generator=g).to(dtype)
    _, av = odd_rows(a if la == _lib.KMAJOR else a.t(), dev, float("nan"))
    _, bv = odd_rows(b.t() if lb == _lib.KMAJOR else b, dev, float("nan"))
    _, biasv = odd_rows(bias, dev, float("nan"))
    diag, st, dt = _lib.load_diag(), _lib.stream_ptr(), _lib.dtype_code(dtype)
    nb = diag.tf_diag_gemm_workspace_bytes(cfg, splits, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device=dev)
    exact = a.double() @ b.double()
    sums = (a.double().abs() @ b.double().abs()) * (k * 2.0 ** -24)  # fp32 sums in any order
    for out, with_bias, dense in ((dtype, True, False), (torch.float32, False, False), (dtype, False, True)):
        if dense:
            cb, cv = None, torch.zeros(m, n, dtype=out, device=dev)
        else:
            cb, cv = odd_rows(torch.zeros(m, n, dtype=out), dev)
        _lib.check(diag.tf_diag_gemm(st, cfg, splits, 0, dt, _lib.dtype_code(out), la, lb, m, n, k, av.data_ptr(),
                                     av.stride(0), bv.data_ptr(), bv.stride(0), cv.data_ptr(), cv.stride(0),
                                     biasv.data_ptr() if with_bias else None, int(with_bias), ws.data_ptr(), nb))
        want = (exact + bias.double()).clamp_min(0) if with_bias else exact
        # the result's own rounding: half a unit in the last place (of the smallest normal number below it)
        ulp = {torch.float16: (2.0 ** -11, 2.0 ** -25), torch.bfloat16: (2.0 ** -8, 1e-30), torch.float32: (2.0 ** -24, 1e-30)}[out]
        bound = sums + (want.abs() + sums) * ulp[0] + ulp[1] + 1e-7 * with_bias
        assert ((cv.double().cpu() - want).abs() <= bound).all()
        assert dense or untouched(cb, n)


# operands whose contraction is strided and whose rows are shorter than a chunk, dense (pitch 1 to 7): no stage goes
# untested then, over one to seven stages, whole and in slices
@pytest.mark.parametrize("m,n", [(1, 1), (3, 5), (7, 7), (5, 300), (257, 3)])
@pytest.mark.parametrize("k", [65, 130, 200, 385])
@pytest.mark.parametrize("cfg,splits", [(0, 1), (1, 1), (0, 2), (1, 3)])
def test_register_staged_gemm_of_rows_shorter_than_a_chunk(m, n, k, cfg, splits, dev):
    g = torch.Generator().manual_seed(m * 1000 + n * 10 + k)
    a, b = torch.randn(m, k, generator=g).half(), torch.randn(k, n, generator=g).half()
    diag, st, dt = _lib.load_diag(), _lib.stream_ptr(), _lib.dtype_code(torch.float16)
    nb = diag.tf_diag_gemm_workspace_bytes(cfg, splits, m, n, k)
    ws = torch.empty(max(nb, 16), dtype=torch.uint8, device=dev)
    exact = a.double() @ b.double()
    bound = (a.double().abs() @ b.double().abs()) * (k * 2.0 ** -24) + exact.abs() * 2.0 ** -24  # fp32 sums in any order
    for la, lb in ((1, 1), (0, 1), (1, 0)):
        # behind the last row lies NaN, which a read past it would bring into a sum
        av, bv = ((torch.cat([t.flatten(), torch.full((64,), float("nan"), dtype=t.dtype)]).to(dev), t.shape[1])
                  for t in (a.t().contiguous() if la else a, b if lb else b.t().contiguous()))
        cb, cv = odd_rows(torch.zeros(m, n), dev)
        _lib.check(diag.tf_diag_gemm(st, cfg, splits, 0, dt, _lib.TF_F32, la, lb, m, n, k, av[0].data_ptr(), av[1],
                                     bv[0].data_ptr(), bv[1], cv.data_ptr(), cv.stride(0), None, 0, ws.data_ptr(), nb))
        assert ((cv.double().cpu() - exact).abs() <= bound).all() and untouched(cb, n)


# the chunk that crosses the end of a row holds r elements of it; alone, behind one whole chunk, behind many
@pytest.mark.parametrize("r", range(1, 8))
def test_row_kernels_at_every_remainder_of_a_chunk(r, dev):
    for n in (r, 8 + r, 640 + r):
        for dtype in (torch.float16, torch.bfloat16):
            if n > 3:  # (the variance of up to three elements may be of any smallness)
                test_layernorm_rows(n, dtype, False, dev)
                test_layernorm_rows(n, dtype, True, dev)
            test_cross_entropy_rows(n, dtype, dev)
        for dtype in (torch.float16, torch.bfloat16, torch.float32):
            test_softmax_rows(n, dtype, dev)
        test_column_sums_and_relu_mask_rows(33, n, dev)
    test_layernorm_rows(2048 + r, torch.float16, True, dev)
    test_softmax_rows(4096 + r, torch.float16, dev)
    test_cross_entropy_rows(51200 + r, torch.float16, dev)


# a NaN or an infinity stays in its row (and its column, where a kernel sums over rows): what is fetched beyond the end of
# a row, or twice, belongs to no result
@pytest.mark.parametrize("n", [33, 65, 519, 1021, 2051, 4099])
def test_non_finite_values_stay_in_their_rows(n, dev):
    g = torch.Generator().manual_seed(n)
    x, dy = (torch.randn(1, 13, n, generator=g).half().to(dev) for _ in range(2))
    gamma, beta = (torch.randn(n, generator=g).half().to(dev) for _ in range(2))
    lab = torch.randint(0, n, (13,), generator=g).to(dev)
    bad = x.clone()
    bad[0, 3, n - 1], bad[0, 7, 0], bad[0, 12, n - 1] = float("nan"), float("inf"), float("inf")
    keep = [r for r in range(13) if r not in (3, 7, 12)]

    def outcomes(t):
        y, mean, rstd = K.layernorm_fwd(t, gamma, beta, 1e-5)
        total, z, _, _ = K.add_layernorm_fwd(t, dy, gamma, beta, 1e-5)
        s = K.softmax_fwd(t)
        loss, lse, _, _ = K.cross_entropy_fwd(t[0], lab)
        ds = K.softmax_bwd(dy, s)
        dl = K.cross_entropy_bwd(torch.ones_like(loss), t[0], lab, lse)
        return [y[0], K.layernorm_bwd(dy, t, gamma, mean, rstd)[0][0], total[0], z[0], s[0], ds[0], loss[:, None], dl]

    for a, b in zip(outcomes(bad), outcomes(x)):
        assert torch.equal(a[keep], b[keep]) and torch.isfinite(a[keep]).all()
    # ReLU mask and its column sums: an activation that is NaN is not positive
    act = bad.clone()
    act[0, 5, n - 1] = 1.0
    grad = dy.clone()
    grad[0, 5, n - 1] = float("nan")
    masked, sums = K.mask_grad_sums(grad, act, torch.float32)
    assert masked[0, 3, n - 1] == 0 and torch.isnan(sums[n - 1]) and torch.isfinite(sums[: n - 1]).all()
    # products: the last row of A and the last column of B, which lie at the edges of their tiles
    b = torch.randn(n, 67, generator=g).half().to(dev)
    worse = b.clone()
    worse[0, 66] = float("inf")
    out, want = K.gemm(bad, worse), K.gemm(x, b)
    assert torch.equal(out[0, keep, :66], want[0, keep, :66]) and not torch.isfinite(out[0, 3]).any()
    assert not torch.isfinite(out[0, :, 66]).any()
