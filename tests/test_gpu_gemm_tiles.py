"""Prefill GEMMs at the edges of every output tile, against float64 products.

Sizes sit at the remainders of the tiles (32, 64 and 128 features by 32 and 64
tokens with K split over the waves; 128 x 64 up to 256 x 384 with shared K
steps): one row, one more or less than a tile, N that is no multiple of 32,
K of one chunk and of fewer chunks than waves.

Tolerance: fp32 sums of K exact 16-bit products in any order differ from the
exact sum by at most (K + 1) 2^-24 sum |a w| (each of at most K additions
rounds a partial sum bounded by sum |a w|), and a 16-bit output by half a unit
in the last place more (2^-8 for bf16, 2^-11 for fp16).
"""

import pytest
import torch

pytestmark = pytest.mark.gpu

HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
SHAPES = [(1, 40, 64), (33, 1000, 192), (65, 1024, 2752), (301, 1024, 1024), (310, 4096, 768), (257, 3080, 1024),
          (301, 5504, 1024), (513, 2688, 512), (1000, 2304, 768), (1025, 10000, 64), (2049, 1024, 192),
          (4100, 2064, 64), (9000, 4100, 64)]


def operands(m, n, k, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.randn((m, k), device="cuda", generator=g).to(dtype)
    w = (torch.randn((n, k), device="cuda", generator=g) * 0.05).to(dtype)
    return a, w


def exact(a, w):
    """The product in float64 and the bound (K + 1) 2^-24 sum |a w| on fp32 sums."""
    a, w = a.double(), w.double().t().contiguous()
    return a @ w, (a.abs() @ w.abs()) * ((a.shape[1] + 1) * 2.0 ** -24)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_plain_and_residual(m, n, k, dtype):
    from systems_for_llms_amd import _lib

    a, w = operands(m, n, k, dtype)
    want, bound = exact(a, w)
    code, st = _lib.dtype_code(dtype), _lib.stream_handle()
    out = torch.full((m, n), float("nan"), device="cuda")
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, code, 0, 0, st)
    assert ((out.double() - want).abs() <= bound).all()
    half = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), half.data_ptr(), m, n, k, code, code, 0, st)
    assert torch.equal(half, out.to(dtype))

    # Residual update that prepares the next norm: x, T(x * gain), sums of x^2 per part.
    x0 = torch.randn((m, n), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    gain = (1 + 0.1 * torch.randn(n, device="cuda", generator=torch.Generator(device="cuda").manual_seed(2))).to(dtype)
    for part in {128, _lib.lib().sfl_gemm_norm_part(m, n, k)}:
        x, act = x0.clone(), torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
        ss = torch.full((-(-n // part), m), float("nan"), device="cuda")
        _lib.call("sfl_gemm_residual_norm_parts", a.data_ptr(), w.data_ptr(), x.data_ptr(), m, n, k, gain.data_ptr(),
                  act.data_ptr(), ss.data_ptr(), part, code, st)
        # x0 takes part in the sum, possibly first: every partial sum grows by up to |x0|.
        assert ((x.double() - (x0.double() + want)).abs() <= bound + x0.double().abs() * ((k + 2) * 2.0 ** -24)).all()
        assert torch.equal(act, (x * gain.float()).to(dtype))
        pad = torch.nn.functional.pad(x.double().square(), (0, -n % part)).view(m, -1, part).sum(-1).t()
        assert ((ss.double() - pad).abs() <= pad * (part + 1) * 2.0 ** -24).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("batch,seq,d,heads,d_ff", [(1, 1, 64, 2, 40), (3, 11, 512, 16, 1344), (1, 301, 1024, 16, 2752),
                                                    (5, 205, 768, 12, 2048), (7, 300, 256, 2, 520), (1, 4097, 128, 2, 1032)])
def test_normed_consumers(batch, seq, d, heads, d_ff, dtype):
    """q/k/v and SwiGLU scaled from the parts of the sum of squares: the bits of the
    given-scale entry points, and those against float64."""
    from systems_for_llms_amd import _lib

    m, dk, cap = batch * seq, d // heads, seq + 3
    a, wqkv = operands(m, 3 * d, d, dtype)
    g = torch.Generator(device="cuda").manual_seed(3)
    parts = torch.rand((d // 32, m), device="cuda", generator=g) * 64
    scale, code, st = torch.empty(m, device="cuda"), _lib.dtype_code(dtype), _lib.stream_handle()
    _lib.call("sfl_norm_scale", parts.data_ptr(), d // 32, m, d, scale.data_ptr(), st)
    angle = torch.rand((dk // 2, cap), device="cuda", generator=g) * 6
    cos, sin = angle.cos(), angle.sin()
    results = []
    for normed in (False, True):
        q = torch.full((batch, heads, seq, dk), float("nan"), device="cuda", dtype=dtype)
        kc, vc = (torch.full((batch, heads, cap, dk), 7.0, device="cuda", dtype=dtype) for _ in range(2))
        lead = (parts.data_ptr(), d // 32) if normed else (scale.data_ptr(),)
        _lib.call("sfl_gemm_qkv_rope_normed" if normed else "sfl_gemm_qkv_rope_scaled", a.data_ptr(), wqkv.data_ptr(),
                  *lead, m, seq, d, heads, cos.data_ptr(), sin.data_ptr(), q.data_ptr(), kc.data_ptr(), vc.data_ptr(),
                  cap, code, st)
        results.append((q, kc, vc))
    for left, right in zip(*results):
        assert torch.equal(left, right)
    q, kc, vc = results[0]
    assert (kc[:, :, seq:] == 7).all() and (vc[:, :, seq:] == 7).all()
    want, bound = exact(a, wqkv)
    want, bound = (y * scale.double()[:, None] for y in (want, bound))
    want, bound = (y.view(batch, seq, 3, heads, dk).permute(2, 0, 3, 1, 4) for y in (want, bound))
    c, s = (t[:, :seq].t().double() for t in (cos, sin))
    for i, got in enumerate((q, kc[:, :, :seq], vc[:, :, :seq])):
        y, tol = want[i], bound[i] + want[i].abs() * 2.0 ** -22
        if i < 2:
            e, o, te, to = y[..., 0::2], y[..., 1::2], tol[..., 0::2], tol[..., 1::2]
            y = torch.stack([e * c - o * s, e * s + o * c], -1).flatten(-2)
            tol = (te + to + 2.0 ** -22 * (e.abs() + o.abs())).repeat_interleave(2, -1)
        assert ((got.double() - y).abs() <= tol + (y.abs() + tol) * HALF_ULP[dtype]).all()

    w13 = operands(m, 2 * d_ff, d, dtype, seed=5)[1]
    h = [torch.full((m, d_ff), float("nan"), device="cuda", dtype=dtype) for _ in range(2)]
    _lib.call("sfl_gemm_swiglu_scaled", a.data_ptr(), w13.data_ptr(), scale.data_ptr(), h[0].data_ptr(), m, d_ff, d,
              code, st)
    _lib.call("sfl_gemm_swiglu_normed", a.data_ptr(), w13.data_ptr(), parts.data_ptr(), d // 32, h[1].data_ptr(), m,
              d_ff, d, code, st)
    assert torch.equal(*h)
    prod, bound = (y * scale.double()[:, None] for y in exact(a, w13))
    (p1, p3), (b1, b3) = ((y.view(m, d_ff // 8, 2, 8).transpose(1, 2).reshape(m, 2, d_ff).unbind(1))
                          for y in (prod, bound))
    want = torch.nn.functional.silu(p1) * p3
    # d silu <= 1.1, |silu(p)| <= |p|; the exponential and reciprocal add a few 2^-23.
    tol = 1.1 * (b1 + 2.0 ** -22 * p1.abs()) * (p3.abs() + b3) + p1.abs() * (b3 + 2.0 ** -20 * p3.abs())
    assert ((h[0].double() - want).abs() <= tol + (want.abs() + tol) * HALF_ULP[dtype] + 2.0 ** -25).all()


# The tiles whose waves share K, with three and five K steps and ragged features and tokens: (features, tokens),
# which the sizes must select.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile,m,n,k", [((128, 64), 2049, 1028, 320), ((128, 128), 8278, 668, 192),
                                        ((256, 256), 9151, 1076, 192), ((256, 384), 9345, 1688, 320)])
def test_plain_and_residual_on_shared_k_tiles(tile, m, n, k, dtype):
    from systems_for_llms_amd import _lib

    assert _lib.gemm_tile(m, n, k) == (*tile, False)
    test_plain_and_residual(m, n, k, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tile,batch,seq,d,heads,d_ff", [((128, 64), 5, 205, 768, 12, 2048),
                                                         ((128, 128), 5, 1966, 192, 3, 344),
                                                         ((256, 256), 17, 641, 384, 6, 536),
                                                         ((256, 384), 31, 339, 576, 9, 840)])
def test_normed_consumers_on_shared_k_tiles(tile, batch, seq, d, heads, d_ff, dtype):
    from systems_for_llms_amd import _lib

    assert _lib.gemm_tile(batch * seq, 3 * d, d, 1) == (*tile, False)
    assert _lib.gemm_tile(batch * seq, 2 * d_ff, d, 2) == (*tile, False)
    test_normed_consumers(batch, seq, d, heads, d_ff, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_rows_of_other_batches_agree_to_rounding(dtype):
    """The order a row's products are added in depends on the tile, so on the rows beside it: equal
    rows agree to twice the bound of any order, not bit for bit; in the same batch size they do."""
    from systems_for_llms_amd import _lib

    a, w = operands(9400, 1688, 1024, dtype)
    want, bound = exact(a[:5], w)
    st, code, outs, tiles = _lib.stream_handle(), _lib.dtype_code(dtype), [], set()
    for m in (5, 301, 1300, 5000, 9400, 9400):
        out = torch.full((m, 1688), float("nan"), device="cuda")
        _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), out.data_ptr(), m, 1688, 1024, code, 0, 0, st)
        outs.append(out[:5])
        if dtype != torch.float32:
            tiles.add(_lib.gemm_tile(m, 1688, 1024))
    assert dtype == torch.float32 or len(tiles) >= 4
    for out in outs:
        assert ((out.double() - want).abs() <= bound).all()
        assert ((out.double() - outs[0].double()).abs() <= 2 * bound).all()
    assert torch.equal(outs[-1], outs[-2])


@pytest.mark.parametrize("m,n,k", [(1, 40, 32), (33, 1000, 96), (65, 512, 1344), (500, 1536, 512), (1000, 520, 64),
                                   (513, 2304, 768), (2049, 1030, 96), (300, 264, 36), (4000, 2312, 32)])
def test_fp32(m, n, k):
    """float32 GEMM at the edges of its tiles, accumulation and SwiGLU included: (K + 9) 2^-24
    sum |a w|, each product off by less than 2^-24 and each addition by half a unit."""
    from systems_for_llms_amd import _lib

    a, w = operands(m, n, k, torch.float32)
    want, bound = exact(a, w)
    bound = bound * (1 + 8 / (k + 1))
    st = _lib.stream_handle()
    x0 = torch.randn((m, n), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    out, x = torch.full((m, n), float("nan"), device="cuda"), x0.clone()
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, 0, 0, 0, st)
    assert ((out.double() - want).abs() <= bound).all()
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), x.data_ptr(), m, n, k, 0, 0, 1, st)
    assert torch.equal(x, x0 + out)
    if n % 16 == 0:
        h = torch.full((m, n // 2), float("nan"), device="cuda")
        _lib.call("sfl_gemm_swiglu", a.data_ptr(), w.data_ptr(), h.data_ptr(), m, n // 2, k, 0, st)
        (p1, p3), (b1, b3) = ((y.view(m, n // 16, 2, 8).transpose(1, 2).reshape(m, 2, n // 2).unbind(1))
                              for y in (want, bound))
        tol = 1.1 * (b1 + 2.0 ** -22 * p1.abs()) * (p3.abs() + b3) + p1.abs() * (b3 + 2.0 ** -21 * p3.abs())
        assert ((h.double() - torch.nn.functional.silu(p1) * p3).abs() <= tol).all()


@pytest.mark.parametrize("m,n,k", [(40, 72, 64), (300, 1040, 96), (1100, 1100, 64)])
def test_fp32_special_values(m, n, k):
    """Infinities and NaN come out as the operation's, values near both ends of the range keep their accuracy."""
    from systems_for_llms_amd import _lib

    a, w = operands(m, n, k, torch.float32)
    a[3, 5], a[17, 9], a[17, 10], w[8, 20] = float("inf"), float("nan"), float("-inf"), float("inf")
    a[20, 1:3], w[:, 20] = float("inf"), w[:, 20].abs()
    w[11, :], w[12, :] = 0.0, 1.0
    a[5], a[6], a[7] = a[5] * 1e-36, a[6] * 1e-30, 2.9e38 / k
    out = torch.full((m, n), 0.0, device="cuda")
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, 0, 0, 0, _lib.stream_handle())
    want = a.double() @ w.double().t().contiguous()
    finite = want.isfinite()
    bound = (a.double().nan_to_num(0, 0, 0).abs() @ w.double().nan_to_num(0, 0, 0).abs().t().contiguous()) \
        * ((k + 9) * 2.0 ** -24) + k * 2.0 ** -126  # products below the normal range may be flushed
    assert ((out.double() - want).abs()[finite] <= bound[finite]).all()
    assert torch.equal(out.isnan(), want.isnan())
    assert torch.equal(out[want.isinf()].double(), want[want.isinf()])


@pytest.mark.parametrize("m,n,k", [(40, 72, 64), (600, 520, 512), (1100, 1100, 96), (3000, 2304, 768)])
@pytest.mark.parametrize("terms", [1, 2, 5])
def test_fp32_sums_of_few_terms(m, n, k, terms):
    """A row with few non-zero values is as exact as fp32 products: each of its T terms is off by
    at most 2^-24 of it (and the partial sums of the smaller pieces by 2^-27 of it), as is each
    of the T additions, half of it on average."""
    from systems_for_llms_amd import _lib

    a, w = operands(m, n, k, torch.float32)
    g = torch.Generator(device="cuda").manual_seed(9)
    keep = torch.zeros_like(a).scatter_(1, torch.rand(a.shape, device="cuda", generator=g).argsort(1)[:, :terms], 1.0)
    a = a * keep
    out = torch.full((m, n), float("nan"), device="cuda")
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, 0, 0, 0, _lib.stream_handle())
    wd = w.double().t().contiguous()
    error, size = out.double() - a.double() @ wd, a.double().abs() @ wd.abs()
    assert (error.abs() <= size * ((2 * terms - 1) * 1.125 * 2.0 ** -24)).all()
    # Uniform mantissas round by 2^-25 sqrt(2/3) rms or less, and to either side.
    relative = error / size
    assert relative.square().mean().sqrt().item() <= (2 * terms - 1) ** 0.5 * 2.0 ** -25
    assert (relative * torch.sign(out)).mean().abs().item() <= 2.0 ** -29


@pytest.mark.parametrize("m,n,k", [(40, 72, 64), (300, 1040, 96), (1100, 1100, 64)])
def test_fp32_operands_near_the_smallest(m, n, k):
    """Operands whose 24 bits reach below the smallest bf16 subnormal keep all of them."""
    from systems_for_llms_amd import _lib

    a, w = operands(m, n, k, torch.float32)
    a[1::2] *= 2.0 ** torch.randint(-124, -108, (m // 2, 1), device="cuda").float()
    w = w * 2.0 ** 30
    out = torch.full((m, n), float("nan"), device="cuda")
    _lib.call("sfl_gemm", a.data_ptr(), w.data_ptr(), out.data_ptr(), m, n, k, 0, 0, 0, _lib.stream_handle())
    want, bound = exact(a, w)
    assert ((out.double() - want).abs() <= bound).all()


def test_part_size_is_checked():
    from systems_for_llms_amd import _lib

    a, w = operands(64, 64, 64, torch.bfloat16)
    x = torch.zeros((64, 64), device="cuda")
    with pytest.raises(RuntimeError, match="part must be"):
        _lib.call("sfl_gemm_residual_norm_parts", a.data_ptr(), w.data_ptr(), x.data_ptr(), 64, 64, 64, w.data_ptr(),
                  a.data_ptr(), x.data_ptr(), 64, 1, _lib.stream_handle())
