"""float32 causal attention at the edges of its tiles and with infinities and NaN.

Tolerance: scores are fp32 sums of D products kept to 2^-24, scaled to log2
units: their error is below e_s = (D + 9) 2^-24 sum |q k| log2(e) D^-1/2, and a
probability's relative error below e_s + 2^-22; numerator and denominator each
add n roundings of 2^-24, so an output is within
(2 max e_s + (2 n + 32) 2^-24) max |v| of the exact one.
"""

import pytest
import torch

from systems_for_llms_amd.attention import causal_prefill

pytestmark = pytest.mark.gpu


def rows_in_float64(q, k, v):
    """Each query over its own keys only, so that later keys cannot touch it."""
    out = torch.empty(q.shape, dtype=torch.float64)
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * q.shape[-1] ** -0.5
    for i in range(q.shape[2]):
        out[:, :, i] = torch.matmul(s[:, :, i:i + 1, :i + 1].softmax(-1), v[:, :, :i + 1].double()).squeeze(2)
    return out


def run(q, k, v):
    b, h, n, d = q.shape
    cache = torch.full((2, b, h, n + 5, d), float("nan"), device="cuda")  # rows past n are never used
    cache[0, :, :, :n], cache[1, :, :, :n] = k.cuda(), v.cuda()
    out = torch.full((b, n, h, d), float("nan"), device="cuda")
    causal_prefill(q.cuda(), cache[0, :, :, :n], cache[1, :, :, :n], out.transpose(1, 2))
    return out.transpose(1, 2).cpu().double()


def inputs(b, h, n, d, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn((b, h, n, d), generator=g) for _ in range(3)]


@pytest.mark.parametrize("d", [16, 32, 64, 128])
@pytest.mark.parametrize("b,h,n", [(1, 1, 1), (2, 3, 31), (1, 2, 33), (3, 1, 64), (1, 5, 65), (2, 2, 97), (1, 9, 200),
                                   (5, 8, 130)])
def test_tile_edges(b, h, n, d):
    q, k, v = inputs(b, h, n, d, 7 * n + d)
    q[:, :, n // 2:] *= 8  # large scores: the running maximum moves
    e_s = ((q.abs() @ k.abs().transpose(-1, -2)).max() * (d + 9) * 2.0 ** -24 * 1.4427 * d ** -0.5).item()
    bound = (2 * e_s + (2 * n + 32) * 2.0 ** -24) * v.abs().max().item()
    assert (run(q, k, v) - rows_in_float64(q, k, v)).abs().max().item() <= bound


@pytest.mark.parametrize("d", [16, 64])
def test_infinities_and_nan_stay_with_their_rows(d):
    """A value at key j reaches the rows from j on as the operation says, and no row before."""
    q, k, v = inputs(2, 3, 140, d, d)
    k[0, 0, 70] = float("inf")           # +-inf or NaN scores
    k[0, 1, 90, 3], q[0, 1, 90:, 3] = float("inf"), -1.0  # -inf scores: the key drops out
    v[0, 2, 50, 5] = float("inf")
    v[1, 0, 139, 0] = float("nan")
    q[1, 1, 20, 1] = float("nan")
    v[1, 2, 100, 2], v[1, 2, 101, 2] = float("inf"), float("-inf")
    got, want = run(q, k, v), rows_in_float64(q, k, v)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    finite = want.isfinite()
    torch.testing.assert_close(got[finite], want[finite], atol=2e-5, rtol=2e-5)


@pytest.mark.parametrize("d", [16, 64, 128])
def test_values_and_queries_near_the_smallest(d):
    """Operands whose 24 bits reach below the smallest bf16 subnormal keep all of them, and one
    admissible key gives its value back bit for bit."""
    q, k, v = inputs(2, 3, 100, d, 5)
    q[0], k[0] = q[0] * 2.0 ** -115, k[0] * 2.0 ** 115
    v[:, 1] *= 2.0 ** -118
    e_s = ((q.abs() @ k.abs().transpose(-1, -2)).max() * (d + 9) * 2.0 ** -24 * 1.4427 * d ** -0.5).item()
    got, want = run(q, k, v), rows_in_float64(q, k, v)
    bound = (2 * e_s + (2 * 100 + 32) * 2.0 ** -24) * v.abs().amax((2, 3), keepdim=True).double()
    assert ((got - want).abs() <= bound).all()
    assert torch.equal(got[:, :, 0], v[:, :, 0].double())
