"""The direct (token-pair) route and the line between it and the state route, GPU parity.

Short sequences are evaluated over token pairs in 16 x 16 tiles (oal_direct.hip),
longer ones through the running state; direct_route in oal_direct.hpp decides
from the geometry. Against the float64 dense oracle, forward and backward with
every upstream gradient given, at the edges of the tiles and of the steps of 64
rows, with groups of one dimension, of more than 16 (further windows), of none, all
64 in one; one and several query heads per KV head; both input types in both
precisions; and at lengths on the state route's side of the line, ragged, for each
precision. Tolerances are the library's bars, rel-L2 1e-5 in fp32 and 2e-2 in
bf16 mode (operands and pair weights rounded to 8 bits: 2^-9 each, a few of them
in turn), over whole tensors; the three coefficient gradients count as one, since
the constant's is a near-cancelling sum.
"""

import pytest
import torch

from oracle import grouped_oracle as go

pytestmark = pytest.mark.gpu

TOL = {"fp32": 1e-5, "bf16": 2e-2}
SIZES = {
    "uneven": (2, 4, 6, 8, 10, 10, 12, 12),
    "one": (64,),
    "wide": (1, 17, 33, 13),
    "empty": (16, 0, 31, 0, 17),
    "tail": (15, 15, 15, 15, 1, 1, 1, 1),
    "long": (57, 1, 1, 1, 1, 1, 1, 1),
    "second": (6, 22, 6, 6, 6, 6, 6, 6),
}


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def _rel(a, b):
    a, b = a.detach().double().cpu(), b.detach().double().cpu()
    return float((a - b).norm() / b.norm())


def _run(b, hq, hkv, n, sizes, precision, dtype, seed, floor=0.0, only=None, upstream=(True, True, True),
         exact=False):
    from oal_amd import _native

    dev, g = _dev(), len(sizes)
    gen = torch.Generator().manual_seed(seed)
    rounded = (lambda t: t.bfloat16().to(t.dtype)) if exact else (lambda t: t)  # exact: operands that bf16 holds
    q, k, v = (rounded(torch.randn((b, h, n, 64), generator=gen)).to(dtype) for h in (hq, hkv, hkv))
    lab = torch.repeat_interleave(torch.arange(g), torch.tensor(sizes)).to(torch.int32)
    labels = torch.stack([lab[torch.randperm(64, generator=gen)] for _ in range(hq)])
    low = torch.tril(torch.randn((hq, g + 1, g + 1), generator=gen) * 0.15) + torch.diag_embed(
        0.5 + 0.5 * torch.rand((hq, g + 1), generator=gen))
    m = low @ low.transpose(-1, -2)
    m = 0.5 * (m + m.transpose(-1, -2))
    c0, lam, gam = m[:, 0, 0].contiguous() + 1e-3, 2 * m[:, 0, 1:].contiguous(), m[:, 1:, 1:].contiguous()
    scale = 0.125
    args = [t.to(dev) for t in (q, k, v, labels, c0, lam, gam)]
    out, num, den, saved = _native.forward(*args, scale=scale, floor=floor, precision=precision)
    dout = torch.randn(out.shape, generator=gen).to(dtype)
    dnum, dden = rounded(torch.randn(num.shape, generator=gen)), torch.randn(den.shape, generator=gen)
    dout, dnum, dden = (t if given else None for t, given in zip((dout, dnum, dden), upstream))
    need = {**dict(need_q=True, need_k=True, need_v=True, need_coef=True), **(only or {})}
    grads = _native.backward(*args, num, den, saved, *(t if t is None else t.to(dev) for t in (dout, dnum, dden)),
                             scale=scale, floor=floor, precision=precision, **need)
    return (q, k, v, labels, c0, lam, gam, scale), (out, num, den), grads, (dout, dnum, dden)


def _check(case, got, grads, up, tol):
    q, k, v, labels, c0, lam, gam, scale = case
    q64, k64, v64 = (t.double() for t in (q, k, v))
    wq = go.feature_coefficients(labels, c0.double(), lam.double(), gam.double(), scale=scale, head_dim=64)
    out, num, den = go.chunked_forward(q64, k64, v64, wq, chunk=64)
    dq, dk, dv, dwq = go.chunked_backward(q64, k64, v64, wq, num, den, *(t.double() for t in up))
    dc0, dlam, dgam = go.coefficient_gradients_from_wq(dwq, labels, lam.shape[1], scale=scale, head_dim=64)
    dgam = go.symmetrize_gamma_gradient(dgam)

    def whole(c, a, g):
        return torch.cat([c[:, None].cpu(), a.cpu(), g.flatten(1).cpu()], 1)

    errs = {name: _rel(a, r) for name, a, r in zip(("out", "num", "den", "dq", "dk", "dv"), (*got, *grads[:3]),
                                                   (out, num, den, dq, dk, dv))}
    errs["coefficients"] = _rel(whole(*grads[3:]), whole(dc0, dlam, dgam))
    assert torch.equal(grads[5], grads[5].transpose(-1, -2))
    assert all(e <= tol for e in errs.values()), errs


@pytest.mark.parametrize("precision,dtype", [("bf16", torch.bfloat16), ("bf16", torch.float32),
                                             ("fp32", torch.float32), ("fp32", torch.bfloat16)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 130])
def test_tile_edges(precision, dtype, n):
    case, got, grads, up = _run(2, 6, 2, n, SIZES["uneven"], precision, dtype, seed=n)
    assert dtype == torch.float32 or got[0].dtype == torch.bfloat16
    # gradients in a 16-bit type carry their own rounding
    _check(case, got, grads, up, max(TOL[precision], 4e-3 if dtype == torch.bfloat16 else 0.0))


@pytest.mark.parametrize("precision", ["bf16", "fp32"])
@pytest.mark.parametrize("sizes", ["one", "wide", "empty", "tail", "long", "second"])
@pytest.mark.parametrize("hq,hkv", [(1, 1), (9, 1)])
def test_group_windows(precision, sizes, hq, hkv):
    """No further window of a group of more than 16 dimensions, one, two and three of
    them, in one group and in several. (9, 1): more query heads per KV head than the bf16 kernels serve, so fp32 arithmetic in both."""
    case, got, grads, up = _run(1, hq, hkv, 83, SIZES[sizes], precision, torch.float32, seed=len(SIZES[sizes]) + hq)
    _check(case, got, grads, up, TOL["fp32" if hq > 8 else precision])


@pytest.mark.parametrize("precision,b,n", [("bf16", 1, 1411), ("bf16", 1, 1601), ("fp32", 1, 1347), ("fp32", 1, 1603)])
def test_both_sides_of_the_line(precision, b, n):
    """14/2 heads: the first length of each precision is direct, the second goes through the state."""
    from oal_amd import _native

    saved = _native.load_library().oal_forward_saved_bytes(b, 14, 2, n, 8, 0, _native._precision_code(precision))
    assert (saved <= 256) == (n in (1411, 1347))
    case, got, grads, up = _run(b, 14, 2, n, SIZES["uneven"], precision, torch.float32, seed=n)
    _check(case, got, grads, up, TOL[precision])


@pytest.mark.parametrize("precision", ["bf16", "fp32"])
def test_requests_do_not_change_results(precision):
    """Every gradient is the same bits whichever others are requested, and on a rerun."""
    full = _run(1, 4, 2, 70, SIZES["wide"], precision, torch.float32, seed=3)[2]
    again = _run(1, 4, 2, 70, SIZES["wide"], precision, torch.float32, seed=3)[2]
    assert all(torch.equal(a, b) for a, b in zip(full, again))
    off = dict(need_q=False, need_k=False, need_v=False, need_coef=False)
    for on, index in (("need_q", (0,)), ("need_k", (1,)), ("need_v", (2,)), ("need_coef", (3, 4, 5))):
        some = _run(1, 4, 2, 70, SIZES["wide"], precision, torch.float32, seed=3, only={**off, on: True})[2]
        for i in range(6):
            assert (some[i] is not None) == (i in index)
            assert some[i] is None or torch.equal(some[i], full[i])


@pytest.mark.parametrize("n", [1, 16, 33, 64])
@pytest.mark.parametrize("sizes", ["one", "uneven"])
def test_one_chunk_sums_coefficients_in_fp32(n, sizes):
    """Up to 64 tokens in bf16 mode the coefficient sums are those of fp32 pair values.
    With an upstream gradient of den alone every term is exact in its bf16
    operands but for fp32 roundings: a group sum of 64 products, its product with
    ds, the three parts' sum and the sums over pairs, a few 2^-24 each on terms
    whose signs are random. 5e-7 is eight of them (1.3e-7 measured); two parts
    give 2e-6 to 3e-6 for lam and 7e-7 to 2e-6 for gam."""
    case, got, grads, up = _run(2, 4, 2, n, SIZES[sizes], "bf16", torch.bfloat16, seed=n, upstream=(False, False, True))
    q, k, v, labels, c0, lam, gam, scale = case
    wq = go.feature_coefficients(labels, c0.double(), lam.double(), gam.double(), scale=scale, head_dim=64)
    _, num, den = go.chunked_forward(q.double(), k.double(), v.double(), wq, chunk=64)
    dwq = go.chunked_backward(q.double(), k.double(), v.double(), wq, num, den, torch.zeros_like(num),
                              torch.zeros_like(num), up[2].double())[3]
    _, dlam, dgam = go.coefficient_gradients_from_wq(dwq, labels, lam.shape[1], scale=scale, head_dim=64)
    assert _rel(grads[4], dlam) <= 5e-7
    assert _rel(grads[5], go.symmetrize_gamma_gradient(dgam)) <= 5e-7


@pytest.mark.parametrize("n", [16, 130, 800])
@pytest.mark.parametrize("sizes", ["uneven", "tail"])
def test_pair_weights_keep_their_bits(n, sizes):
    """kappa goes into num and dv in two bf16 parts. With operands that bf16 holds
    and an upstream gradient of num alone nothing else is rounded to bf16: 2^-17 =
    7.6e-6 of each term at most (2.6e-6 measured; in one part 1.7e-3)."""
    case, got, grads, up = _run(1, 4, 2, n, SIZES[sizes], "bf16", torch.float32, seed=n, upstream=(False, True, False),
                                exact=True)
    q, k, v, labels, c0, lam, gam, scale = case
    wq = go.feature_coefficients(labels, c0.double(), lam.double(), gam.double(), scale=scale, head_dim=64)
    _, num, den = go.chunked_forward(q.double(), k.double(), v.double(), wq, chunk=64)
    dv = go.chunked_backward(q.double(), k.double(), v.double(), wq, num, den, torch.zeros_like(num), up[1].double(),
                             torch.zeros_like(den))[2]
    assert _rel(got[1], num) <= 7.6e-6
    assert _rel(grads[2], dv) <= 7.6e-6
