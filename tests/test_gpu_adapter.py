"""Factor expansion and the device checks around the operator (oal_adapter.hip).

The expansion and its VJP against the torch formula in float64 (a sum of at
most 65 products: 65 x 6e-8 = 4e-6 in float32, 8e-15 in float64); the label check
against the host's rule on every kind of bad label; the output check on a bad
value at either end of each operand, in whole and in sliced outputs of every type.
"""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 4e-6), (torch.float64, 8e-15)])
@pytest.mark.parametrize("groups,shared", [(1, False), (8, False), (8, True), (22, False), (64, False), (64, True)])
def test_factor_expansion_and_its_vjp(dtype, tol, groups, shared):
    from oal_amd import grouped_quadratic as gq

    dev, hq, side = _dev(), 3, groups + 1
    gen = torch.Generator().manual_seed(groups)
    shape = (side * (side + 1) // 2,) if shared else (hq, side * (side + 1) // 2)
    host = torch.randn(shape, generator=gen, dtype=torch.float64).to(dtype)
    factor = host.to(dev).requires_grad_()
    got = gq._expand_factor_coefficients(factor, query_heads=hq, gmax=groups, kernel_eps=1e-3, working_dtype=dtype)
    ref = host.double().requires_grad_()
    want = gq._expand_factor_coefficients(ref, query_heads=hq, gmax=groups, kernel_eps=1e-3, working_dtype=torch.float64)
    assert torch.equal(got[2], got[2].transpose(-1, -2))
    # positive: a shared factor's gradient of c0 alone is a sum over the heads, and the
    # bound holds relative to the terms' size (of random signs it cancelled to 2e-3 of
    # them once, at an error of 6e-8 of them)
    up = [0.5 + torch.rand(t.shape, generator=gen, dtype=torch.float64) for t in want]
    for name, a, r in zip(("c0", "lam", "gam"), got, want):
        assert a.dtype == dtype
        assert float((a.detach().cpu().double() - r.detach()).norm() / r.detach().norm()) <= tol, name
    for used in ((0, 1, 2), (0,), (1,), (2,)):
        da = torch.autograd.grad([got[i] for i in used], factor, [up[i].to(dev, dtype) for i in used], retain_graph=True)
        dr = torch.autograd.grad([want[i] for i in used], ref, [up[i].to(dtype).double() for i in used], retain_graph=True)
        assert float((da[0].cpu().double() - dr[0]).norm() / dr[0].norm()) <= tol, used


@pytest.mark.parametrize("groups", [1, 8, 22, 64])
@pytest.mark.parametrize("heads", [1, 2, 5, 130])
def test_shared_factor_gradient_over_heads(groups, heads):
    """One factor for all heads: the threads of a row share its heads out (256 / (groups
    + 1) parts at most: more than the heads, and with and without a remainder of
    them). Sums in fp64 of fp32 gradients, rounded once: 2^-24, and each product's
    operands are exact."""
    from oal_amd import _native

    dev, side = _dev(), groups + 1
    gen = torch.Generator().manual_seed(groups + heads)
    packed = torch.randn(side * (side + 1) // 2, generator=gen)
    up = [torch.randn(s, generator=gen) for s in ((heads,), (heads, groups), (heads, groups, groups))]
    got = _native.expand_factor_backward(packed.to(dev), heads, groups, *(t.to(dev) for t in up))
    rows, cols = torch.tril_indices(side, side)
    low = torch.zeros(side, side, dtype=torch.float64)
    low[rows, cols] = packed.double()
    dm = torch.zeros(heads, side, side, dtype=torch.float64)
    dm[:, 0, 0], dm[:, 0, 1:], dm[:, 1:, 1:] = up[0].double(), 2 * up[1].double(), up[2].double()
    want = ((dm + dm.transpose(1, 2)).sum(0) @ low)[rows, cols]
    # rounded to float32 once: half a unit in the last place
    assert float((got.cpu().double() - want).norm() / want.norm()) <= 2.0 ** -24


@pytest.mark.parametrize("d", [1, 5, 48, 64])
def test_pair_expansion_and_its_vjp(d):
    """Copies and sums of two values: the same bits as the indexed assignment."""
    from oal_amd import _native
    from oal_amd.hd_block_gemm_autograd import logical_to_grouped

    dev, hq = _dev(), 3
    gen = torch.Generator().manual_seed(d)
    a, b, c = (torch.randn(s, generator=gen) for s in ((hq,), (hq, d), (hq, d * (d + 1) // 2)))
    c0, lam, gam, labels = logical_to_grouped(a.to(dev), b.to(dev), c.to(dev), d)
    rows, cols = torch.tril_indices(d, d)
    want = torch.zeros(hq, 64, 64)
    want[:, rows, cols] = c
    want[:, cols, rows] = c
    assert torch.equal(c0.cpu(), a) and torch.equal(gam.cpu(), want)
    assert torch.equal(lam.cpu(), torch.nn.functional.pad(b, (0, 64 - d)))
    assert torch.equal(labels.cpu(), torch.arange(64, dtype=torch.int32).expand(hq, -1))
    dgam = torch.randn((hq, 64, 64), generator=gen)
    dc = torch.where(rows == cols, dgam[:, rows, cols], dgam[:, rows, cols] + dgam[:, cols, rows])
    assert torch.equal(_native.expand_pairs_backward(dgam.to(dev), d).cpu(), dc)
    # gradients that autograd is to record: the same values, and the same VJP
    bg, cg = b.to(dev).requires_grad_(), c.to(dev).requires_grad_()
    _, lam_g, gam_g, _ = logical_to_grouped(a.to(dev), bg, cg, d)
    assert torch.equal(gam_g, gam) and torch.equal(lam_g, lam)
    db, dcg = torch.autograd.grad((lam_g.sum(), (gam_g * dgam.to(dev)).sum()), (bg, cg))
    assert torch.equal(dcg.cpu(), dc) and torch.equal(db.cpu(), torch.ones_like(b))
    shared = logical_to_grouped(a.to(dev), b[0].to(dev), c[:1].to(dev), d)
    assert torch.equal(shared[1][2].cpu()[:d], b[0]) and torch.equal(shared[2][2].cpu(), want[0])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,n,hq,hkv", [(1, 1, 1, 1), (2, 7, 14, 2), (3, 65, 4, 4)])
def test_rotary_heads(dtype, b, n, hq, hkv):
    """Against apply_rotary in float64: two products and a sum in fp32 (3 x 6e-8), then
    one rounding to bf16 (2^-9)."""
    from oal_amd.qwen_oal import apply_rotary, rotary_heads, rotary_tables

    dev, tol = _dev(), 2e-7 if dtype == torch.float32 else 2.0 ** -9
    gen = torch.Generator().manual_seed(n)
    leaves = [torch.randn((b, n, h * 64), generator=gen).to(dtype) for h in (hq, hkv, hkv)]
    cos, sin = rotary_tables(n, 64, 1e6, dev, dtype)
    mine = [t.to(dev).requires_grad_() for t in leaves]
    got = rotary_heads(*mine, cos, sin, hq, hkv, 64)
    ref = [t.double().requires_grad_() for t in leaves]
    c64, s64 = cos.cpu().double(), sin.cpu().double()
    heads = [t.view(b, n, h, 64).transpose(1, 2) for t, h in zip(ref, (hq, hkv, hkv))]
    want = [apply_rotary(heads[0], c64, s64), apply_rotary(heads[1], c64, s64), heads[2]]
    up = [torch.randn(t.shape, generator=gen).to(dtype) for t in want]
    for used in ((0, 1, 2), (0,), (1, 2)):
        da = torch.autograd.grad([got[i] for i in used], [mine[i] for i in used], [up[i].to(dev) for i in used],
                                 retain_graph=True)
        dr = torch.autograd.grad([want[i] for i in used], [ref[i] for i in used], [up[i].double() for i in used],
                                 retain_graph=True)
        for a, r in zip(da, dr):
            assert a.is_contiguous() and float((a.cpu().double() - r).norm() / r.norm()) <= tol
    for a, r in zip(got, want):
        assert a.dtype == dtype and a.is_contiguous()
        assert float((a.detach().cpu().double() - r.detach()).norm() / r.detach().norm()) <= tol


def test_rotary_heads_under_tracers_and_twice():
    """What replaces the module's attention may be traced or differentiated twice: the
    rotation is linear, so its gradient's gradient is the rotation again."""
    from torch.fx.experimental.proxy_tensor import make_fx

    from oal_amd.qwen_oal import rotary_heads, rotary_tables

    dev, n = _dev(), 7
    cos, sin = rotary_tables(n, 64, 1e6, dev, torch.float32)
    one, two = ([torch.randn((2, n, h * 64), device=dev) for h in (4, 2, 2)] for _ in range(2))

    def turn(q, k, v):
        return rotary_heads(q, k, v, cos, sin, 4, 2, 64)

    for a, r in zip(make_fx(turn)(*one)(*two), turn(*two)):
        assert torch.allclose(a, r, rtol=1e-6, atol=1e-6)
    leaves = [t.requires_grad_() for t in one]
    up = [torch.randn_like(t).requires_grad_() for t in turn(*two)]
    grads = torch.autograd.grad(turn(*leaves), leaves, up, create_graph=True)
    plain = torch.autograd.grad(turn(*leaves), leaves, [t.detach() for t in up])
    assert all(torch.allclose(a, r, rtol=1e-6, atol=1e-6) for a, r in zip(grads, plain))
    for a, r in zip(torch.autograd.grad(grads, up, two), turn(*two)):
        assert torch.allclose(a, r, rtol=1e-6, atol=1e-6)


def _prefix(row, groups):
    used = sorted(set(row))
    return 1 if any(x < 0 or x >= groups for x in row) else 0 if used == list(range(len(used))) else 2


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
def test_label_check(dtype):
    from oal_amd import _native

    dev = _dev()
    rows = [[0], [1], [0, 1, 2], [0, 2], [2, 2, 2], [-1, 0], [0, 5], [63 - i for i in range(64)], [0] * 63 + [2],
            list(range(63)) + [64], [0, 1 << 30], [3, 2, 1, 0]]
    for row in rows:
        for groups in (1, 3, 5, 64, 100):
            labels = torch.tensor(row, dtype=dtype, device=dev)
            for given, hq in ((labels, 2), (torch.stack([labels, torch.zeros_like(labels)]), 2)):
                verdict = _native.Verdict(dev)
                table = verdict.check_labels(given, hq, groups)
                bits = verdict.read()[0]
                assert bits == _prefix(row, groups), (row, groups, bits)
                if bits == 0:
                    assert table.shape == (hq, 64) and table[0].tolist() == row + [0] * (64 - len(row))


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("shape,width", [((1, 1, 1), 1), ((2, 3, 5), 64), ((2, 3, 5), 17), ((1, 7, 301), 48)])
def test_output_check(out_dtype, wide, shape, width):
    from oal_amd import _native

    dev, dtype = _dev(), torch.float64 if wide else torch.float32
    num = torch.ones((*shape, 64), dtype=dtype, device=dev)[..., :width]
    out = torch.ones((*shape, 64), dtype=out_dtype, device=dev)[..., :width]
    den = torch.ones((*shape, 1), dtype=dtype, device=dev)

    def bits(n=num, d=den, o=out):
        verdict = _native.Verdict(dev)
        verdict.check_outputs(n, d, o)
        return verdict.read()[1]

    assert bits() == 0 and bits(n=num.contiguous(), o=out.contiguous()) == 0 and bits(n=None, o=None) == 0
    for at in (0, -1):
        for value in (float("inf"), float("nan")):
            for sliced in (True, False):
                bad = num.clone() if not sliced else num.new_ones((*shape, 64))[..., :width]
                bad[at, at, at, at] = value
                assert bits(n=bad) == 1
                bad = out.clone() if not sliced else out.new_ones((*shape, 64))[..., :width]
                bad[at, at, at, at] = -value
                assert bits(o=bad) == 4
        for value, want in ((0.0, 2), (-1.0, 2), (float("nan"), 3), (float("inf"), 1), (float("-inf"), 3)):
            bad = den.clone()
            bad[at, at, at] = value
            assert bits(d=bad) == want


def test_errors_come_in_the_reference_order():
    """Bad labels are reported before a bad scale or a size that the kernels refuse."""
    from oal_amd import oal_attention

    dev = _dev()
    q, k, v = (torch.randn(1, 2, 5, 4, device=dev) for _ in range(3))
    factor = torch.eye(3, device=dev)[tuple(torch.tril_indices(3, 3))]
    good, bad = torch.tensor([0, 1, 1, 0], device=dev), torch.tensor([1, 1, 1, 1], device=dev)
    with pytest.raises(ValueError, match="continuous prefix"):
        oal_attention(q, k, v, bad, factor, scale=float("nan"))
    with pytest.raises(ValueError, match="continuous prefix"):
        oal_attention(q, k, torch.randn(1, 2, 5, 70, device=dev), bad, factor)
    with pytest.raises(ValueError, match="scale must be finite"):
        oal_attention(q, k, v, good, factor, scale=float("nan"))
    with pytest.raises(ValueError, match="0 <= id < Gmax"):
        oal_attention(q, k, v, good + 2, factor)
    with pytest.raises(RuntimeError, match="result must be finite"):
        oal_attention(q * float("inf"), k, v, good, factor)


def test_calls_under_a_default_device():
    """torch.device("cuda") as the caller's default moves neither the checks' host words nor any table."""
    from oal_amd import oal_attention
    from oal_amd.hd_block_gemm_adapters import prepare_grouped_hd_block_gemm, run_prepared_grouped_hd_block_gemm

    dev = _dev()
    q, k, v = (torch.randn(1, 2, 70, 64, device=dev) for _ in range(3))
    factor = torch.eye(3, device=dev)[tuple(torch.tril_indices(3, 3))].expand(2, -1).contiguous()
    labels = (torch.arange(64, device=dev) % 2).to(torch.int32)

    def both():
        prepared = prepare_grouped_hd_block_gemm(q, k, v, labels, factor, kernel_eps=1e-6, precision="bf16_tensorcore")
        return oal_attention(q, k, v, labels, factor), run_prepared_grouped_hd_block_gemm(prepared, q, k, v, factor)[0]

    want = both()
    with torch.device("cuda"):
        got = both()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def _expansion(groups=8, heads=2):
    from oal_amd import grouped_quadratic as gq

    gen = torch.Generator().manual_seed(groups)
    factor = torch.randn((heads, (groups + 1) * (groups + 2) // 2), generator=gen).to(_dev())

    def expand(t):
        return gq._expand_factor_coefficients(t, query_heads=heads, gmax=groups, kernel_eps=1e-3, working_dtype=torch.float32)

    return factor, expand


def test_expansion_under_tracers():
    """A traced expansion is the operations, not this call's result: it follows other inputs."""
    from torch.fx.experimental.proxy_tensor import make_fx

    factor, expand = _expansion()
    other = factor.flip(0) + 1
    want = expand(other)
    graphs = [make_fx(expand, tracing_mode=mode)(factor) for mode in ("real", "fake")]
    graphs += [torch.compile(expand, backend="eager", fullgraph=True), torch.jit.trace(expand, factor, check_trace=False)]
    for graph in graphs:
        for a, r in zip(graph(other), want):
            # sums of at most 9 products in float32, where the kernel's are in float64
            assert float((a - r).norm() / r.norm()) <= 9 * 2.0 ** -24


def test_expansion_under_transforms():
    """vmap, forward mode, functorch's grad and a second derivative: M = L L^T is
    quadratic, so its derivative along L itself is twice its value, and the gradient
    of its gradient's sum is a constant."""
    factor, expand = _expansion()
    c0, lam, gam = expand(factor)
    batched = torch.func.vmap(expand)(torch.stack([factor, 2 * factor]))
    assert torch.allclose(batched[2][0], gam, rtol=1e-5, atol=1e-5)
    assert torch.allclose(batched[2][1], 4 * gam, rtol=1e-5, atol=1e-5)
    _, tangent = torch.func.jvp(expand, (factor,), (factor,))
    assert torch.allclose(tangent[2], 2 * gam, rtol=1e-5, atol=1e-5)
    with torch.autograd.forward_ad.dual_level():
        dual = expand(torch.autograd.forward_ad.make_dual(factor, factor))
        assert torch.allclose(torch.autograd.forward_ad.unpack_dual(dual[1]).tangent, 2 * lam, rtol=1e-5, atol=1e-5)
    leaf = factor.clone().requires_grad_()
    up = [torch.randn_like(t) for t in (c0, lam, gam)]
    first = torch.autograd.grad(expand(leaf), leaf, up)[0]
    again = torch.autograd.grad(expand(leaf), leaf, up, create_graph=True)[0]
    assert torch.allclose(again, first, rtol=1e-5, atol=1e-5)
    value = torch.func.grad(lambda t: sum((o * u).sum() for o, u in zip(expand(t), up)))(factor)
    assert torch.allclose(value, first, rtol=1e-5, atol=1e-5)
    # the gradient is linear in the factor and its Jacobian symmetric: applied to the factor it is the gradient
    assert torch.allclose(torch.autograd.grad(again, leaf, factor)[0], first, rtol=1e-5, atol=1e-5)
