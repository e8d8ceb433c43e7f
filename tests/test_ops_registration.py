"""The registered operators (oal_amd/ops.py) without a GPU: schemas, fake
kernels (output metadata and argument checks) and tracing of the forward into
a graph of the operator. Runs on fake ROCm tensors, so no
device is touched; the library is loaded only for its size query."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx

from oal_amd import _native, ops


def _lib_or_skip():
    try:
        _native.load_library()
    except RuntimeError as exc:
        pytest.skip(str(exc))


def _fake_inputs(dtype=torch.bfloat16, b=1, hq=14, hkv=2, n=300, dv=64, groups=8):
    dev = "cuda"
    q = torch.empty(b, hq, n, 64, device=dev, dtype=dtype)
    k = torch.empty(b, hkv, n, 64, device=dev, dtype=dtype)
    v = torch.empty(b, hkv, n, dv, device=dev, dtype=dtype)
    labels = torch.zeros(hq, 64, device=dev, dtype=torch.int32)
    c0 = torch.empty(hq, device=dev)
    lam = torch.empty(hq, groups, device=dev)
    gam = torch.empty(hq, groups, groups, device=dev)
    return q, k, v, labels, c0, lam, gam


def test_schemas():
    fwd = str(torch.ops.oal_amd.forward.default._schema)
    bwd = str(torch.ops.oal_amd.backward.default._schema)
    assert fwd == ("oal_amd::forward(Tensor q, Tensor k, Tensor v, Tensor labels, Tensor c0, Tensor lam, "
                   "Tensor gam, float scale, float floor, str precision) -> (Tensor, Tensor, Tensor, Tensor)")
    assert bwd.startswith("oal_amd::backward(Tensor q, Tensor k, Tensor v, Tensor labels, Tensor c0, Tensor lam, "
                          "Tensor gam, Tensor num, Tensor den, Tensor saved, Tensor? dout, Tensor? dnum, "
                          "Tensor? dden, float scale, float floor, bool need_q, bool need_k, bool need_v, "
                          "bool need_coef, str precision)")


@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, "bf16"), (torch.float32, "fp32")])
def test_fake_forward_metadata(dtype, precision):
    _lib_or_skip()
    with FakeTensorMode():
        q, k, v, labels, c0, lam, gam = _fake_inputs(dtype)
        out, num, den, saved = torch.ops.oal_amd.forward(q, k, v, labels, c0, lam, gam, 0.125, 0.0, precision)
        assert out.shape == q.shape and out.dtype == dtype and out.device == q.device
        assert num.shape == q.shape and num.dtype == torch.float32
        assert den.shape == (1, 14, 300, 1) and den.dtype == torch.float32
        assert saved.dtype == torch.uint8 and saved.ndim == 1
    lib = _native.load_library()
    want = lib.oal_forward_saved_bytes(1, 14, 2, 300, 8, _native._dtype_code(dtype), _native._precision_code(precision))
    assert saved.numel() == want


def test_fake_backward_metadata_follows_the_requests():
    _lib_or_skip()
    with FakeTensorMode():
        q, k, v, labels, c0, lam, gam = _fake_inputs()
        out, num, den, saved = torch.ops.oal_amd.forward(q, k, v, labels, c0, lam, gam, 0.125, 0.0, "bf16")
        grads = torch.ops.oal_amd.backward(q, k, v, labels, c0, lam, gam, num, den, saved, out, None, None,
                                           0.125, 0.0, True, False, False, True, "bf16")
        assert [tuple(g.shape) for g in grads] == [tuple(q.shape), (0,), (0,), (14,), (14, 8), (14, 8, 8)]


def test_fake_forward_checks_arguments():
    _lib_or_skip()
    with FakeTensorMode():
        q, k, v, labels, c0, lam, gam = _fake_inputs()
        with pytest.raises(RuntimeError, match="labels must have shape"):
            torch.ops.oal_amd.forward(q, k, v, labels[:, :32], c0, lam, gam, 0.125, 0.0, "bf16")
        with pytest.raises(RuntimeError, match="query head count must be divisible"):
            torch.ops.oal_amd.forward(q[:, :13].contiguous(), k, v, labels[:13], c0[:13], lam[:13], gam[:13],
                                      0.125, 0.0, "bf16")


def test_make_fx_traces_the_forward():
    # (the backward is traced in tests/test_gpu_ops.py: the autograd engine
    # needs a device for ROCm tensors, fake or not)
    _lib_or_skip()

    def fwd(q, k, v, labels, c0, lam, gam):
        return ops.grouped_oal_op(q, k, v, labels, c0, lam, gam, scale=0.125, floor=0.0, precision="bf16")

    with FakeTensorMode():
        gm = make_fx(fwd, tracing_mode="fake")(*_fake_inputs(dv=48))
    targets = [str(n.target) for n in gm.graph.nodes if n.op == "call_function"]
    assert "oal_amd.forward.default" in targets


def test_make_fx_traces_the_factor_expansion():
    """Code above the operators expands a factor or per-pair coefficients in the
    traced function: the graph holds that expansion, on fake tensors as on real ones."""
    from oal_amd.grouped_quadratic import _expand_factor_coefficients
    from oal_amd.hd_block_gemm_autograd import logical_to_grouped

    _lib_or_skip()

    def fwd(q, k, v, labels, factor, a, b, c):
        coef = _expand_factor_coefficients(factor, query_heads=14, gmax=8, kernel_eps=1e-6, working_dtype=torch.float32)
        kw = dict(scale=0.125, floor=0.0, precision="bf16")
        c0, lam, gam, each = logical_to_grouped(a, b, c, 64)
        return ops.grouped_oal_op(q, k, v, labels, *coef, **kw)[0], ops.grouped_oal_op(q, k, v, each, c0, lam, gam, **kw)[0]

    with FakeTensorMode():
        q, k, v, labels, *_ = _fake_inputs()
        small = [torch.empty(s, device="cuda") for s in ((14, 45), (14,), (14, 64), (14, 2080))]
        gm = make_fx(fwd, tracing_mode="fake")(q, k, v, labels, *small)
    inputs = [n for n in gm.graph.nodes if n.op == "placeholder"]
    assert all(n.users for n in inputs)  # none baked in


def test_rotary_heads_of_fake_tensors():
    """A traced layer with an attention of its own sees the rotation's operations."""
    from oal_amd.qwen_oal import rotary_heads

    with FakeTensorMode():
        cos = torch.empty(20, 64, device="cuda")
        turned = rotary_heads(*(torch.empty(2, 20, 64 * h, device="cuda") for h in (14, 2, 2)), cos, cos, 14, 2, 64)
        assert [tuple(t.shape) for t in turned] == [(2, 14, 20, 64), (2, 2, 20, 64), (2, 2, 20, 64)]
