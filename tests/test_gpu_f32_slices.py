"""The fp32 backward's key side in three slices of the state, GPU parity.

Up to f32_sliced's size (oal_internal.hpp) the dk and dv kernels walk the state's
tiles in three blocks each and a sum kernel adds the parts and the heads' local
terms; above it in one. Against the float64 oracle on both sides of the line, at
ragged lengths, with several query heads per KV head and both input types, on the
state route's side of the direct route's line. Tolerance: the library's fp32 bar,
rel-L2 1e-5 (4e-3 where the gradients themselves are stored in bf16, 2^-8).
"""

import pytest
import torch

from test_gpu_direct import SIZES, _check, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,hq,hkv,n,dtype", [
    (1, 2, 2, 5120, torch.float32),  # 160 blocks: the last sliced size
    (1, 2, 2, 5121, torch.float32),  # 162: in one
    (1, 14, 2, 1601, torch.float32),
    (2, 6, 2, 1603, torch.bfloat16),
    (1, 9, 1, 4031, torch.float32),
])
def test_key_side_slices(b, hq, hkv, n, dtype):
    case, got, grads, up = _run(b, hq, hkv, n, SIZES["uneven"], "fp32", dtype, seed=n)
    _check(case, got, grads, up, 4e-3 if dtype == torch.bfloat16 else 1e-5)


@pytest.mark.parametrize("key,value", [(True, False), (False, True)])
def test_one_of_dk_and_dv(key, value):
    """The gradient that is asked for alone has the same bits as with the other."""
    args = (1, 14, 2, 1700, SIZES["uneven"], "fp32", torch.float32)
    both = _run(*args, seed=3)[2]
    only = dict(need_q=False, need_k=key, need_v=value, need_coef=False)
    alone = _run(*args, seed=3, only=only)[2]
    i = 1 if key else 2
    assert alone[3 - i] is None
    assert torch.equal(alone[i], both[i])
