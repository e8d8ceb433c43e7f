"""Which route a geometry takes, by the library's own rule.

Short sequences of up to 8 groups are evaluated over token pairs (the direct
route, oal_direct.hip), everything else through the running state. The size
query tells them apart: a direct call saves nothing (256 bytes that nothing
reads). A test that is about the state's kernels asks here, so that a later
shift of the line cannot send it past them unseen."""

import torch

from oal_amd import _native


def takes_state(b, hq, hkv, n, groups, precision, dtype=torch.bfloat16) -> bool:
    size = _native.load_library().oal_forward_saved_bytes(
        b, hq, hkv, n, groups, _native._dtype_code(dtype), _native._precision_code(precision))
    assert size > 0
    return size > 256


def past_the_line(b, hq, hkv, groups, precision, dtype=torch.bfloat16) -> int:
    """The first length 64 c + 37 that goes through the state, as all longer ones do."""
    n = 37
    while not takes_state(b, hq, hkv, n, groups, precision, dtype):
        n += 64
    return n
