"""cl_conv3d_bwd_weight_noalloc names the HIP error that made it fail.  The
failure is one that HIP already holds when the call is made (a device number
past the last, refused on the host): the call's own launches are valid."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


def hip_runtime():
    """the HIP runtime this process has loaded"""
    with open("/proc/self/maps") as f:
        paths = {line.split()[-1] for line in f if "libamdhip64" in line}
    assert len(paths) == 1, paths
    return ctypes.CDLL(paths.pop())


@pytest.mark.parametrize("by", [0, 1])   # 16-byte aligned, and the general kernel's
def test_error_is_named(by):
    import torch
    from citcom_amd.learn import _cl, _p
    L = _cl()
    nv = 5 * 7 * 9
    x = torch.randn((nv * 16 + by,), device="cuda").bfloat16()[by:]
    g = torch.zeros(16 * 27 * 16 + 16, device="cuda")
    args = (_p(x), _p(x), 1, 5, 7, 9, _p(g), None)
    assert L.cl_conv3d_bwd_weight_noalloc(*args) == 0, L.cl_last_error()
    torch.cuda.synchronize()
    hip = hip_runtime()
    hip.hipGetErrorString.restype = ctypes.c_char_p
    rc = hip.hipSetDevice(1 << 20)
    assert rc != 0
    assert L.cl_conv3d_bwd_weight_noalloc(*args) == -1
    msg = L.cl_last_error()
    torch.cuda.synchronize()
    assert hip.hipGetErrorString(rc) in msg and msg.startswith(b"cl_conv3d_bwd_weight_noalloc: "), msg
    # the error is used up: the next call is fine
    assert L.cl_conv3d_bwd_weight_noalloc(*args) == 0, L.cl_last_error()
    torch.cuda.synchronize()
