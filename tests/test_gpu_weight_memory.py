"""Device memory of a single layer: the copies of its filters that its kernels read, in one allocation of that size."""
import numpy as np
import pytest
import torch

from nncv_amd import abi
from gpu_util import Conv

pytestmark = pytest.mark.gpu

MB = 1 << 20


def taken(make):
    """Bytes of device memory that `make()` keeps."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    layer = make()
    torch.cuda.synchronize()
    used = before - torch.cuda.mem_get_info()[0]
    layer.close()
    return used


# copies of the filters: as rows, for conv_direct, for the patch kernel, for the stream kernel
@pytest.mark.parametrize("dt,C,F,R,stride,copies", [
    (abi.F32, 512, 512, 3, 1, 3),      # rows, direct, patch
    (abi.F32, 512, 512, 3, 2, 2),      # rows, direct
    (abi.F16, 512, 512, 3, 1, 4),      # all of them
    (abi.F16, 512, 512, 3, 2, 3),      # rows, direct, patch
    (abi.F32, 512, 4096, 1, 1, 2),     # rows, direct
    (abi.F16, 64, 65536, 1, 1, 1),     # rows: one round of K never goes to conv_direct
    (abi.F32, 1024, 1024, 5, 1, 2),
])
def test_a_layer_keeps_what_its_kernels_read(dt, C, F, R, stride, copies):
    w = np.zeros((F, C, R, R), abi.np_dtype(dt))
    bn = [np.ones(F, np.float32)] * 4
    make = lambda: Conv(dt, w, stride, R // 2, bn=bn, relu=True)
    make().close()  # (staging memory, code objects)
    used = taken(make)
    filters = w.nbytes
    print("%.1f MB for filters of %.1f MB" % (used / MB, filters / MB), flush=True)
    # scale and shift, and what the driver rounds an allocation up to
    assert copies * filters <= used + MB and used <= copies * filters + 8 * F + 5 * MB
