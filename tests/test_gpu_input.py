"""Device fields handed to a context: copy and check in one pass, for aligned and
unaligned sources and both layouts; the padding cells are neither read into the
field nor checked."""
import numpy as np
import pytest
import torch

from _cases import field, lib_params
from conftest import announce
from prc_d2z import D2Z, D2ZError, DENSE, FUSED_FP32, PADDED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("offset", [0, 1, 2])
@pytest.mark.parametrize("layout", [DENSE, PADDED])
@pytest.mark.parametrize("N", [16, 32, 192])
def test_device_field(N, layout, offset):
    announce(f"device field N={N} layout={layout} offset={offset}")
    f = field(N)
    w = N + 2 if layout == PADDED else N
    buf = torch.full((offset + N * N * w + 3,), float("nan"), device="cuda")
    body = buf[offset:offset + N * N * w].view(N, N, w)
    body[:, :, :N] = torch.from_numpy(f).cuda()
    torch.cuda.synchronize()
    with D2Z(lib_params(N, nscales=2, mode=FUSED_FP32)) as d:
        d.set_delta_device(body.data_ptr(), layout)
        assert np.array_equal(d.delta(), f)
        for cell, value in (((0, 0, 0), float("nan")), ((N - 1, N - 1, N - 1), float("inf")),
                            ((N // 2, 1, N - 1), float("-inf"))):
            keep = body[cell].item()
            body[cell] = value
            torch.cuda.synchronize()
            with pytest.raises(D2ZError, match="NaN or Inf"):
                d.set_delta_device(body.data_ptr(), layout)
            with pytest.raises(D2ZError):  # no field after a refused one
                d.run()
            body[cell] = keep
        torch.cuda.synchronize()
        d.set_delta_device(body.data_ptr(), layout)
        d.run()
        a = d.zreion()
        d.set_delta(f)
        d.run()
        assert np.array_equal(d.zreion(), a)
