"""Host paths around the sizes where their transfers change: a copy kernel up to
1 MiB, chunks of at least 2 MiB shared with helper threads above (at most eight).
The output must be the device-resident run's, whatever the size and the rows'
stride."""

from __future__ import annotations

import numpy as np
import pytest

from arthip_amd import models, vs
from arthip_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _device_run(e, x):
    import torch
    out = torch.empty(e.output_shape(x.shape), dtype=torch.float16, device="cuda")
    e.run_device(torch.from_numpy(x).cuda(), out)
    torch.cuda.synchronize()
    return out.cpu().numpy()


# Output bytes 8 h w: just below, at and above 1 MiB; two chunks; an odd size; the
# eight-chunk cap.
@pytest.mark.parametrize("h,w", [(256, 511), (256, 512), (256, 513), (512, 1025), (733, 1011), (1440, 1600)])
def test_run_equals_run_device(h, w):
    x = models.synthetic_input((1, 1, h, w), seed=6)
    with Engine(0) as e:
        e.build(models.c4f32(seed=1))
        want = _device_run(e, x)
        np.testing.assert_array_equal(e.run(x), want)
        np.testing.assert_array_equal(e.run(x[:, :, ::-1].copy()), _device_run(e, x[:, :, ::-1].copy()))


@pytest.mark.parametrize("h,w", [(256, 511), (256, 513), (733, 1011), (1080, 1920)])
def test_filter_rows(h, w):
    spec = models.c4f32(seed=1)
    x = models.synthetic_input((1, 1, h, w), seed=7)
    with Engine(0) as e:
        want = _device_run(e.build(spec), x)[0, 0]
    with vs.Model("GRAYH", w, h, spec.bytes()) as m:
        for pad in (0, 5):
            (y,) = m.get_frame([x[0, 0]], out_row_pad=pad)
            np.testing.assert_array_equal(y.view(np.uint16), want.view(np.uint16))


# Uploads of 2 h w bytes with several callers: below 256 KiB always by kernel;
# up to 1 MiB by kernel or on the copy stream, as other frames are in flight or not;
# above on the copy stream.
@pytest.mark.parametrize("h,w", [(250, 511), (256, 513), (480, 853), (733, 1011)])
def test_filter_with_several_callers(h, w):
    from concurrent.futures import ThreadPoolExecutor
    spec = models.c4f32(seed=1)
    xs = [models.synthetic_input((1, 1, h, w), seed=s) for s in range(5)]
    with Engine(0) as e:
        e.build(spec)
        want = [_device_run(e, x)[0, 0].view(np.uint16) for x in xs]
    with vs.Model("GRAYH", w, h, spec.bytes()) as m, ThreadPoolExecutor(4) as pool:
        got = list(pool.map(lambda i: m.get_frame([xs[i % 5][0, 0]])[0].view(np.uint16), range(40)))
    for i, y in enumerate(got):
        np.testing.assert_array_equal(y, want[i % 5])
