"""Gradients of the guiding network at the edges of the kernel's split: part
of a wave's 16 samples, of a chunk's 64, and more chunks than workgroups.
Samples of weight zero change nothing, so a batch filled up with them to
whole chunks has the same gradients bit for bit; and both agree with the
oracle that emulates the kernel's roundings as in test_guide_gpu (FP32
accumulation noise; a misplaced sample moves them by its own size)."""

import numpy as np
import pytest

from test_guide_gpu import batch, compare, emulated_backward, gpu, net, params_for_test  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129, 16385])
def test_gradients_of_partial_chunks(gpu, net, n):  # noqa: F811
    import torch

    params = params_for_test(7)
    net.set_params(gpu.flatten(params))
    full = (n + 63) // 64 * 64
    x, d, t = batch(full, 8)
    t = np.asarray(t).copy()
    t[n:] = 0
    print(f"{n} of {full} samples", flush=True)
    a = net.gradients(x[:n], d[:n], t[:n])
    b = net.gradients(x, d, t)
    assert torch.equal(a, b)
    g = gpu.unflatten(a.cpu().numpy())
    emu = emulated_backward(params, x[:n], d[:n], t[:n])
    for li in range(4):
        for k in range(2):
            cos, rel = compare(g[li][k], emu[li][k])
            assert cos > 0.9995 and rel < 0.03, (li, k, cos, rel)
