"""Q4_K and Q6_K matrices of one small-batch call (one launch up to 4096 columns): every row's bits are those of a call
on its matrix and token alone, at the edges of the 16- and 32-row workgroups and of the launch's rule."""
import numpy as np
import pytest
import torch

from kq import ops, quantize as kqq

from test_gpu_kernels import dev_t, host, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,rows", [
    (4096, ((4096, 12), (1024, 12), (1024, 14))),
    (256, ((8, 14), (4104, 12))),
    (3328, ((24, 14), (4096, 12), (40, 14))),       # 13 super-blocks; two Q6_K matrices
    (1024, ((136, 12), (72, 14))),                  # fewer than 4096 Q4_K rows: one launch from 4 tokens
    (512, ((4096, 12), (4096, 14))),                # a Q6_K part that fills the GPU: a launch per type
    (4352, ((4096, 12), (1024, 14))),               # 17 super-blocks: a launch per type
])
def test_mixed_types_small_batch(dev, C, rows):
    mats = [(dev_t(synth(R, C, ty, 50 + i), dev), R, C, ty) for i, (R, ty) in enumerate(rows)]
    x = dev_t(kqq.synthetic_activations(16, C, seed=C), dev)
    one = []
    for w, R, _, ty in mats:
        y = torch.empty((16, R), device=dev)
        for n in range(16):
            ops.gemv_q8k(w, R, C, ty, ops.q8k_quantize(x[n]), 1, y[n])
        one.append(host(y))
    for N in (2, 3, 4, 5, 8, 9, 16):
        print("mixed batch", C, rows, N, flush=True)
        ys = [torch.full((N, R + 8), -9.0, device=dev) for _, R, _, _ in mats]
        ops.gemv_q8k_multi(mats, ops.q8k_quantize(x[:N]), N, ys)
        for (_, R, _, _), y, ref in zip(mats, ys, one):
            np.testing.assert_array_equal(host(y)[:, :R], ref[:N])
            assert np.all(host(y)[:, R:] == -9.0)
