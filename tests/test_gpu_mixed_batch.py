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


def test_group_beyond_32767_workgroups(dev):
    """A second matrix whose first workgroup number (16 rows each) needs all 16 of its bits."""
    print("tall group", flush=True)
    C, R0, R1, N = 256, 16 * 32776, 40, 2
    w0 = dev_t(np.tile(synth(1024, C, 12, 1), R0 // 1024 + 1)[: R0 * 144], dev)
    w1 = dev_t(synth(R1, C, 12, 2), dev)
    xq = ops.q8k_quantize(dev_t(kqq.synthetic_activations(N, C, seed=N), dev))
    y0, y1, ref = (torch.empty((N, r), device=dev) for r in (R0, R1, R1))
    ops.gemv_q8k_multi([(w0, R0, C, 12), (w1, R1, C, 12)], xq, N, [y0, y1])
    ops.gemv_q8k_multi([(w1, R1, C, 12)], xq, N, [ref])
    np.testing.assert_array_equal(host(y1), host(ref))
    np.testing.assert_array_equal(host(y0)[:, 1024:2048], host(y0)[:, :1024])
