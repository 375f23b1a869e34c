"""The prefill GEMM of at most 64 tokens (gemm_small.hip): every edge of its tiles (32-token and 32-row tiles, the K
waves' and the split's shares of 1..17 super-blocks) against the oracle, the three entry points against one another."""
import numpy as np
import pytest
import torch

from kq import ops, quantize as kqq

from test_gpu_kernels import assert_close_inf, dev_t, host, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ty", [12, 14])
@pytest.mark.parametrize("R,C,M", [
    (8, 256, 1), (8, 256, 64),              # one 8-row tile, one super-block: the second K wave has none
    (40, 768, 31), (32, 512, 32),           # one tile of tokens, partly and wholly filled; rows past one row wave
    (136, 1280, 33), (264, 768, 40),        # two tiles, the second nearly empty; the last row wave past R
    (1032, 4352, 63), (512, 4096, 64),      # K split (17 super-blocks in unequal shares)
    (8, 61440, 17),                         # the widest matrix
    (200, 512, 65),                         # one token past the range
])
def test_gemm_few_tokens(dev, orc, ty, R, C, M):
    print("gemm small", ty, R, C, M, flush=True)
    W = synth(R, C, ty, R + M)
    X = kqq.synthetic_activations(M, C, seed=R + C + M)
    xq = orc.quantize_q8k(X)
    ref = orc.gemv_q8k(W, R, C, ty, xq, M)      # assert_close_inf's 1e-5 is the kernels' contract for any sum order
    wd, xqd = dev_t(W, dev), dev_t(xq, dev)
    direct = torch.full((M, R + 8), -3.0, device=dev)
    ops.gemm_q8k(wd, R, C, ty, xqd, M, direct, R + 8)
    ws = torch.full((M, R + 8), -4.0, device=dev)
    ops.gemm_q8k(wd, R, C, ty, xqd, M, ws, R + 8, ws=ops.gemm_workspace(R, C, M, dev))
    assert np.all(host(direct)[:, R:] == -3.0) and np.all(host(ws)[:, R:] == -4.0)
    assert_close_inf(host(direct)[:, :R], ref)
    assert_close_inf(host(ws)[:, :R], ref)
    if ops.gemm_workspace_bytes(R, C, M) == -(-M // 256) * 256 * C:     # no K split: one order of the sums
        np.testing.assert_array_equal(host(ws)[:, :R], host(direct)[:, :R])
    # a group of this matrix, a taller one and one of the other type, from fp32 rows: the same bits
    mats = [(wd, R, C, ty), (dev_t(synth(R + 512, C, ty, 3), dev), R + 512, C, ty),
            (dev_t(synth(16, C, 26 - ty, 4), dev), 16, C, 26 - ty)]
    ys = [torch.empty((M, m[1]), device=dev) for m in mats]
    buf = torch.empty(ops.gemm_f32_multi_workspace_bytes([m[1] for m in mats], C, M) + 256, dtype=torch.uint8, device=dev)
    ops.gemm_f32_multi(mats, dev_t(X, dev), ys, buf)
    np.testing.assert_array_equal(host(ys[0]), host(ws)[:, :R])


@pytest.mark.parametrize("C,M,rows", [
    (4096, 65, (4096, 1024, 1024)),             # smallest chunk of the tile kernels, K split
    (2048, 200, (72, 1032, 8)),                 # ragged tiles
    (512, 300, (264, 136, 5000)),               # the Q6_K part largest
    (256, 4096, (64, 64, 1024)),                # 16 x 32 Q6_K tiles fill the GPU: launches of their own
])
def test_gemm_both_types_in_one_launch(dev, orc, C, M, rows):
    """Q4_K, Q4_K and Q6_K matrices in one call, in any order: each the bits of a call of its own."""
    print("gemm mixed", C, M, rows, flush=True)
    mats = [(dev_t(synth(R, C, ty, 20 + i), dev), R, C, ty) for i, (R, ty) in enumerate(zip(rows, (12, 12, 14)))]
    xqd = dev_t(orc.quantize_q8k(kqq.synthetic_activations(M, C, seed=M)), dev)
    ref = []
    for w, R, _, ty in mats:
        y = torch.empty((M, R), device=dev)
        ops.gemm_q8k(w, R, C, ty, xqd, M, y, ws=ops.gemm_workspace(R, C, M, dev))
        ref.append(host(y))
    for order in ((0, 1, 2), (2, 0, 1), (1, 2)):
        sub = [mats[i] for i in order]
        ys = [torch.full((M, m[1] + 4), -7.0, device=dev) for m in sub]
        ws = torch.empty(ops.gemm_multi_workspace_bytes([m[1] for m in sub], C, M) + 256, dtype=torch.uint8, device=dev)
        ops.gemm_q8k_multi(sub, xqd, M, ys, ws)
        for i, y in zip(order, ys):
            np.testing.assert_array_equal(host(y)[:, :rows[i]], ref[i])
            assert np.all(host(y)[:, rows[i]:] == -7.0)
