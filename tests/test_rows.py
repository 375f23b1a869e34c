"""kq_gemv_rows: several rows of fp32 activations in one launch, each output row with the bits of
kq_gemv_multi on that row, so the tolerance is equality."""
import ctypes

import pytest
import torch

from kq import _lib, ops
from kq import quantize as kqq


# rows either side of a unit (4 rows), a workgroup (8 waves) and the GPU; one to 15 column passes, whole
# and partial; token groups of one size and of two (N just past 4, 8 and 16), both kernels (N <= 4, N > 4)
@pytest.mark.gpu
@pytest.mark.parametrize("Rs,C,types,N", [
    ((8,), 256, (12,), 2), ((8,), 256, (14,), 5),
    ((136, 24), 4096, (12, 12), 4), ((264, 40, 8), 4096, (12, 14, 12), 9), ((2056, 512, 512), 4096, (12, 12, 14), 24),
    ((40,), 4352, (14,), 3), ((72,), 12288, (12,), 8), ((264,), 12288, (14,), 17), ((24,), 17408, (12,), 6),
    ((16,), 61440, (14,), 11), ((16,), 61440, (12,), 4),
    # two and three rows against short, wide Q6_K matrices: either side of the lines where they go row by row
    ((512, 512), 16640, (14, 14), 2), ((1032,), 16640, (14,), 2), ((1024,), 16384, (14,), 2),
    ((64, 8), 33024, (14, 12), 3), ((72,), 33024, (14,), 3), ((64,), 32768, (14,), 3), ((8,), 61440, (14,), 3),
    ((16,), 61440, (14,), 3), ((8,), 61440, (14,), 2),
])
def test_rows_equal_one_row_calls(dev, Rs, C, types, N):
    mats = [(torch.from_numpy(kqq.synthetic_matrix(R, C, t, seed=R + i)).to(dev), R, C, t)
            for i, (R, t) in enumerate(zip(Rs, types))]
    X = torch.from_numpy(kqq.synthetic_activations(N, C + 4, seed=C + N)).to(dev)[:, :C]   # ldx = C + 4
    ys = [torch.full((N, R), -1.0, device=dev) for R in Rs]
    ops.gemv_rows(mats, X, ys)
    for n in range(N):
        want = [torch.empty(R, device=dev) for R in Rs]
        ops.gemv_multi(mats, X[n], want)
        for y, z in zip(ys, want):
            assert torch.equal(y[n], z), (n, z.numel())


@pytest.mark.gpu
@pytest.mark.parametrize("ty", [12, 14])
def test_rows_special_activations(dev, ty):
    """Infinities, NaN, zeros of both signs and values near the fp32 limits, bit for bit."""
    R, C, N = 24, 4352, 6
    X = torch.from_numpy(kqq.synthetic_activations(N, C, seed=3)).to(dev)
    X[0, 17], X[1, 300], X[2, 4351] = float("inf"), float("nan"), float("-inf")
    X[3] *= 1e36
    X[4] = -0.0
    X[5] *= 1e-38
    mats = [(torch.from_numpy(kqq.synthetic_matrix(R, C, ty, seed=5)).to(dev), R, C, ty)]
    y = torch.empty((N, R), device=dev)
    ops.gemv_rows(mats, X, [y])
    for n in range(N):
        z = torch.empty(R, device=dev)
        ops.gemv_multi(mats, X[n], [z])
        # NaN payloads aside, the same bits (the sign of zero included)
        same = (y[n].view(torch.int32) == z.view(torch.int32)) | (y[n].isnan() & z.isnan())
        assert same.all(), n


@pytest.mark.parametrize("N,ldx,ldy,msg", [(0, 256, 64, "N=0 must be positive"), (4, -256, 64, "ldx=-256 is negative"),
                                           (4, 256, 63, "ldy[0] is smaller than R")])
def test_rows_argument_errors(N, ldx, ldy, msg):
    lib = _lib.kq()
    P, I, L = ctypes.c_void_p * 1, ctypes.c_int * 1, ctypes.c_int64 * 1
    rc = lib.kq_gemv_rows(1, P(4096), I(64), 256, I(12), ctypes.c_void_p(4096), ldx, N, P(8192), L(ldy), None)
    assert rc == _lib.KQ_ERR_ARG and msg in lib.kq_last_error().decode()


@pytest.mark.gpu
def test_rows_refuse_views_narrower_than_the_matrix(dev):
    """A column view of fewer than R values a row holds enough elements once it has rows to spare, and its stride is
    wide enough: the call is refused, as one row at a time is, and the columns beside the view stay as they were."""
    from kq.gpu4 import Engine, Weights
    R, C, N = 200, 256, 3
    w = Weights(dev)
    w.add("m", kqq.synthetic_matrix(R, C, 12, seed=1), R, C, 12)
    eng = Engine(w, mode="f32", chunk=0)
    X = torch.from_numpy(kqq.synthetic_activations(N, C, seed=2)).to(dev)
    base = torch.full((10, 300), -5.0, device=dev)
    for y, err in ((base[:, :100], ValueError), (base.clone().as_strided((2, 300), (200, 1)), IndexError)):
        with pytest.raises(ValueError):                  # (the second: elements for three rows, but two of them)
            ops.gemv_rows([w["m"]], X, [y])
        with pytest.raises(err):
            eng.gemv_batch(["m"], X, [y])
    assert (base == -5.0).all()
    ref, got = torch.empty((N, R), device=dev), torch.full((N, 300), -5.0, device=dev)
    eng.gemv_batch(["m"], X, [ref])
    eng.gemv_batch(["m"], X, [got])                      # rows wider than R
    assert torch.equal(got[:, :R], ref) and (got[:, R:] == -5.0).all()
    cube = torch.empty((1, 1, R), device=dev)
    eng.gemv_batch(["m"], X[:1], [cube])                 # any shape that holds one row
    assert torch.equal(cube.view(R), ref[0])


@pytest.mark.gpu
def test_rows_beyond_one_launch(dev):
    """More rows of x than one launch has threads for (2^32 at 8 rows a workgroup of 512): every row is written, and
    those around the parts' edges have the one-row call's bits.  The rows of x overlap, each one float further on."""
    R, C, N = 8, 256, (1 << 23) + 5
    mat = (torch.from_numpy(kqq.synthetic_matrix(R, C, 12, seed=4)).to(dev), R, C, 12)
    base = torch.randn(N + C, generator=torch.Generator(device=dev).manual_seed(1), device=dev)
    X = base.as_strided((N, C), (1, 1))
    y = torch.full((N, R), float("nan"), device=dev)
    ops.gemv_rows([mat], X, [y])
    assert not y.isnan().any()
    for n in (0, 1, N // 4, N // 2 - 1, N // 2, N // 2 + 1, N - 9, N - 1):
        want = torch.empty(R, device=dev)
        ops.gemv_multi([mat], X[n], [want])
        assert torch.equal(y[n], want), n
