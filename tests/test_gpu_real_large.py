"""Real transforms beyond the fused sizes, whose resolve runs inside a column
launch: every length of that launch, in full tiles and in the narrow ones a
small batch takes, at odd distances, against FP64."""
import numpy as np
import pytest

from tests.helpers import empty_dev, from_dev, real, rel_rms, to_dev

pytestmark = pytest.mark.gpu

# (log2 of the complex length, split code log2 N1 << 8 | log2 A << 4 | log2 B, batches).
# r2c resolves in the last launch (N2 = N / N1 or B rows), c2r in the first (N1
# rows, 256 to 1024 of them).  The larger batch gives each more than 128 tiles.
CASES = [
    (17, 9 << 8, (1, 9)),                 # r2c 256 rows, c2r 512
    (17, 8 << 8, (1, 17)),                # r2c 512, c2r 256
    (17, 7 << 8, (1, 33)),                # r2c 1024, c2r unfused
    (17, 10 << 8, (1, 33)),               # r2c 128, c2r 1024
    (17, 11 << 8, (2,)),                  # r2c 64, c2r unfused
    (20, 8 << 8 | 6 << 4 | 6, (2,)),      # three launches, r2c 64 rows
    (22, 7 << 8 | 6 << 4 | 9, (1,)),      # three launches, r2c 512 rows
]


@pytest.mark.parametrize("logn,code,batches", CASES)
def test_real_resolve_in_column_launch(gpu, logn, code, batches):
    import torch
    import mufft_amd as M
    from mufft_amd import api
    n = 1 << logn
    N = 2 * n
    try:
        api.set_large_split(n, "c2c_forward", code)
        p, q = M.Plan1D("r2c", N), M.Plan1D("c2r", N)
        for b in batches:
            print(f"real {N} split {code:#x} batch {b}", flush=True)
            sd, xd = n + 1 + 2, N + 6   # odd distance of the spectra
            x = real(0xA000 + logn + b, b * xd, 0.5).reshape(b, xd)
            dX = torch.full((b, sd), 3.0 + 0j, dtype=torch.complex64, device=gpu)
            p.execute_batched(dX, to_dev(x, gpu), b, xd, sd)
            dy = torch.full((b, xd), 3.0, dtype=torch.float32, device=gpu)
            q.execute_batched(dy, dX, b, sd, xd)
            torch.cuda.synchronize()
            X, y = from_dev(dX), from_dev(dy)
            assert np.all(X[:, n + 1:] == 3.0) and np.all(y[:, N:] == 3.0)   # nothing past a transform
            for g in sorted({0, b // 2, b - 1}):
                ref = np.fft.rfft(x[g, :N].astype(np.float64))
                assert rel_rms(X[g, : n + 1], ref) < 2e-6, (b, g)
                # bins 0, n/2 and n and their neighbours, per element
                edge = [0, 1, 2, n // 2 - 1, n // 2, n // 2 + 1, n - 2, n - 1, n]
                assert np.max(np.abs(X[g][edge] - ref[edge])) < 2e-6 * np.sqrt(N), (b, g)
                assert rel_rms(y[g, :N] / N, x[g, :N]) < 2e-6, (b, g)
    finally:
        api.set_large_split(n, "c2c_forward", 0)


def test_c2r_reads_imaginary_parts_of_bins_0_and_n(gpu):
    """The imaginary parts of the first and last bin reach the output of the
    fused first launch as they do in the smaller kernels (kernel.c:36-45):
    c2r(i e_0) = -(-1)^m, c2r(i e_n) = -1."""
    import torch
    import mufft_amd as M
    N = 1 << 18
    q = M.Plan1D("c2r", N)
    dX = torch.zeros((2, N // 2 + 1), dtype=torch.complex64, device=gpu)
    dX[0, 0] = 1j
    dX[1, N // 2] = 1j
    dy = empty_dev((2, N), np.float32, gpu)
    q.execute_batched(dy, dX, 2)
    torch.cuda.synchronize()
    y = from_dev(dy)
    sign = np.where(np.arange(N) % 2 == 0, -1.0, 1.0)
    assert np.max(np.abs(y[0] - sign)) < 2e-6 and np.max(np.abs(y[1] + 1.0)) < 2e-6
