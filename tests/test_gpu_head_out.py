"""Half outputs and the batch reduction of the gradients: the multiply entry
point that writes only the first half of each output against the one that
writes all of it (same bits), and the reduction's splits against FP64."""
import ctypes

import numpy as np
import pytest

from tests.helpers import cplx, from_dev, rel_rms, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,N", [("c2c", 4), ("c2c", 64), ("c2c", 1024), ("c2c", 8192), ("c2c", 16384), ("c2c", 32768),
                                    ("c2c", 65536), ("r2c", 8), ("r2c", 512), ("r2c", 4096), ("r2c", 32768), ("r2c", 65536)])
@pytest.mark.parametrize("conj", [False, True])
def test_first_half_of_the_adjoint(gpu, kind, N, conj):
    import mufft_amd as M
    import torch
    B = 3
    nb = N if kind == "c2c" else N // 2 + 1
    dt = torch.complex64 if kind == "c2c" else torch.float32
    p = M.Plan1D(kind, N, M.FORWARD, M.FLAG_ZERO_PAD_UPPER_HALF)
    g = to_dev(cplx(0xB000 + N, B * nb, 0.5).reshape(B, nb), gpu)
    h = to_dev(cplx(0xB001 + N, nb, 0.5), gpu)
    full = torch.empty((B, N), dtype=dt, device=gpu)
    half = torch.full((B, N // 2), 3.0, dtype=dt, device=gpu)
    apart = torch.full((B, N // 2 + 6), 3.0, dtype=dt, device=gpu)
    kw = dict(norm=1.0 / N, conj2=conj, adjoint=True)
    p.execute_mul_batched(full, g, h, B, **kw)
    p.execute_mul_batched(half, g, h, B, head=True, **kw)
    p.execute_mul_batched(apart, g, h, B, odist=N // 2 + 6, head=True, **kw)
    torch.cuda.synchronize()
    ref = from_dev(full)[:, : N // 2]
    # the fixed-flag kernel may contract differently: same values to rounding
    assert rel_rms(from_dev(half), ref) < 5e-7
    assert rel_rms(from_dev(apart)[:, : N // 2], ref) < 5e-7
    assert np.all(from_dev(apart)[:, N // 2:] == 3.0)


def test_first_half_refused_beyond_the_fused_sizes(gpu):
    import mufft_amd as M
    import torch
    from mufft_amd import _lib
    N = 1 << 17
    p = M.Plan1D("c2c", N, M.FORWARD)
    x = torch.zeros(N, dtype=torch.complex64, device=gpu)
    y = torch.zeros(N, dtype=torch.complex64, device=gpu)
    a = [ctypes.c_void_p(t.data_ptr()) for t in (y, x, x)]
    assert _lib.load().mufft_hip_execute_plan_1d_mul_head_batched(p.handle, *a, 1, 0, 0, 0, ctypes.c_float(1.0), 0, 0, None) != 0


# Every split of the batch over a workgroup (4 to 256 bins, and one group), with
# batches that do not fill the groups.
@pytest.mark.parametrize("n,B", [(1, 1), (3, 2000), (129, 32), (2049, 257), (5000, 70), (9000, 33), (17000, 17), (33000, 9),
                                 (70000, 5), (140000, 3)])
def test_mul_reduce_splits(gpu, n, B):
    import torch
    from mufft_amd import api as A
    a = cplx(0xB100 + n, B * n).reshape(B, n)
    b = cplx(0xB101 + n, B * n).reshape(B, n)
    out = torch.empty(n, dtype=torch.complex64, device=gpu)
    A.mul_reduce(out, to_dev(a, gpu), to_dev(b, gpu), n, B, norm=0.25, conj_b=True)
    torch.cuda.synchronize()
    ref = 0.25 * np.sum(a.astype(np.complex128) * np.conj(b.astype(np.complex128)), axis=0)
    assert rel_rms(from_dev(out), ref) < 1e-6
