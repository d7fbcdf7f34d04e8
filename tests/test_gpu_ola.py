"""Streaming overlap-add filtering against FP64 convolution, and
streaming in several calls equals one call (the tail carries over)."""
import numpy as np
import pytest
from scipy.signal import fftconvolve

from oracle import inputs
from tests.helpers import from_dev, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,ntaps", [(4, 2), (256, 100), (4096, 2048), (65536, 1000)])
def test_ola_matches_direct_convolution(gpu, N, ntaps):
    import torch
    from mufft_amd.api import OverlapAdd
    hop = N // 2
    nblocks = max(3, (1 << 20) // hop) if N < 65536 else 8
    x = inputs.uniform(0x7001 + N, nblocks * hop)
    h = inputs.gaussian(0x7002 + N, ntaps) / np.float32(np.sqrt(ntaps))
    ola = OverlapAdd(N, torch.from_numpy(h).to(gpu))
    dx = to_dev(x, gpu)
    out = torch.zeros(nblocks * hop, dtype=torch.float32, device=gpu)
    ola(out, dx, nblocks)
    torch.cuda.synchronize()
    ref = fftconvolve(x.astype(np.float64), h.astype(np.float64))[: nblocks * hop]
    y = from_dev(out)
    rel = np.sqrt(np.mean((y - ref) ** 2) / np.mean(ref ** 2))
    assert rel < 2e-6, rel
    # streaming: the same signal in three calls (tail carried) gives the same samples
    ola.reset()
    parts = [1, nblocks - 2, 1]
    outs, off = [], 0
    for nb in parts:
        o = torch.zeros(nb * hop, dtype=torch.float32, device=gpu)
        ola(o, dx[off * hop:(off + nb) * hop], nb)
        outs.append(o)
        off += nb
    torch.cuda.synchronize()
    y2 = np.concatenate([from_dev(o) for o in outs])
    np.testing.assert_array_equal(y2.view(np.uint32), y.view(np.uint32))


def test_ola_rejects_bad_arguments(gpu):
    import mufft_amd as M
    from mufft_amd.api import OverlapAdd
    h = np.ones(10, np.float32)
    for N, taps in ((6, h), (8, h)):  # non power of two; more taps than N/2
        with pytest.raises(M.MufftError):
            OverlapAdd(N, taps)


# Block sizes of the one-launch kernel: one point per slot up to its largest,
# one and several rounds of blocks per workgroup (N = 4096 beyond 1024 blocks),
# partial workgroups, and the first size of the three-launch path.
@pytest.mark.parametrize("N,nblocks", [(4, 1), (8, 511), (16, 600), (32, 37), (64, 129), (128, 1), (512, 33), (1024, 9),
                                       (2048, 3), (4096, 2), (4096, 1024), (4096, 1027), (4096, 5003), (8192, 7), (16384, 3)])
def test_ola_block_counts(gpu, N, nblocks):
    import torch
    from mufft_amd.api import OverlapAdd
    print(f"overlap-add N={N} x {nblocks}", flush=True)
    hop = N // 2
    x = inputs.uniform(0x7100 + N, nblocks * hop)
    h = inputs.gaussian(0x7101 + N, hop) / np.float32(np.sqrt(hop))
    ola = OverlapAdd(N, h)
    out = torch.full((nblocks * hop + 8,), 3.0, dtype=torch.float32, device=gpu)
    ola(out, to_dev(x, gpu), nblocks)
    ola(out[nblocks * hop:], torch.zeros(8, dtype=torch.float32, device=gpu), 0)   # nothing to do
    tail = torch.full((hop,), 3.0, dtype=torch.float32, device=gpu)
    ola(tail, torch.zeros(hop, dtype=torch.float32, device=gpu), 1)   # the carried tail alone
    torch.cuda.synchronize()
    ref = fftconvolve(np.concatenate([x, np.zeros(hop)]).astype(np.float64), h.astype(np.float64))[: (nblocks + 1) * hop]
    y = np.concatenate([from_dev(out)[: nblocks * hop], from_dev(tail)])
    assert np.sqrt(np.mean((y - ref) ** 2) / np.mean(ref ** 2)) < 2e-6
    assert np.all(from_dev(out)[nblocks * hop:] == 3.0)


def test_ola_in_place(gpu):
    """Output over the input: the three-launch path, same samples to rounding."""
    import torch
    from mufft_amd.api import OverlapAdd
    N, nblocks = 1024, 50
    x = to_dev(inputs.uniform(0x7200, nblocks * N // 2), gpu)
    h = inputs.gaussian(0x7201, N // 2)
    a, b = OverlapAdd(N, h), OverlapAdd(N, h)
    y = torch.empty_like(x)
    a(y, x, nblocks)
    b(x, x, nblocks)
    torch.cuda.synchronize()
    p, q = from_dev(y).astype(np.float64), from_dev(x).astype(np.float64)
    assert np.sqrt(np.mean((p - q) ** 2) / np.mean(p ** 2)) < 2e-6
