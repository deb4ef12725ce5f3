"""The relative bound of small fields (min and max found by one workgroup):
streams byte-identical to the CPU oracle's at the sizes around its vectors,
its strides and its limit of 256 KiB, with the field on and off a 16-byte
boundary, and with NaN and signed zeros."""
import numpy as np
import pytest

import oracle_lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("dt,n", [(0, n) for n in (1, 3, 4, 5, 4095, 4096, 16385, 65535, 65536, 65537)] +
                         [(1, n) for n in (1, 2, 3, 2049, 32767, 32768, 32769)])
def test_small_relative_bound(dt, n, shift):
    import torch
    import szp_amd as szp
    print("small range", dt, n, shift, flush=True)
    rng = np.random.default_rng(n)
    base = rng.standard_normal(n).astype(np.float64 if dt else np.float32)
    lo, hi = base.copy(), base.copy()
    lo[n - 1], lo[n // 2] = -9.0, np.nan     # extreme last; a NaN that is skipped
    hi[0], hi[n // 3] = 9.0, -0.0
    nan = base.copy()
    nan[0] = np.nan                          # leading NaN: the bound is NaN
    for x in (base, lo, hi, nan, np.full_like(base, -0.0)):
        want = oracle_lib.compress_mode(1, x, 1, 0.0, 1e-3, 32, 2)
        room = torch.empty(n + 4, dtype=torch.float64 if dt else torch.float32, device="cuda")
        room.fill_(1e30)                     # past the field: no part of its range
        y = room[shift:shift + n]
        y.copy_(torch.from_numpy(x))
        codec = szp.DeviceCodec(block_size=32, threads=2)
        got, size = codec.compress(y, rel=1e-3)[:2]
        codec.check()
        size = int(size)
        assert size == want.size
        assert np.array_equal(got[:size].cpu().numpy(), want)
