"""GPU parity of the fused parse and decode of a bare stream against the CPU
oracle: block sizes at both ends of its range and of every section count,
ragged ones, chunks shorter than a tile and than a block, sparse and
barely compressible streams, a stream length that is only an upper bound, and
damaged streams.  Bar: values bit-identical; damage is reported."""
import sys

import numpy as np
import pytest

import oracle_lib
from golden_inputs import make_input, make_input_f64

pytestmark = pytest.mark.gpu

CASES = [
    # dtype, fastMode, kind, n, B, T, mode, abs_eb, rel
    (0, 1, "waves", (1 << 22) + 5, 128, 16, 1, 0.0, 1e-4),
    (0, 1, "waves", 3000001, 256, 5, 1, 0.0, 1e-4),
    (0, 1, "waves", 1 << 20, 8, 3, 1, 0.0, 1e-5),
    (0, 1, "walk", 400001, 100, 7, 0, 0.01, 0.0),
    (0, 1, "walk", 200000, 9, 40, 0, 0.01, 0.0),
    (0, 1, "uniform", 700000, 64, 3, 0, 1e-7, 0.0),
    (0, 1, "zeroblocks", 800003, 16, 2, 1, 0.0, 1e-3),
    (0, 1, "constant", 6000000, 32, 1, 0, 0.5, 0.0),
    (0, 1, "sparsewide", 900000, 128, 2, 0, 1.0, 0.0),
    (0, 1, "walk", 37, 8, 16, 0, 0.01, 0.0),
    (1, 1, "waves", (1 << 20) + 3, 64, 16, 1, 0.0, 1e-6),
    (1, 1, "walk", 70001, 200, 5, 0, 1e-9, 0.0),
    (0, 2, "waves", (1 << 21) + 129, 128, 16, 1, 0.0, 1e-4),
    (0, 2, "walk", 300001, 20, 7, 0, 0.01, 0.0),
    (0, 2, "constant", 5000000, 256, 2, 0, 0.5, 0.0),
    (1, 2, "waves", 500001, 32, 3, 1, 0.0, 1e-6),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "f%d-m%d-%s-n%d-B%d-T%d" % (
    64 if c[0] else 32, c[1], c[2], c[3], c[4], c[5]))
def test_bare_stream_matches_oracle(case):
    import torch
    import szp_amd as szp
    dt, fast, kind, n, B, T, mode, ab, rel = case
    print("bare stream", case, flush=True)
    sys.stdout.flush()
    x = (make_input_f64 if dt else make_input)(kind, n, 29 + n)
    st = oracle_lib.compress_mode(fast, x, mode, ab, rel, B, T)
    want = oracle_lib.decompress_mode(fast, st, n, B, T, dtype=x.dtype)
    codec = szp.DeviceCodec(block_size=B, threads=T, fast_mode=fast)
    tdt = torch.float64 if dt else torch.float32
    bits = np.uint64 if dt else np.uint32

    def decode(a):
        t = torch.from_numpy(a).cuda()
        return codec.decompress(t, a.size, n, dtype=tdt)

    for tail in (0, 1, 5003):  # bytes of the buffer past the stream
        y = decode(np.concatenate([st, np.full(tail, 0x11, np.uint8)]))
        codec.check()
        bad = np.nonzero(y.cpu().numpy().view(bits) != want.view(bits))[0]
        assert bad.size == 0, (tail, bad[:8])
    if st.size > 100000:  # cut short: reported, and the next call is whole again
        decode(st[:st.size - st.size // 3])
        with pytest.raises(szp.SzpError):
            codec.check()
        y = decode(st)
        codec.check()
        assert np.array_equal(y.cpu().numpy().view(bits), want.view(bits))
