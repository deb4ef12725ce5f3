"""Host arrays through the pinned staging buffers (8 MiB and more per copy, in
chunks of 2 MiB): sizes at the edges of both, against the CPU oracle, with two
threads calling at once."""
import threading

import numpy as np
import pytest

import oracle_lib
from golden_inputs import make_input, make_input_f64

pytestmark = pytest.mark.gpu

MIB = 1 << 20


@pytest.mark.parametrize("dt,nbytes", [(0, 8 * MIB - 4), (0, 8 * MIB), (0, 8 * MIB + 4),
                                       (0, 22 * MIB + 12), (1, 10 * MIB + 8)])
def test_staged_copies(dt, nbytes):
    import torch
    assert torch.cuda.is_available(), "no HIP device visible"
    import szp_amd as szp
    print("staged copies", dt, nbytes, flush=True)
    n = nbytes // (8 if dt else 4)
    x = (make_input_f64 if dt else make_input)("uniform", n, n)  # a stream of several chunks
    T, eb = 16, 1e-7
    want = oracle_lib.compress_mode(1, x, 0, eb, 0.0, 128, T)
    dec = oracle_lib.decompress_mode(1, want, n, 128, T, dtype=x.dtype)
    if nbytes > 16 * MIB:
        assert want.size > 8 * MIB  # the stream is staged too
    res = [None, None]

    def call(k):
        st, size = szp.szp_compress(1, dt, x, 0, eb, 0.0, n, 128)
        res[k] = (st, szp.szp_decompress(1, dt, st, size, n, 128))

    szp.set_threads(T)
    try:
        th = [threading.Thread(target=call, args=(k,)) for k in range(2)]
        for t in th:
            t.start()
        for t in th:
            t.join()
    finally:
        szp.set_threads(0)
    for st, y in res:
        assert np.array_equal(st, want)
        assert np.array_equal(y.view(np.uint8), dec.view(np.uint8))
