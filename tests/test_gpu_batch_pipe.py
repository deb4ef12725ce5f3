"""The batched decode's pipeline at the edges of its queue: fewer entries than
workgroups, one workgroup, tickets longer than a class's entries, fields of
one value, of chunks shorter than a tile, and barely compressible ones, against
the CPU oracle (bit-identical)."""
import numpy as np
import pytest

import oracle_lib
from golden_inputs import make_input

pytestmark = pytest.mark.gpu

SIZES = (1, 7, 129, 4097, 70001, 300000)


@pytest.mark.parametrize("B,T", [(128, 16), (8, 3), (256, 1)])
@pytest.mark.parametrize("ticket,grid", [(1, 1), (1, 0), (3, 5), (2, 9), (1 << 30, 40), (7, 4096)])
def test_batch_decode_queue_edges(B, T, ticket, grid):
    import torch
    from szp_amd import ABS
    from szp_amd.batch import CompressBatch, DecompressBatch
    print("batch decode", B, T, ticket, grid, flush=True)
    kinds = ("waves", "uniform", "zeroblocks")
    xs = [make_input(kinds[k % 3], n, 5 + k) for k, n in enumerate(SIZES * 2)]
    modes = [(ABS, 1e-7 if k % 3 == 1 else 1e-3, 0.0) for k in range(len(xs))]
    cb = CompressBatch([torch.from_numpy(x).cuda() for x in xs], modes, block_size=B, threads=T)
    cb.launch()
    cb.check()
    sizes = cb.byte_sizes()
    db = DecompressBatch([cb.stream(k, s) for k, s in enumerate(sizes)], sizes, [x.size for x in xs],
                         [cb.index_of(k) for k in range(len(xs))], block_size=B, threads=T)
    for _ in range(2):
        for o in db.outs:
            o.fill_(-1.0)
        db.launch(ticket=ticket, grid=grid)
        db.check()
        for k, x in enumerate(xs):
            st = oracle_lib.compress(x, modes[k][0], modes[k][1], 0.0, B, T)
            want = oracle_lib.decompress(st, x.size, B, T)
            assert np.array_equal(db.outs[k].cpu().numpy().view(np.uint32), want.view(np.uint32)), k
