"""Host emulation of the fused parse and decode's boundaries and walks
(tests/cpu/fused_check.cc) under AddressSanitizer: on oracle streams of every
geometry class it serves, with garbage tails, and on damaged streams, the block
positions equal a serial walk's and a stream is reported exactly when the
serial walk rejects it."""
import os
import subprocess

import numpy as np
import pytest

import test_parse_emulation as parse

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def fused_check(tmp_path_factory):
    d = tmp_path_factory.mktemp("fused")
    exe = str(d / "fused_check")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-Wall", "-fsanitize=address,undefined",
                    "-fno-sanitize-recover=undefined", "-I", os.path.join(ROOT, "szp_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpu", "fused_check.cc"), "-o", exe], check=True)
    return exe, d


# kind, n, B, T, mode, abs_eb, rel: B at both ends of the served range and of
# every section count, ragged B, chunks shorter than a tile and than a block,
# sparse streams, all widths.
CASES = [
    ("waves", 1 << 21, 128, 4, 1, 0.0, 1e-4),
    ("waves", 1 << 20, 32, 3, 1, 0.0, 1e-2),
    ("waves", 1 << 20, 8, 2, 1, 0.0, 1e-5),
    ("walk", 700001, 256, 5, 1, 0.0, 1e-4),
    ("walk", 200000, 9, 5, 0, 0.01, 0.0),
    ("walk", 400001, 100, 7, 0, 0.01, 0.0),
    ("uniform", 400000, 128, 3, 0, 1e-7, 0.0),
    ("zeroblocks", 800003, 128, 3, 1, 0.0, 1e-3),
    ("zeroblocks", 500000, 16, 2, 1, 0.0, 1e-3),
    ("constant", 4000000, 8, 2, 1, 0.0, 1e-3),
    ("constant", 3000000, 64, 1, 0, 0.5, 0.0),
    ("specials", 300000, 32, 4, 0, 0.5, 0.0),
    ("sparsewide", 400000, 64, 2, 0, 1.0, 0.0),
    ("walk", 40, 8, 16, 0, 0.01, 0.0),
    ("walk", 3, 8, 8, 0, 0.01, 0.0),
]


@pytest.mark.parametrize("fast", [1, 2])
def test_fused_boundaries(fused_check, fast):
    rng = np.random.default_rng(40 + fast)
    entries = []
    for k, c in enumerate(CASES):
        n, B, T = c[1:4]
        st = parse._stream(c, 300 + k) if fast == 1 else parse._ra_stream(c, 300 + k)
        widths = (parse._width_positions if fast == 1 else parse._unit_width_positions)(st, n, B, T)
        entries.append((st, n, B, T, fast))
        for tail, hi in ((7, 256), (70000, 256), (3000, 33), (5000, 1)):
            t = rng.integers(0, hi, tail, dtype=np.uint8)
            entries.append((np.concatenate([st, t]), n, B, T, fast))
        entries.append((st[:-1].copy(), n, B, T, fast))
        entries.append((st[:max(4 + 8 * T, st.size * 2 // 3)].copy(), n, B, T, fast))
        for trial in range(6):
            s2 = st.copy()
            if widths:
                p = widths[int(rng.integers(0, len(widths)))]
                s2[p] = (33 + int(rng.integers(0, 223)), int(rng.integers(0, 33)), 0)[trial % 3]
            entries.append((s2, n, B, T, fast))
        if T > 1:
            for d in (1, 1 << 40):
                s3 = st.copy()
                off = int.from_bytes(st[12:20].tobytes(), "little")
                s3[12:20] = np.frombuffer(np.uint64(off + d).tobytes(), np.uint8)
                entries.append((s3, n, B, T, fast))
        s4 = st.copy()
        s4[4 + 8 * T:] = rng.integers(0, 256, s4.size - 4 - 8 * T, dtype=np.uint8)
        entries.append((s4, n, B, T, fast))
    out = parse._run(fused_check, entries)
    assert int(out.split("(")[1].split()[0]) > 40, out  # damaged streams among them


@pytest.mark.parametrize("n,B,stream", [(1 << 20, 128, 1 << 21), (1 << 20, 8, 1 << 21),
                                        (1 << 20, 256, 3 << 20), (100003, 32, 200000)])
def test_short_workspace_is_refused(n, B, stream):
    """A workspace that holds the block positions of the two-kernel path no
    more is refused before any launch, also where the fused words would fit:
    the addresses below are never used.  Those positions alone are 8 bytes a
    block."""
    import torch  # noqa: F401  (its HIP runtime is loaded first)
    import szp_amd as szp
    short = 8 * (n // B) // 256 * 256
    rc = szp.lib.szp_amd_decompress_dev(0x10000, stream, n, B, 4, 0x20000, 0x30000, short, None)
    assert rc == 2  # SZP_AMD_ERR_CAPACITY
    assert szp.lib.szp_amd_decompress_workspace_size(stream, n, B, 4) > short
