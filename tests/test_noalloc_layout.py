"""Host side of the allocation-free E_RPA from stored Pi(u): the buffers of every chunk,
laid out here as the call lays them out, end inside the 256 MiB scratch array, and a
chunk of one more frequency would not.  No GPU is used."""
import ctypes as C
import re
from pathlib import Path

import pytest

from brpa import _lib

ARRAY = 256 << 20
INT = Path(__file__).resolve().parent.parent / "beyond-rpa_amd" / "csrc" / "internal.h"


def _lists():
    """Number of work lists of the Cholesky."""
    m = re.search(r"enum \{ ([^}]*), CHOL_NLISTS \};", INT.read_text())
    return len(m.group(1).split(","))


def _laid_out(n, nf, packed, frag):
    """Bytes of StoredBufs for nf matrices of order n: every array on 256 bytes."""
    steps = -(-n // 64)
    sizes = [frag, 8 * (2 + 2 * _lists() * steps)]
    if packed:
        sizes.append(8 * nf * (n * (n + 1) // 2))
    sizes += [8 * nf * n * n, 8 * nf * n, 16 * nf * steps, 8 * nf, 8 * nf, 8, 4 * nf,
              8 * nf * 64 * 64]
    return sum(-(-s // 256) * 256 for s in sizes)


@pytest.fixture(scope="module")
def fns():
    lib = _lib.load()
    size, chunk = getattr(lib, "_Z13noalloc_bytesllb"), getattr(lib, "_Z13noalloc_chunkllb")
    size.restype, size.argtypes = C.c_size_t, [C.c_int64, C.c_int64, C.c_bool]
    chunk.restype, chunk.argtypes = C.c_int64, [C.c_int64, C.c_int64, C.c_bool]
    return size, chunk


@pytest.mark.parametrize("packed", [False, True])
def test_chunks_fit(fns, packed):
    size, chunk = fns
    # one descriptor, from an order whose other arrays are known
    frag = size(1, 1, packed) - (_laid_out(1, 1, packed, 0))
    assert frag in (256, 512)
    orders = [1, 2, 63, 64, 65, 100, 128, 129, 255, 256, 257, 295, 320, 367, 400, 512, 777, 1024,
              1500, 2048, 2500, 3000, 3543, 4000, 4032, 5000, 5700, 5760, 5790, 5793, 5800, 8000]
    orders += list(range(280, 310)) + list(range(3500, 3600, 7))
    for n in orders:
        for nf in (1, 2, 3, 5, 12, 16, 24, 100, 367, 368, 400, 1000, 4096):
            fc = chunk(n, nf, packed)
            assert 0 <= fc <= nf
            if fc == 0:
                assert _laid_out(n, 1, packed, frag) > ARRAY, n
                continue
            assert _laid_out(n, fc, packed, frag) <= ARRAY, (n, nf, fc)
            if fc < nf:
                assert _laid_out(n, fc + 1, packed, frag) > ARRAY, (n, nf, fc)
