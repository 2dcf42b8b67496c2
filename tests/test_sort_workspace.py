"""rfx_sort_workspace on the host (no device call): never smaller for more
rows, so a context reserved for its largest sort holds every smaller one."""
import ctypes

import pytest


@pytest.fixture(scope="module")
def need():
    import redfox_amd

    f = ctypes.CDLL(redfox_amd.LIB_PATH).rfx_sort_workspace
    f.restype = ctypes.c_uint64
    f.argtypes = [ctypes.c_uint64, ctypes.c_int, ctypes.c_int, ctypes.c_int]
    return f


@pytest.mark.parametrize("kb", [1, 2, 4, 8, 16])
@pytest.mark.parametrize("vb", [0, 1, 2, 4, 8, 16])
def test_never_decreases(need, kb, vb):
    top = (1 << 31) - 1
    sizes = {1, 2, 8191, 8192, 8193, (1 << 30) - 2, (1 << 30) - 1, 1 << 30, (1 << 30) + 1, top}
    for unit in (1000, 1024):  # every power of two in rows, and 1.5 % steps
        n = unit
        while n < top:
            sizes.update((n - 1, n, n + 1))
            n = n + max(1, n // 64) if unit == 1000 else 2 * n
    for ipt in (4, 8, 12, 14, 16, 20, 24, 32):  # counts of tiles about the grouped look-back's limit
        for nt in (512, 1024):
            for tiles in (511, 512, 2047, 2048, 2049, 2050, 2063, 2064, 4096):
                sizes.update(min(top, nt * ipt * tiles + d) for d in (-1, 0, 1, 30_000))
    for bits in {1, 8, 17, 20, 22, 27, 32, 61, 64, 128, 8 * kb}:
        if bits > 8 * kb:
            continue
        last = 0
        for n in sorted(sizes):
            w = need(n, kb, bits, vb)
            assert w >= last, (bits, n, w, last)
            assert w >= n * (kb + vb)  # the second buffers alone
            last = w
