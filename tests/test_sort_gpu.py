"""Radix sort parity on the GPU: rfx_sort_pairs vs the oracle's stable LSD
sort (bit-exact keys and values), plus full-size properties."""
import numpy as np
import pytest

from redfox_amd import datagen

pytestmark = pytest.mark.gpu

DT = {1: np.uint8, 2: np.uint16, 4: np.uint32, 8: np.uint64, 16: np.uint64}


def make(width, n, seed):
    raw = datagen.splitmix64(seed, (n * width + 7) // 8 + 1).view(np.uint8)
    return np.ascontiguousarray(raw[: n * width]).view(DT[width]).copy()


def run_sort(rf, ctx, keys, vals, kb, bits, vb):
    n = keys.nbytes // kb
    kbuf = rf.DeviceBuffer.from_numpy(keys)
    vbuf = rf.DeviceBuffer.from_numpy(vals) if vb else None
    ctx.sort_pairs(kbuf, vbuf, n, kb, bits, vb)
    ctx.synchronize()
    k = kbuf.download(keys.dtype, keys.size)
    v = vbuf.download(vals.dtype, vals.size) if vb else None
    return k, v


WIDTHS = [(kb, vb) for kb in (1, 2, 4, 8, 16) for vb in (0, 1, 2, 4, 8, 16)]


@pytest.mark.parametrize("kb,vb", WIDTHS)
def test_widths_match_oracle(rf, ctx, orc, kb, vb):
    n = 50_003
    keys = make(kb, n, 11 + kb)
    vals = make(vb, n, 97 + vb) if vb else None
    bits = 8 * kb
    gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    ok, ov = orc.sort_pairs(keys, vals, kb, bits, vb)
    assert np.array_equal(gk, ok)
    if vb:
        assert np.array_equal(gv, ov)


# key_bits values the reference dispatches on (b40cSort.cu:85-826) and the
# widths it keeps them in; high bits above key_bits are random and ignored.
@pytest.mark.parametrize("kb,bits", [(1, 2), (1, 3), (1, 5), (2, 14), (4, 18), (4, 23),
                                     (4, 26), (4, 32), (8, 37), (8, 64), (16, 100)])
def test_key_bits_low_bits_only(rf, ctx, orc, kb, bits):
    n = 70_001
    keys = make(kb, n, 5 + bits)
    vals = np.arange(n, dtype=np.uint32)
    gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, 4)
    ok, ov = orc.sort_pairs(keys, vals, kb, bits, 4)
    assert np.array_equal(gk, ok)
    assert np.array_equal(gv, ov)


@pytest.mark.parametrize("n", [0, 1, 2, 3, 63, 64, 65, 4095, 4096, 4097, 8191, 8193,
                               100_003, (1 << 20) + 7])
def test_sizes(rf, ctx, orc, n):
    keys = make(4, n, 1000 + n)
    vals = np.arange(n, dtype=np.uint32)
    gk, gv = run_sort(rf, ctx, keys, vals, 4, 32, 4)
    ok, ov = orc.sort_pairs(keys, vals, 4, 32, 4)
    assert np.array_equal(gk, ok)
    assert np.array_equal(gv, ov)


def test_all_equal_keys_skip_every_pass(rf, ctx, orc):
    n = 30_000
    keys = np.full(n, 0xDEADBEEF, dtype=np.uint32)
    vals = np.arange(n, dtype=np.uint32)[::-1].copy()
    gk, gv = run_sort(rf, ctx, keys, vals, 4, 32, 4)
    assert np.array_equal(gk, keys) and np.array_equal(gv, vals)


def test_odd_number_of_passes_copies_back(rf, ctx, orc):
    # keys < 2^16 in u32 with 24 key bits: pass 2 is an identity and is
    # skipped, leaving an odd number of passes.
    n = 123_457
    keys = (make(4, n, 3) & np.uint32(0xFFFF)).astype(np.uint32)
    vals = np.arange(n, dtype=np.uint32)
    gk, gv = run_sort(rf, ctx, keys, vals, 4, 24, 4)
    ok, ov = orc.sort_pairs(keys, vals, 4, 24, 4)
    assert np.array_equal(gk, ok) and np.array_equal(gv, ov)


def test_zipf_u64_keys(rf, ctx, orc):
    n = 200_000
    ranks = datagen.zipf_ranks(datagen.BASE_SEED + 2, n, 1.1, 1 << 32)
    keys = datagen.mix64(ranks)
    vals = np.arange(n, dtype=np.uint32)
    gk, gv = run_sort(rf, ctx, keys, vals, 8, 64, 4)
    ok, ov = orc.sort_pairs(keys, vals, 8, 64, 4)
    assert np.array_equal(gk, ok) and np.array_equal(gv, ov)


def test_repeat_calls_reuse_workspace(rf, ctx, orc):
    for n in (300_000, 1000, 77_777):
        keys = make(4, n, n)
        vals = np.arange(n, dtype=np.uint32)
        gk, gv = run_sort(rf, ctx, keys, vals, 4, 32, 4)
        ok, ov = orc.sort_pairs(keys, vals, 4, 32, 4)
        assert np.array_equal(gk, ok) and np.array_equal(gv, ov)


def test_full_size_u32_pairs_properties(rf, ctx):
    """2^28 (u32 key, u32 row index) pairs: the result is sorted, stable
    (indices ascend within equal keys) and a permutation of the input
    (each key equals the input key at its index)."""
    n = 1 << 28
    seed = datagen.BASE_SEED + 1
    kbuf = rf.DeviceBuffer(4 * n)
    vbuf = rf.DeviceBuffer(4 * n)
    ctx.gen_u32(kbuf, n, seed)
    ctx.iota_u32(vbuf, n)
    ctx.sort_pairs(kbuf, vbuf, n, 4, 32, 4)
    ctx.synchronize()
    k = kbuf.download(np.uint32, n)
    v = vbuf.download(np.uint32, n)
    kbuf.close()
    vbuf.close()
    assert np.all(k[1:] >= k[:-1])
    same = k[1:] == k[:-1]
    assert np.all(v[1:][same] > v[:-1][same])
    src = datagen.u32(seed, n)
    assert np.array_equal(src[v], k)


def test_full_size_u64_zipf_pairs_properties(rf, ctx):
    """2^27 (u64 Zipf(1.1) key, u32 row index) pairs, the size the sort is
    measured at: sorted, stable and a permutation of the input (the keys
    are generated on the device and copied before the sort)."""
    n = 1 << 27
    seed = datagen.BASE_SEED + 2
    k0 = rf.DeviceBuffer(8 * n)
    kbuf = rf.DeviceBuffer(8 * n)
    vbuf = rf.DeviceBuffer(4 * n)
    ctx.gen_zipf_u64(k0, n, seed, 1.1, 1 << 32)
    ctx.copy(kbuf, k0, 8 * n)
    ctx.iota_u32(vbuf, n)
    ctx.sort_pairs(kbuf, vbuf, n, 8, 64, 4)
    ctx.synchronize()
    src = k0.download(np.uint64, n)
    k = kbuf.download(np.uint64, n)
    v = vbuf.download(np.uint32, n)
    for b in (k0, kbuf, vbuf):
        b.close()
    assert np.all(k[1:] >= k[:-1])
    same = k[1:] == k[:-1]
    assert same.mean() > 0.3  # Zipf(1.1): many rows repeat a key
    assert np.all(v[1:][same] > v[:-1][same])
    assert np.array_equal(src[v], k)
    assert np.array_equal(np.sort(v), np.arange(n, dtype=np.uint32))


@pytest.mark.parametrize("digit", [8, 9, 10])
@pytest.mark.parametrize("ipt", [0, 12])
@pytest.mark.parametrize("kb,vb,bits", [(4, 0, 32), (4, 4, 18), (4, 4, 20), (4, 4, 26),
                                        (4, 8, 31), (8, 4, 64), (8, 0, 37), (8, 8, 45)])
def test_wider_digits_match_oracle(rf, ctx, orc, digit, ipt, kb, vb, bits):
    """sort.digit 8, 9 and 10 forced over the width chosen from the key bits
    (9 for 17-18 bits, 10 for 19-20): digits that straddle the 32-bit halves
    of 64-bit keys, a narrow last digit, a skipped pass, a ragged last tile;
    keys and values bit-exact against the oracle."""
    n = 300_007
    keys = make(kb, n, 700 + bits)
    if bits == 26:
        keys &= DT[kb](0x3FFFC00)  # bits 0-9 zero: the first pass is skipped
    vals = make(vb, n, 800 + vb) if vb else None
    try:
        ctx.tune("sort.digit", digit)
        ctx.tune("sort.ipt", ipt)
        gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    finally:
        ctx.tune("sort.digit", 0)
        ctx.tune("sort.ipt", 0)
    ok, ov = orc.sort_pairs(keys, vals, kb, bits, vb)
    assert np.array_equal(gk, ok)
    if vb:
        assert np.array_equal(gv, ov)


@pytest.mark.parametrize("kb,vb,bits", [(4, 4, 32), (4, 0, 20), (8, 4, 64), (16, 8, 100), (2, 2, 16)])
def test_wide_status_words_match_oracle(rf, ctx, orc, kb, vb, bits):
    """The 64-bit look-back status words that sorts of more than 2^30 - 1
    rows take, forced on a small sort (knob sort.status = 64): keys and
    values bit-exact against the oracle."""
    n = 250_007
    keys = make(kb, n, 900 + bits)
    vals = make(vb, n, 901) if vb else None
    try:
        ctx.tune("sort.status", 64)
        gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    finally:
        ctx.tune("sort.status", 0)
    ok, ov = orc.sort_pairs(keys, vals, kb, bits, vb)
    assert np.array_equal(gk, ok)
    if vb:
        assert np.array_equal(gv, ov)


def test_more_than_2p30_rows_properties(rf, ctx):
    """2^30 + 12,345 (u32 key, u32 row index) pairs, past the 32-bit status
    words' 2^30 - 1 rows: sorted, stable and a permutation of the input."""
    n = (1 << 30) + 12_345
    k0 = rf.DeviceBuffer(4 * n)
    kbuf, vbuf = rf.DeviceBuffer(4 * n), rf.DeviceBuffer(4 * n)
    ctx.gen_u32(k0, n, datagen.BASE_SEED + 77)
    ctx.copy(kbuf, k0, 4 * n)
    ctx.iota_u32(vbuf, n)
    ctx.sort_pairs(kbuf, vbuf, n, 4, 32, 4)
    ctx.synchronize()
    src = k0.download(np.uint32, n)
    k0.close()
    k = kbuf.download(np.uint32, n)
    kbuf.close()
    v = vbuf.download(np.uint32, n)
    vbuf.close()
    assert np.all(k[1:] >= k[:-1])
    same = k[1:] == k[:-1]
    assert np.all(v[1:][same] > v[:-1][same])
    assert np.array_equal(src[v], k)
    seen = np.zeros(n, dtype=bool)
    seen[v] = True
    assert seen.all()


# Past 2 x 256 CUs x 2 blocks of the largest tile, where blocks that stay take
# their tiles from one ticket; the last size of the small tiles and the next; group
# and tile edges of the small tiles; 7 bit digits with a skipped pass, odd
# numbers of 8 bit digits.
@pytest.mark.parametrize("kb,vb,bits,n", [
    (4, 4, 32, 12_582_912 + 12_289), (4, 0, 32, 16_777_216 + 1), (8, 4, 64, 7_340_032 + 77),
    (8, 8, 24, 6_291_456 + 12_287), (4, 8, 20, 7_340_032 + 14_337),
    (4, 4, 32, 2_097_152), (4, 4, 32, 2_097_153), (4, 8, 18, 3_145_729),
    (8, 0, 64, 65_536), (8, 8, 64, 65_537), (4, 4, 23, 4_096 * 15), (4, 4, 21, 4_096 * 32 + 1),
    (4, 4, 27, 5_000_001), (8, 4, 25, 4_097), (4, 4, 28, 2_500_000), (8, 0, 22, 3_000_003)])
def test_tile_queues_and_small_tiles_match_numpy(rf, ctx, kb, vb, bits, n):
    keys = make(kb, n, 1000 + bits) & DT[kb]((1 << bits) - 1 if bits < 64 else -1 % (1 << 64))
    if bits == 27:
        keys &= DT[kb](0x7F03FFF)  # the third 7-bit digit is zero: its pass is skipped
    vals = make(vb, n, 1001) if vb else None
    gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(gk, keys[order])
    if vb:
        assert np.array_equal(gv, vals[order])


# 6 and 7 bit digits, in even and odd numbers, on the small tiles (their group
# edges and the last size) and on the large one.
@pytest.mark.parametrize("digit", [6, 7])
@pytest.mark.parametrize("kb,vb,bits,n", [
    (4, 4, 23, 4_096 * 15), (4, 4, 21, 4_096 * 32 + 1), (8, 0, 22, 3_000_003), (8, 8, 24, 6_291_456 + 12_287),
    (4, 8, 32, 2_097_152), (8, 4, 37, 100_003), (4, 0, 14, 2_097_153)])
def test_narrow_digits_match_numpy(rf, ctx, digit, kb, vb, bits, n):
    keys = make(kb, n, 1600 + bits)
    vals = make(vb, n, 1601) if vb else None
    try:
        ctx.tune("sort.digit", digit)
        gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    finally:
        ctx.tune("sort.digit", 0)
    order = np.argsort(keys & DT[kb]((1 << bits) - 1), kind="stable")
    assert np.array_equal(gk, keys[order])
    if vb:
        assert np.array_equal(gv, vals[order])


# The first sizes past which tiles come from the queues (4, 8, 24 and 64 tiles
# for each block that runs at once), and the last below, where one ticket
# hands them out.
@pytest.mark.parametrize("kb,vb,bits,n", [
    (4, 4, 16, 2048 * 12_288), (4, 4, 16, 2048 * 12_288 + 1), (8, 4, 11, 2048 * 7168 + 5),
    (8, 8, 16, 1024 * 12_288 + 5), (4, 8, 20, 1024 * 14_336 + 5), (8, 1, 16, 4096 * 7168 + 5),
    (16, 0, 12, 4096 * 4096 + 5), (16, 4, 9, 2048 * 4096 + 5), (8, 0, 8, 12_288 * 7168 + 5)])
def test_tile_queues_begin(rf, ctx, kb, vb, bits, n):
    keys = make(kb, n, 1300 + bits)  # bits above key_bits vary and do not count
    vals = make(vb, n, 1301) if vb else None
    gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    low = keys[::2] if kb == 16 else keys  # word 0 is the low one
    low = (low & low.dtype.type((1 << bits) - 1)).astype(np.uint16 if bits <= 16 else np.uint32)
    order = np.argsort(low, kind="stable")
    if kb == 16:
        keys, gk = keys.reshape(-1, 2), gk.reshape(-1, 2)
    assert np.array_equal(gk, keys[order])
    if vb:
        assert np.array_equal(gv, vals[order])


# 4-byte elements beside narrower ones: the last size of the smaller tile, the
# next one, and past the first queue sizes of both tiles.
@pytest.mark.parametrize("kb,vb,bits", [(2, 4, 16), (4, 1, 16), (4, 2, 13)])
@pytest.mark.parametrize("n", [8193, 2_097_152, 2_097_153, 2048 * 12_288 + 12_289, 4096 * 12_288 + 7])
def test_narrow_columns_match_numpy(rf, ctx, kb, vb, bits, n):
    keys = make(kb, n, 1400 + vb)
    vals = make(vb, n, 1401)
    gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    order = np.argsort((keys & DT[kb]((1 << bits) - 1)).astype(np.uint16), kind="stable")
    assert np.array_equal(gk, keys[order])
    assert np.array_equal(gv, vals[order])


# Sorts of one block: steps and waves that are full, one row past, and the
# last size (8192 rows, 4096 of 16-byte elements) with the next one; digits
# that no key varies in, a narrow last digit, few distinct keys.
@pytest.mark.parametrize("n", [2, 63, 65, 1024, 1025, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("kb,vb,bits", [(4, 4, 32), (8, 4, 64), (8, 8, 61), (2, 1, 11), (1, 16, 8),
                                        (16, 0, 128), (16, 16, 67), (4, 0, 5)])
def test_one_block_sorts_match_oracle(rf, ctx, orc, kb, vb, bits, n):
    keys = make(kb, n, 1100 + bits)
    if kb >= 4:
        keys.view(np.uint8)[kb - 2::kb] = 7  # a byte that is the same in every key
    vals = make(vb, n, 1101) if vb else None
    gk, gv = run_sort(rf, ctx, keys, vals, kb, bits, vb)
    ok, ov = orc.sort_pairs(keys, vals, kb, bits, vb)
    assert np.array_equal(gk, ok)
    if vb:
        assert np.array_equal(gv, ov)


@pytest.mark.parametrize("digit,ipt,bits,passes", [
    (0, 0, 26, 4), (0, 8, 22, 3), (0, 12, 27, 4), (0, 16, 24, 3), (8, 0, 22, 3), (6, 0, 32, 6), (7, 0, 32, 5),
    (7, 0, 28, 4), (0, 8, 28, 4), (6, 8, 22, 4), (0, 12, 20, 2)])
def test_sort_knobs_are_honoured(rf, ctx, digit, ipt, bits, passes):
    """6 and 7-bit digits can be asked for (the number of passes tells), and
    every combination of the two knobs sorts."""
    n = 200_003
    keys = make(4, n, 1200 + bits)
    vals = np.arange(n, dtype=np.uint32)
    try:
        ctx.tune("sort.digit", digit)
        ctx.tune("sort.ipt", ipt)
        ctx.profile(True)
        gk, gv = run_sort(rf, ctx, keys, vals, 4, bits, 4)
        launches, _ = ctx.profile_read("sort.onesweep")
    finally:
        ctx.profile(False)
        ctx.tune("sort.digit", 0)
        ctx.tune("sort.ipt", 0)
    order = np.argsort(keys & np.uint32((1 << bits) - 1), kind="stable")
    assert np.array_equal(gk, keys[order]) and np.array_equal(gv, vals[order])
    assert launches == passes


@pytest.mark.parametrize("vb,n,ipt,passes", [
    (4, 1_500_000, 0, 3), (4, 19_999_999, 0, 3), (4, 20_000_000, 0, 4), (4, 20_000_000, 16, 3),
    (0, 20_000_000, 0, 3), (0, 64_000_000, 0, 4)])
def test_six_bit_digits_where_they_pay(rf, ctx, vb, n, ipt, passes):
    """23-bit keys: three passes of 8 bits below the rows where four of 6 bits
    are faster, and with sort.ipt set, which has tiles for 8 bits only."""
    keys = make(4, n, 1500) & np.uint32(0x7F00FF)  # 15 bits vary: a quick check on the host
    vals = np.arange(n, dtype=np.uint32) if vb else None
    try:
        ctx.tune("sort.ipt", ipt)
        ctx.profile(True)
        gk, gv = run_sort(rf, ctx, keys, vals, 4, 23, vb)
        launches, _ = ctx.profile_read("sort.onesweep")
    finally:
        ctx.profile(False)
        ctx.tune("sort.ipt", 0)
    order = np.argsort((keys & 0xFF | keys >> 8).astype(np.uint16), kind="stable")
    assert np.array_equal(gk, keys[order])
    if vb:
        assert np.array_equal(gv, order.astype(np.uint32))
    assert launches == passes
