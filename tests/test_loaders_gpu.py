"""Text loading on the GPU (rfx_tbl_parse) against the oracle's parser on
the same bytes: the reference's TC.tbl fixture, edge rows (no final
newline, CRLF, short and empty rows, signs and spaces), texts across the
64 KB tile edges and at every alignment, the capacity limit, and the Q1 plan
run from lineitem.tbl text; device memory as the loader uses it: large
copies, kept blocks, refused frees."""
import ctypes
import os

import numpy as np
import pytest

import oracle
from redfox_amd import datagen, loaders, raplan

pytestmark = pytest.mark.gpu
GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


def check(rf, ctx, text, spec, delim="|"):
    cols, n, short = loaders.parse_tbl(ctx, text, spec, delim)
    want, wshort = oracle.parse_tbl(text, spec, delim.encode())
    assert short == wshort
    got = [c.download(loaders.NUMPY[s], n) for c, s in zip(cols, spec) if s != "skip"]
    for g, w, s in zip(got, want, [s for s in spec if s != "skip"]):
        assert len(g) == len(w) == n
        if s == "f64":
            assert np.array_equal(g.view(np.uint64), w.view(np.uint64)), s
        else:
            assert np.array_equal(g, w), s
    return got, n


def test_reference_tc_fixture(rf, ctx):
    text = open(os.path.join(GOLDEN, "TC.tbl"), "rb").read()
    (a, b), n = check(rf, ctx, text, ["i32", "i32"], "\t")
    assert n == 5 and a.tolist() == [1, 2, 3, 4, 5] and b.tolist() == [6, 7, 8, 9, 10]


@pytest.mark.parametrize("text", [
    b"", b"\n", b"42", b"1|a|2.5|\r\n-3|b\n\n7|c|0.125|extra|\n8",
    b"  -12|  +7|-0.50|1996-02-29|R|\n|||||\n9999999999|1|123456789.123|1998-12-31|N|",
    b"1|2|3.5|19a96-0 2-+3x|Z\n1|2|3.5| 1996- 02-29|Z\n",
])
def test_edge_rows(rf, ctx, text):
    check(rf, ctx, text, ["i64", "i32", "f64", "date", "char"])


@pytest.mark.parametrize("n_orders", [1, 60, 61, 62, 200, 4000, 60_000])
def test_lineitem_text_sizes(rf, ctx, n_orders):
    text = datagen.lineitem_tbl(n_orders, n_orders)[0]
    check(rf, ctx, text, loaders.LINEITEM_SPEC + ["skip", "skip", "skip", "char"])


def test_tile_edge_newlines(rf, ctx):
    # Newlines at 8191/8192/8193, at the ends of 16-byte words, and a block
    # whose rows span more text than the field pass stages in LDS.
    rows = []
    for L in (8190, 1, 14, 15, 16, 17, 8191, 31, 50_000, 3):  # 50000: past the LDS stage
        rows.append(b"7" * L)
    text = b"\n".join(rows) + b"\n"
    check(rf, ctx, text, ["u32"])


@pytest.mark.parametrize("first", [65_533, 65_534, 65_535, 65_536, 131_071])
def test_newlines_about_tile_ends(rf, ctx, first):
    """Empty and short rows across the end of a 64 KB tile of the row-ends pass."""
    text = b"8" * first + b"\n\n\n12\n\n" + b"3|4\n" * 20_000
    check(rf, ctx, text, ["u32"])


@pytest.mark.parametrize("delim,text", [
    # Empty fields between spaces: a field is its own bytes only, never the
    # next field's digits after the delimiter.
    (" ", b"12 34 5.5 1996-01-02 x\n 7  8\n-1 +2 .25 1998-12-31\n  \n"),
    (".", b"1.2.3.1996-01-02.x\n7..8\n"),
    ("+", b"1+-2+3.5+1992-01-01+y\n+5\n"),
    ("5", b"1525352.51996-01-025x\n555\n"),
])
def test_delimiters_that_numbers_use(rf, ctx, delim, text):
    check(rf, ctx, text, ["i32", "i32", "f64", "date", "char"], delim)


def test_unaligned_text_and_capacity(rf, ctx):
    text = datagen.lineitem_tbl(3000, 5)[0]
    buf = rf.DeviceBuffer(len(text) + 16)
    buf.upload(np.frombuffer(text, dtype=np.uint8), offset=3)

    class At:
        ptr = buf.ptr + 3
    cols, n, short = loaders.parse_tbl(ctx, At(), ["u32", "skip", "skip", "u8"], "|", len(text))
    want, _ = oracle.parse_tbl(text, ["u32", "skip", "skip", "u8"])
    assert n == len(want[0]) and short == 0
    assert np.array_equal(cols[0].download(np.uint32, n), want[0])
    assert np.array_equal(cols[3].download(np.uint8, n), want[1])
    # Capacity below the row count: every row counted, the first `cap` stored.
    cap = 1000
    out = rf.DeviceBuffer(4 * cap)
    types = (ctypes.c_int * 1)(loaders.TBL["u32"])
    ptrs = (ctypes.c_void_p * 1)(out.ptr)
    rows, sh = rf.u64_cell(), rf.u64_cell()
    assert rf.lib().rfx_tbl_parse(ctx.handle, At.ptr, len(text), b"|", types, 1, ptrs, cap,
                                  rows.ptr, sh.ptr) == 0
    assert rf.read_u64(rows) == n
    assert np.array_equal(out.download(np.uint32, cap), want[0][:cap])


def test_bad_arguments_are_refused(rf, ctx):
    types = (ctypes.c_int * 1)(42)
    ptrs = (ctypes.c_void_p * 1)(None)
    cell = rf.u64_cell()
    buf = rf.DeviceBuffer(16)
    assert rf.lib().rfx_tbl_parse(ctx.handle, buf.ptr, 4, b"|", types, 1, ptrs, 0, cell.ptr,
                                  cell.ptr) == -1
    types[0] = loaders.TBL["u32"]
    assert rf.lib().rfx_tbl_parse(ctx.handle, buf.ptr, 4, b"\n", types, 1, ptrs, 0, cell.ptr,
                                  cell.ptr) == -1


def test_q1_plan_from_lineitem_text(rf, ctx):
    """lineitem.tbl text -> column relations -> the reference's Q1 plan."""
    text, order, ln, qty, price, disc, tax, rfl, lsl, ship = datagen.lineitem_tbl(30_000, 9)
    n, rels = loaders.lineitem_q1_relations(ctx, text)
    assert n == len(order)
    p = raplan.Plan(ctx, raplan.q1_plan())
    p.set("+$logicQ1:_dateDelta", [np.array([90 * 86400])])
    for name, cols in rels.items():
        p.set_columns(name, cols, n)
    p.run()
    keep = ship <= 912470400 - 90 * 86400
    fid = (rfl == ord("N")) * 1 + (rfl == ord("R")) * 2
    g = fid.astype(np.int64) * 2 + (lsl == ord("O"))
    groups = sorted(np.unique(g[keep]).tolist())
    k0, k1, cnt = p.get("+$logicQ1:_count_order")
    assert (k0.astype(np.int64) * 2 + k1).tolist() == groups
    assert cnt.tolist() == [int((keep & (g == k)).sum()) for k in groups]
    _, _, charge = p.get("+$logicQ1:_sum_charge")
    for k, got in zip(groups, charge):
        sel = keep & (g == k)
        want = (price * (1 - disc) * (1 + tax))[sel].sum()
        assert abs(got - want) <= 1e-12 * abs(want)


@pytest.mark.parametrize("size", [1 << 20, (64 << 20) + 5, (64 << 20) - 16, (66 << 20) + 65_536 * 3 + 16,
                                  (128 << 20) - 16, 128 << 20, (128 << 20) + 5, (130 << 20) + 65_536 * 3 + 16])
def test_copies_of_any_size(rf, ctx, size):
    """rfx_copy below and past the size where its own kernel takes over:
    whole blocks, a last block, last bytes, and an unaligned source."""
    src, dst = rf.DeviceBuffer(size + 16), rf.DeviceBuffer(size + 16)
    ctx.gen_u32(src, (size + 16) // 4, 5)
    want = src.download(np.uint8, size + 16)
    for off in (0, 3):
        dst.zero()
        ctx.copy(dst, src, size, dst_off=0, src_off=off)
        ctx.synchronize()
        got = dst.download(np.uint8, size + 16)
        assert np.array_equal(got[:size], want[off:size + off]) and not got[size:].any()


def test_freed_blocks_are_handed_out_again_whole(rf):
    """Blocks that rfx_free keeps: of the size asked for or more, never two
    owners, whatever the order; sizes that are not kept."""
    rng = np.random.default_rng(3)
    live = []
    for step in range(300):
        if live and rng.random() < 0.5:
            buf, tag = live.pop(int(rng.integers(len(live))))
            assert (buf.download(np.uint8) == tag).all()
            buf.close()
        else:
            n = int(rng.choice([1, 255, 4097, 100_000, 3 << 20, (64 << 20) + 1]) + rng.integers(0, 50))
            buf = rf.DeviceBuffer(n)
            assert rf.lib().rfx_memset(buf.ptr, step % 251, n) == 0
            live.append((buf, step % 251))
    for buf, tag in live:
        assert (buf.download(np.uint8) == tag).all()



@pytest.mark.parametrize("size", [1000, 3 << 20, (64 << 20) + 1])
def test_second_free_is_refused(rf, size):
    """Freed twice: refused, whether the block is kept or the runtime's, and
    the address is handed to one owner only."""
    lib = rf.lib()

    def get():
        p = ctypes.c_void_p()
        assert lib.rfx_malloc(ctypes.byref(p), size) == 0
        return p.value

    a = get()
    assert lib.rfx_free(a) == 0
    assert lib.rfx_free(a) != 0
    b, c = get(), get()
    assert b != c
    for p, tag in ((b, 1), (c, 2)):
        assert lib.rfx_memset(p, tag, size) == 0
    host = np.empty(size, np.uint8)
    for p, tag in ((b, 1), (c, 2)):
        assert lib.rfx_memcpy_dtoh(host.ctypes.data, p, size) == 0
        assert (host == tag).all()
        assert lib.rfx_free(p) == 0



def test_freed_memory_is_free(rf):
    """rfx_mem_info after rfx_free: what was freed counts, kept or not."""
    def free():
        f, t = ctypes.c_uint64(), ctypes.c_uint64()
        assert rf.lib().rfx_mem_info(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    bufs = [rf.DeviceBuffer(48 << 20) for _ in range(6)]
    held = free()
    for b in bufs:
        b.close()
    assert free() >= held + 6 * (48 << 20)



@pytest.mark.parametrize("short", ["dst", "src"])
def test_copy_past_an_allocation_is_refused(rf, ctx, short):
    """The library's own copy kernel is not started on a range that leaves
    its allocation (the runtime's copy refused it too).  The range ends far
    beyond any memory, so the host refuses it whatever lies in between."""
    big, small = rf.DeviceBuffer(160 << 20), rf.DeviceBuffer(140 << 20)
    src, dst = (big, small) if short == "dst" else (small, big)
    with pytest.raises(rf.RfxError):
        ctx.copy(dst, src, 1 << 45)
    ctx.copy(dst, src, 140 << 20)  # whole allocations are fine
    ctx.synchronize()


def test_copies_within_one_buffer(rf, ctx):
    """Both ranges in one allocation, side by side up to its last byte."""
    half = (130 << 20) + 16
    buf = rf.DeviceBuffer(2 * half)
    ctx.gen_u32(buf, half // 2, 9)
    want = buf.download(np.uint8, half)
    ctx.copy(buf, buf, half, dst_off=half, src_off=0)
    ctx.synchronize()
    got = buf.download(np.uint8, 2 * half)
    assert np.array_equal(got[:half], want) and np.array_equal(got[half:], want)



def test_a_refused_call_leaves_the_next_launch_alone(rf, ctx):
    """An error of the runtime belongs to the call that met it: the next
    operator of the thread, which checks its launch, does not report it."""
    p = ctypes.c_void_p()
    assert rf.lib().rfx_malloc(ctypes.byref(p), (64 << 20) + 1) == 0
    assert rf.lib().rfx_free(p.value) == 0
    assert rf.lib().rfx_free(p.value) != 0
    buf = rf.DeviceBuffer(4096)
    ctx.gen_u32(buf, 1024, 5)
    assert np.array_equal(buf.download(np.uint32, 1024), datagen.u32(5, 1024))


# Row ends where a text's first and last 16-byte words are cut: every
# alignment of the first byte, lengths about whole words, one tile of 64 KB
# and two, with newlines at both ends of the text and neighbours outside it.
@pytest.mark.parametrize("size", [1, 15, 16, 17, 40, 65_519, 65_520, 65_521, 65_535, 65_536, 65_537, 131_075])
def test_row_ends_at_any_alignment(rf, ctx, size):
    rng = np.random.default_rng(size)
    for off in range(16):
        body = rng.choice(np.frombuffer(b"0123456789\n", np.uint8), size, p=[0.08] * 10 + [0.2])
        if off % 3 == 0:
            body[0] = 10
        if off % 2 == 0:
            body[-1] = 10
        text = body.tobytes()
        host = np.full(off + size + 64, 10, np.uint8)  # newlines all around
        host[off:off + size] = body
        buf = rf.DeviceBuffer.from_numpy(host)

        class At:
            ptr = buf.ptr + off
        want, _ = oracle.parse_tbl(text, ["i64"])
        for cap in (max(1, len(want[0])), 7):
            out, cells = rf.DeviceBuffer(8 * cap), rf.DeviceBuffer(16)
            types = (ctypes.c_int * 1)(loaders.TBL["i64"])
            ptrs = (ctypes.c_void_p * 1)(out.ptr)
            assert rf.lib().rfx_tbl_parse(ctx.handle, At.ptr, size, b"|", types, 1, ptrs, cap,
                                          cells.ptr, cells.ptr + 8) == 0
            assert cells.download(np.uint64, 2)[0] == len(want[0]), off
            m = min(cap, len(want[0]))
            assert np.array_equal(out.download(np.int64, m), want[0][:m]), off


def test_a_cut_tile_costs_about_a_whole_one(rf, ctx):
    """Row ends of a text one byte short of a tile (4.5 times a whole tile's
    time where the cut tile was read byte by byte), and of an unaligned one."""
    size = 65_536
    buf = rf.DeviceBuffer.from_numpy(np.frombuffer((b"12345|abcdefghij|0.25\n" * 4000)[:size + 16], np.uint8))
    out, cells = rf.DeviceBuffer(8 * size), rf.DeviceBuffer(16)
    types = (ctypes.c_int * 1)(loaders.TBL["i64"])
    ptrs = (ctypes.c_void_p * 1)(out.ptr)

    def row_ends_ms(off, n):
        best = 1e9
        for _ in range(5):
            ctx.profile(True)
            for _ in range(20):
                assert rf.lib().rfx_tbl_parse(ctx.handle, buf.ptr + off, n, b"|", types, 1, ptrs, size,
                                              cells.ptr, cells.ptr + 8) == 0
            launches, ms = ctx.profile_read("tbl.rows")
            ctx.profile(False)
            assert launches == 20
            best = min(best, ms / launches)
        return best

    whole = row_ends_ms(0, size)
    assert row_ends_ms(0, size - 1) < 3 * whole
    assert row_ends_ms(3, size - 16) < 3 * whole


# Fields that the word-wise conversion takes and those it leaves to the byte
# loop: lengths about 8 digits, signs, spaces, points first, last, twice, 0 to
# 3 digits after them, letters inside; dates of other shapes; rows short of
# fields; blocks whose text fits the stage and blocks whose text does not.
# (Delimiters that keep the columns: an 11-digit year or a decimal past 2^64
# overflows where the oracle's integers do not.)
@pytest.mark.parametrize("wide", [0, 300])
@pytest.mark.parametrize("delim", ["|", ","])
def test_field_shapes_match_oracle(rf, ctx, wide, delim):
    rng = np.random.default_rng(wide + len(delim))
    ints = ["", "0", "7", "12345678", "123456789", "99999999999", "-5", "+5", " 42", "4 2", "1x", "x1",
            "00000012", "2147483648", "12.5", "-", "18446744073709551616"]
    decs = ["", "1.5", "12.25", "1234567.89", "12345678.9", "123456789.01", ".5", "5.", "1.234", "-1.25",
            " 2.50", "1.2.3", "1e3", "12345678", "0.07", "0.1", "x", "1.x", "1.2x", "99999999.99"]
    dates = ["1994-07-01", "1992-02-29", "1998-12-31", "94-7-1", "1994/07/01", "", "1994-07", "1994-07-0x",
             " 1996-03-01", "1996-03-01 ", "+1995-+1-+2", "12345-01-01"]
    rows = []
    for i in range(1500):
        f = [rng.choice(ints), rng.choice(decs), rng.choice(dates), rng.choice(ints), rng.choice(decs),
             "A" * int(rng.integers(0, 3)), rng.choice(ints)]
        rows.append(delim.join(f[: int(rng.choice([7, 7, 7, 7, 1, 4, 6]))]) + delim * int(rng.integers(0, 3))
                    + "c" * int(rng.integers(0, wide + 1)) + ("\r" if i % 11 == 0 else ""))
    text = ("\n".join(rows) + ("\n" if wide else "")).encode()
    check(rf, ctx, text, ["i32", "f64", "date", "i64", "f64", "char", "u8"], delim)
