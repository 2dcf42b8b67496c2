"""What the operator library is timed on: the sorts, joins, aggregates, set
operations, filters, text loads and whole plans that a Red Fox program asks
of it, through the Python host interface, over the sizes from a single tile
to the largest relations that the benchmark uses.

A case is a plain dict; its "op" names the path:

  sort    stable radix sort of a key column with an optional payload
  join    a whole sort-merge join: both sorts, the search, the size read
          back, the output tuples
  group   GROUP BY over unsorted rows: sort by key, then one pass of the
          aggregate with COUNT
  setop   union, difference or intersection of two sorted sets
  select  a filter over packed tuples
  q1      TPC-H Q1 fused over columns
  tbl     lineitem text to typed columns
  strings a join on string keys: both string sorts, the search, the pairs
  plan    the reference's TPC-H Q1 plan (21 commands) over keyed relations

Columns are torch tensors on the GPU, handed over by address.  The sorts
work in place, so a program that keeps its columns copies them first, and
so do the cases here.
"""
from __future__ import annotations

import numpy as np
import torch

import redfox_amd as rf
from redfox_amd import loaders, raplan

DEV = "cuda"
Q1_CUTOFF = 2436  # days: 90 days before the end of the shipdate range
DAY = 86400
PLAN_DELTA_DAYS = 90
START_DATE = 912470400  # the Q1 plan's constant, seconds since 1970
PREFIXES = {"supplier": b"Supplier#", "customer": b"Customer#", "clerk": b"Clerk#"}
Q = "+$logicQ1:_"
PLAN_SUMS = ("sum_qty", "sum_base_price", "avg_disc_adt", "sum_disc_price", "sum_charge")

_ctx = None


def context():
    """The program's one context, on torch's default stream."""
    global _ctx
    if _ctx is None:
        _ctx = rf.Context(0)
    return _ctx


class Column:
    """A torch tensor as the library takes a buffer: by address."""

    def __init__(self, t: torch.Tensor):
        self.t = t
        self.ptr = t.data_ptr()
        self.nbytes = t.numel() * t.element_size()


def empty(n: int, dtype) -> Column:
    return Column(torch.zeros(max(int(n), 1), dtype=dtype, device=DEV))


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # A dimension table's sort: launches and latency are all there is.
        dict(name="sort_u32_4k", op="sort", n=4099, key_bytes=4, key_bits=32, val_bytes=4,
             dist="uniform"),
        # An ordinary 64-bit key column, skewed as foreign keys are.
        dict(name="sort_u64_1m", op="sort", n=1_000_003, key_bytes=8, key_bits=64, val_bytes=4,
             dist="zipf"),
        # The largest sort, the benchmark's headline.
        dict(name="sort_u32_256m", op="sort", n=1 << 28, key_bytes=4, key_bits=32, val_bytes=4,
             dist="uniform"),
        # The reference's own join size, many-to-many.
        dict(name="join_64k_256k", op="join", nr=65_536, ns=262_144, key_bits=16,
             keys="uniform"),
        # A join that fills the memory system.
        dict(name="join_16m_64m", op="join", nr=1 << 24, ns=1 << 26, key_bits=24,
             keys="uniform"),
        # GROUP BY a skewed foreign key.
        dict(name="group_32m", op="group", n=(1 << 25) + 77, groups=1 << 20, agg="sum"),
        # Set operations keep relations as sorted sets.
        dict(name="union_64m", op="setop", kind="union", na=1 << 26, nb=(1 << 26) - 12_345,
             elem_bytes=8),
        # A filter on packed tuples that keeps half.
        dict(name="select_64m", op="select", n=(1 << 26) + 33, tuple_bytes=8, keep=0.5),
        # TPC-H Q1 fused, scale factor 10.
        dict(name="q1_60m", op="q1", n=60_000_000),
        # A lineitem.tbl of scale factor 0.17: about a million rows.
        dict(name="tbl_1m", op="tbl", n_orders=1 << 18),
        # A join of two string columns as the loader leaves them.
        dict(name="strings_64k_1m", op="strings", nl=1 << 16, nr=1 << 20, prefix="supplier"),
        # The whole Q1 plan as Red Fox runs it, about four million rows.
        dict(name="plan_q1_4m", op="plan", n_orders=1 << 20),
    ]


def _log(rng, lo: float, hi: float) -> int:
    """A size between lo and hi, even over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    op = rng.choice(["sort", "sort", "join", "join", "group", "setop", "select", "q1", "tbl",
                     "strings", "plan"])
    if op == "sort":
        kb, bits, vb = rng.choice([(4, 32, 4), (4, 32, 0), (4, 24, 4), (4, 20, 8), (8, 64, 4),
                                   (8, 64, 0), (8, 64, 8), (8, 40, 4)])
        return dict(op=op, n=_log(rng, 1 << 10, (1 << 27) // (kb // 4)), key_bytes=kb,
                    key_bits=bits, val_bytes=vb, dist=rng.choice(["uniform", "zipf"]))
    if op == "join":
        nr = _log(rng, 1 << 10, 1 << 23)
        keys = rng.choice(["uniform", "fk"])
        return dict(op=op, nr=nr, ns=int(nr * rng.uniform(1, 6)), keys=keys,
                    key_bits=nr.bit_length() + (rng.choice([-1, 0, 1]) if keys == "uniform" else 1))
    if op == "group":
        n = _log(rng, 1 << 12, 1 << 26)
        return dict(op=op, n=n, groups=_log(rng, 4, min(n, 1 << 22)),
                    agg=rng.choice(["sum", "min", "max"]))
    if op == "setop":
        na = _log(rng, 1 << 10, 1 << 26)
        return dict(op=op, kind=rng.choice(["union", "difference", "intersection"]), na=na,
                    nb=max(1, int(na * rng.uniform(0.1, 1.2))), elem_bytes=rng.choice([4, 8]))
    if op == "select":
        tb = rng.choice([4, 8, 16])
        return dict(op=op, n=_log(rng, 1 << 12, (1 << 30) // tb), tuple_bytes=tb,
                    keep=round(rng.uniform(0.02, 0.98), 3))
    if op == "q1":
        return dict(op=op, n=_log(rng, 1 << 12, 60_000_000))
    if op == "tbl":
        return dict(op=op, n_orders=_log(rng, 1 << 8, 1 << 19))
    if op == "strings":
        nl = _log(rng, 1 << 8, 1 << 18)
        return dict(op=op, nl=nl, nr=int(nl * rng.uniform(1, 16)),
                    prefix=rng.choice(sorted(PREFIXES)))
    return dict(op=op, n_orders=_log(rng, 1 << 8, 1 << 21))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFFFFFF)


def _randint(g, lo: int, hi: int, n: int) -> torch.Tensor:
    return torch.randint(lo, hi, (n,), generator=g, device=DEV, dtype=torch.int64)


def _uniform(g, n: int) -> torch.Tensor:
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float64)


def _zipf(g, n: int, n_max: int, s: float = 1.1) -> torch.Tensor:
    """Ranks 1 .. n_max of a power law with exponent s."""
    e = 1.0 - s
    x = ((n_max ** e - 1.0) * _uniform(g, n) + 1.0) ** (1.0 / e)
    return x.to(torch.int64).clamp_(1, n_max)


def _mix64(x: torch.Tensor) -> torch.Tensor:
    """A bijection of 64-bit words (splitmix64's finaliser)."""
    x = (x ^ ((x >> 30) & ((1 << 34) - 1))) * -0x40A7B892E31B1A47
    x = (x ^ ((x >> 27) & ((1 << 37) - 1))) * -0x6B2FB644ECCEEE15
    return x ^ ((x >> 31) & ((1 << 33) - 1))


def _int_type(nbytes: int):
    return {1: torch.uint8, 4: torch.int32, 8: torch.int64}[nbytes]


def _in_sort(case, seed):
    g = _gen(seed)
    n, bits = case["n"], case["key_bits"]
    if case["dist"] == "zipf":
        k = _mix64(_zipf(g, n, 1 << 24))
    else:
        k = _randint(g, -(1 << 63), (1 << 63) - 1, n)
    if bits < 64:
        k &= (1 << bits) - 1
    v = torch.arange(n, device=DEV, dtype=_int_type(case["val_bytes"])) if case["val_bytes"] \
        else None
    return k.to(_int_type(case["key_bytes"])), v


def _in_join(case, seed):
    """Keys and payloads of both sides.  "fk": every left key once, every
    right key one of them; "uniform": keys repeat on both sides."""
    g = _gen(seed)
    out = []
    for side, n in enumerate((case["nr"], case["ns"])):
        if case["keys"] == "uniform":
            k = _randint(g, 0, 1 << case["key_bits"], n)
        elif side == 0:
            k = torch.randperm(n, generator=g, device=DEV)
        else:
            k = _zipf(g, n, case["nr"]) - 1
        out.append(k.to(torch.int32))
        out.append(_randint(g, 0, 1 << 32, n).to(torch.int32))
    return out


def _join_rows(case) -> int:
    """Output rows the program has room for: uniform keys give a binomial
    number of pairs, of which this is well past the largest."""
    mean = case["nr"] * case["ns"] / (1 << case["key_bits"])
    return case["ns"] if case["keys"] == "fk" else int(1.1 * mean + 20 * mean ** 0.5 + 1024)


def _in_group(case, seed):
    g = _gen(seed)
    n = case["n"]
    perm = torch.randperm(case["groups"], generator=g, device=DEV).to(torch.int32)
    keys = perm[_zipf(g, n, case["groups"]) - 1]
    return keys, _randint(g, 0, 100_001, n).to(torch.float64) / 100.0


def _in_setop(case, seed):
    """Sorted sets in unsigned order; about half of the smaller one is in
    both (members of the evenly spread even and odd slots)."""
    g = _gen(seed)
    na, nb = case["na"], case["nb"]
    m = max(na, nb)
    gap = max(2, ((1 << (8 * case["elem_bytes"] - 1)) - 1) // (2 * m))
    gap = min(gap, 1 << 40)
    slot = torch.arange(2 * m, device=DEV, dtype=torch.int64) * gap
    slot += _randint(g, 0, gap, 2 * m)
    sets = []
    for n in (na, nb):
        pick = torch.rand(m, generator=g, device=DEV) < 0.5
        idx = 2 * torch.arange(m, device=DEV) + pick
        if n < m:
            idx = idx[torch.arange(n, device=DEV) * m // n]
        sets.append(slot[idx].to(_int_type(case["elem_bytes"])))
    return sets


def _in_select(case, seed):
    """Tuples of tuple_bytes whose low (16-byte: high word's low) 32-bit
    field is uniform."""
    g = _gen(seed)
    n, tb = case["n"], case["tuple_bytes"]
    if tb == 4:
        return _randint(g, 0, 1 << 32, n).to(torch.int32)
    return _randint(g, -(1 << 63), (1 << 63) - 1, n * tb // 8)


def _in_q1(case, seed):
    g = _gen(seed)
    n = case["n"]
    ship = _randint(g, 0, 2526, n).to(torch.int32)
    flag = _randint(g, 0, 3, n).to(torch.uint8)
    status = _randint(g, 0, 2, n).to(torch.uint8)
    qty = _randint(g, 1, 51, n).to(torch.int32)
    price = qty.to(torch.float64) * (_randint(g, 90_000, 200_001, n).to(torch.float64) / 100.0)
    disc = _randint(g, 0, 11, n).to(torch.float64) / 100.0
    tax = _randint(g, 0, 9, n).to(torch.float64) / 100.0
    return ship, flag, status, qty, price, disc, tax


def _digits(v: torch.Tensor, width: int, keep_zeros: bool):
    """Decimal digits of v, and which of them the text holds."""
    cols, keep = [], []
    for i in range(width - 1, -1, -1):
        p = 10 ** i
        cols.append(((v // p) % 10 + 48).to(torch.uint8))
        keep.append(torch.ones_like(v, dtype=torch.bool) if keep_zeros or i == 0 else v >= p)
    return torch.stack(cols, 1), torch.stack(keep, 1)


def _lines(g, orders: int) -> torch.Tensor:
    """Lines of each order: 1 to 7, equally often, in any order."""
    return torch.randperm(orders, generator=g, device=DEV) % 7 + 1


def _tbl_values(case, seed):
    g = _gen(seed)
    orders = case["n_orders"]
    lines = _lines(g, orders)
    order = torch.repeat_interleave(torch.arange(1, orders + 1, device=DEV), lines)
    start = torch.repeat_interleave(torch.cumsum(lines, 0) - lines, lines)
    n = int(order.numel())
    return g, dict(order=order, part=_randint(g, 1, 200_000, n), supp=_randint(g, 1, 10_000, n),
                   line=torch.arange(n, device=DEV) - start + 1, qty=_randint(g, 1, 51, n),
                   cents=_randint(g, 90_000, 10_500_000, n), disc=_randint(g, 0, 11, n),
                   tax=_randint(g, 0, 9, n), rf=_randint(g, 0, 3, n), ls=_randint(g, 0, 2, n),
                   ship=_randint(g, 0, 2557, n), commit=_randint(g, 0, 2557, n),
                   receipt=_randint(g, 0, 2557, n), instr=_randint(g, 0, 4, n),
                   mode=_randint(g, 0, 7, n), comment=_randint(g, 10, 44, n))


def _bytes(table, pick):
    """Rows of a table of texts, padded, and which bytes belong to them."""
    width = max(len(t) for t in table)
    flat = torch.tensor([list(t.ljust(width, b"\0")) for t in table], dtype=torch.uint8,
                        device=DEV)[pick]
    return flat, flat != 0


def _in_tbl(case, seed):
    """dbgen's lineitem rows: numbers without leading zeros, comments of 10
    to 43 characters, a '|' after every field."""
    g, v = _tbl_values(case, seed)
    n = int(v["order"].numel())
    dates = np.datetime_as_string(np.datetime64("1992-01-01") + np.arange(2557))
    dates = [d.encode() for d in dates.tolist()]
    zero = torch.zeros(n, dtype=torch.int64, device=DEV)
    bar, dot = _bytes([b"|"], zero), _bytes([b"."], zero)
    cols = []
    for name, width in (("order", 8), ("part", 6), ("supp", 5), ("line", 1), ("qty", 2)):
        cols += [_digits(v[name], width, False), bar]
    cols += [_digits(v["cents"] // 100, 6, False), dot, _digits(v["cents"] % 100, 2, True), bar]
    for name in ("disc", "tax"):
        cols += [_bytes([b"0."], zero), _digits(v[name], 2, True), bar]
    cols += [_bytes([b"A", b"N", b"R"], v["rf"]), bar, _bytes([b"F", b"O"], v["ls"]), bar]
    for name in ("ship", "commit", "receipt"):
        cols += [_bytes(dates, v[name]), bar]
    cols += [_bytes([b"DELIVER IN PERSON", b"COLLECT COD", b"NONE", b"TAKE BACK RETURN"],
                    v["instr"]), bar]
    cols += [_bytes([b"REG AIR", b"AIR", b"RAIL", b"SHIP", b"TRUCK", b"MAIL", b"FOB"],
                    v["mode"]), bar]
    text = b"carefully final deposits sleep furiously ab"
    body, _ = _bytes([text], zero)
    cols += [(body, torch.arange(len(text), device=DEV)[None, :] < v["comment"][:, None]), bar,
             _bytes([b"\n"], zero)]
    chars = torch.cat([c for c, _ in cols], 1)
    keep = torch.cat([k for _, k in cols], 1)
    return chars[keep]


def _in_strings(case, seed):
    """Names of the left side (each once, in any order) and of the right
    side (drawn from them), NUL-terminated, with their offsets."""
    g = _gen(seed)
    nl, nr = case["nl"], case["nr"]
    ids = (torch.randperm(nl, generator=g, device=DEV) * 37 + 1,
           _randint(g, 0, nl, nr) * 37 + 1)
    out = []
    for i in ids:
        d, _ = _digits(i, 9, True)
        zero = torch.zeros(len(i), dtype=torch.int64, device=DEV)
        name = _bytes([PREFIXES[case["prefix"]]], zero)[0]
        text = torch.cat([name, d, torch.zeros_like(d[:, :1])], 1)
        out.append((text.contiguous().view(-1),
                    torch.arange(len(i), device=DEV, dtype=torch.int64) * text.shape[1]))
    return out


def _in_plan(case, seed):
    """lineitem as relations keyed by (LINENUMBER, ORDER), sorted by them."""
    g = _gen(seed)
    lines = _lines(g, case["n_orders"])
    od = [torch.nonzero(lines >= i).view(-1) + 1 for i in range(1, 8)]
    ln = torch.cat([torch.full_like(o, i + 1) for i, o in enumerate(od)]).to(torch.uint8)
    n = int(ln.numel())
    return dict(
        ln=ln, od=torch.cat(od).to(torch.int32), L_SHIPDATE=_randint(g, 8035, 8035 + 2557, n) * DAY,
        L_RETURNFLAG=_randint(g, 0, 3, n).to(torch.uint8),
        L_LINESTATUS=_randint(g, 0, 2, n).to(torch.uint8),
        L_QUANTITY=_randint(g, 1, 51, n).to(torch.float64),
        L_EXTENDEDPRICE=_uniform(g, n) * 1e4,
        L_DISCOUNT=_randint(g, 0, 11, n).to(torch.float64) / 100.0,
        L_TAX=_randint(g, 0, 9, n).to(torch.float64) / 100.0)


PLAN_TYPES = {"L_SHIPDATE": "i64", "L_RETURNFLAG": "u8", "L_LINESTATUS": "u8"}


def prepare(case, seed):
    op = case["op"]
    st = {"case": case}
    if op == "sort":
        k, v = _in_sort(case, seed)
        st["src"] = (Column(k), Column(v) if v is not None else None)
        st["work"] = (empty(k.numel(), k.dtype), empty(v.numel(), v.dtype) if v is not None else None)
    elif op == "join":
        st["src"] = [Column(t) for t in _in_join(case, seed)]
        st["work"] = [empty(c.t.numel(), c.t.dtype) for c in st["src"]]
        st["bounds"] = (empty(case["nr"], torch.int32), empty(case["nr"], torch.int32))
        st["total"] = rf.u64_cell(0)
        st["out"] = empty(2 * _join_rows(case), torch.int64)
    elif op == "group":
        k, v = _in_group(case, seed)
        st["src"] = (Column(k), Column(v))
        st["work"] = (empty(k.numel(), k.dtype), empty(v.numel(), v.dtype))
        cap = case["groups"]
        st["out"] = (empty(cap, torch.int32), empty(cap, torch.float64), empty(cap, torch.int32))
        st["n_out"] = empty(1, torch.int64)
        st["n"] = Column(torch.tensor([case["n"]], dtype=torch.int64, device=DEV))
    elif op == "setop":
        a, b = _in_setop(case, seed)
        st["src"] = (Column(a), Column(b))
        cap = case["na"] + (case["nb"] if case["kind"] == "union" else 0)
        st["out"], st["n_out"] = empty(cap, a.dtype), empty(1, torch.int64)
    elif op == "select":
        t = _in_select(case, seed)
        st["src"] = Column(t)
        st["out"], st["n_out"] = empty(t.numel(), t.dtype), empty(1, torch.int64)
    elif op == "q1":
        st["src"] = [Column(t) for t in _in_q1(case, seed)]
        st["out"] = empty(48, torch.float64)
    elif op == "tbl":
        st["text"] = Column(_in_tbl(case, seed))
    elif op == "strings":
        st["text"] = _in_strings(case, seed)
        st["src"] = [Column(t.data_ptr() + o) for t, o in st["text"]]
        st["work"] = [empty(c.t.numel(), torch.int64) for c in st["src"]]
        st["scratch"] = empty(max(case["nl"], case["nr"]) + 1, torch.int64)
        st["bounds"] = (empty(case["nl"], torch.int32), empty(case["nl"], torch.int32))
        st["total"] = rf.u64_cell(0)
    else:
        ctx = context()
        v = _in_plan(case, seed)
        n = int(v["ln"].numel())
        p = raplan.Plan(ctx, raplan.q1_plan())
        p.set(Q + "dateDelta", [np.array([PLAN_DELTA_DAYS * DAY])])
        key = [(Column(v["ln"]), "u8"), (Column(v["od"]), "u32")]
        torch.cuda.synchronize()
        for name, t in v.items():
            if name.startswith("L_"):
                p.set_columns(name, key + [(Column(t), PLAN_TYPES.get(name, "f64"))], n,
                              sorted_by=2)
        ctx.synchronize()
        st["plan"] = p
    return st


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def _copy_in(ctx, st):
    for s, w in zip(st["src"], st["work"]):
        if s is not None:
            ctx.copy(w, s, s.nbytes)


def _run_sort(ctx, case, st):
    _copy_in(ctx, st)
    k, v = st["work"]
    ctx.sort_pairs(k, v, case["n"], case["key_bytes"], case["key_bits"], case["val_bytes"])
    return [k.t] + ([v.t] if v is not None else [])


def _run_join(ctx, case, st):
    """Both sides sorted, then (key, left value, right value) tuples of 16
    bytes.  The program reads the size back, as it has to know what it holds."""
    _copy_in(ctx, st)
    rk, rv, sk, sv = st["work"]
    nr, ns, (lb, lc), tot = case["nr"], case["ns"], st["bounds"], st["total"]
    ctx.sort_pairs(rk, rv, nr, 4, case["key_bits"], 4)
    ctx.sort_pairs(sk, sv, ns, 4, case["key_bits"], 4)
    ctx.join_find_bounds(lb, lc, tot, rk, nr, sk, ns, 4)
    total = rf.read_u64(tot)
    if total > _join_rows(case):
        raise ValueError(f"{total} joined rows, room for {_join_rows(case)}")
    ctx.join_expand_gather(st["out"], 16, rk, 4, rv, 4, sv, 4, lb, lc, nr, tot, total, 64, 32)
    return st["out"].t, total


def _run_group(ctx, case, st):
    _copy_in(ctx, st)
    (k, v), (ok, ov, oc), n, g = st["work"], st["out"], case["n"], case["groups"]
    ctx.sort_pairs(k, v, n, 4, max(1, (g - 1).bit_length()), 8)
    ctx.reduce_count_by_key_f64(ok, ov, oc, st["n_out"], k, v, st["n"], n, 4,
                                {"sum": 0, "min": 1, "max": 2}[case["agg"]], out_cap=g)
    return {"keys": ok.t, "vals": ov.t, "counts": oc.t, "n": st["n_out"].t}


def _run_setop(ctx, case, st):
    a, b = st["src"]
    op = {"union": 0, "difference": 1, "intersection": 2}[case["kind"]]
    ctx.set_op(op, st["out"], st["n_out"], a, case["na"], b, case["nb"], case["elem_bytes"])
    return st["out"].t, st["n_out"].t


def _run_select(ctx, case, st):
    tb = case["tuple_bytes"]
    ctx.select(st["out"], st["n_out"], st["src"], case["n"], tb, 64 if tb == 16 else 0, 32, 2,
               int(case["keep"] * (1 << 32)))
    return st["out"].t, st["n_out"].t


def _run_q1(ctx, case, st):
    ctx.q1(st["out"], *st["src"], case["n"], Q1_CUTOFF)
    return st["out"].t


class _View:
    """A column that the library allocated, for torch to read in place."""

    def __init__(self, buf, n: int, typestr: str):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "version": 2,
                                         "data": (buf.ptr, False), "strides": None}


def _run_tbl(ctx, case, st):
    text = st["text"]
    cols, n, short = loaders.parse_tbl(ctx, text, loaders.LINEITEM_SPEC, "|", text.nbytes)
    kinds = [{"u32": "<i4", "u8": "|u1", "char": "|u1", "f64": "<f8", "date": "<i8"}[s]
             for s in loaders.LINEITEM_SPEC if s != "skip"]
    return [torch.as_tensor(_View(c, n, k), device=DEV)
            for c, k in zip([c for c in cols if c is not None], kinds)] + [n, short]


def _run_strings(ctx, case, st):
    """Addresses sorted by their strings on both sides, then the row pairs.
    The program keeps offsets into its texts, not addresses."""
    _copy_in(ctx, st)
    (left, right), (lb, lc), tot = st["work"], st["bounds"], st["total"]
    nl, nr = case["nl"], case["nr"]
    ctx.sort_strings(left, st["scratch"], nl)
    ctx.sort_strings(right, st["scratch"], nr)
    ctx.join_find_bounds_string(lb, lc, tot, left, nl, right, nr)
    total = rf.read_u64(tot)
    li = Column(torch.empty(max(total, 1), dtype=torch.int32, device=DEV))
    ri = Column(torch.empty(max(total, 1), dtype=torch.int32, device=DEV))
    ctx.join_main(li, ri, tot, total, lb, lc, nl)
    offs = [w.t - t.data_ptr() for w, (t, _) in zip(st["work"], st["text"])]
    return [li.t[:total], ri.t[:total], lb.t, lc.t] + offs


def _run_plan(ctx, case, st):
    p = st["plan"]
    p.run()
    return {o: p.get(Q + o) for o in PLAN_SUMS + ("count_order",)}


def run(state):
    case = state["case"]
    return globals()["_run_" + case["op"]](context(), case, state)


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how close it has to be
# ---------------------------------------------------------------------------
def work(case):
    op = case["op"]
    if op == "sort":
        b = 2 * case["n"] * (case["key_bytes"] + case["val_bytes"])
    elif op == "join":
        rows = case["ns"] * (1 if case["keys"] == "fk" else case["nr"] / (1 << case["key_bits"]))
        b = 8 * (case["nr"] + case["ns"]) + 16 * rows
    elif op == "group":
        b = 12 * case["n"] + 16 * min(case["n"], case["groups"])
    elif op == "setop":
        na, nb = case["na"], case["nb"]
        both = min(na, nb) / 2
        out = {"union": na + nb - both, "difference": na - both, "intersection": both}
        b = case["elem_bytes"] * (na + nb + out[case["kind"]])
    elif op == "select":
        b = case["n"] * case["tuple_bytes"] * (1 + case["keep"])
    elif op == "q1":
        b = 34 * case["n"] + 48 * 8
    elif op == "tbl":
        b = 4 * case["n_orders"] * (125 + 47)  # text and columns of a row
    elif op == "strings":
        width = len(PREFIXES[case["prefix"]]) + 10
        b = (8 + 8 + width) * (case["nl"] + case["nr"]) + 8 * (case["nl"] + case["nr"])
    else:
        b = 4 * case["n_orders"] * (5 + 8 + 1 + 1 + 32)  # each column, and the keys once
    return {"bytes": float(b), "flops": 0.0}


def tolerance(case):
    # Sums of up to ten million doubles: in two orders (the library's and a
    # pairwise one) they differ by 3e-16, chunks of a few hundred terms added
    # one after another by ten times that.  Everything else is whole numbers,
    # bytes, or one correctly rounded operation.
    if case["op"] in ("q1", "plan") or (case["op"] == "group" and case["agg"] == "sum"):
        return {"rel": 1e-14, "max": 1e-13, "differ": 0.0}
    return "exact"


# ---------------------------------------------------------------------------
# The same results in plain torch and numpy
# ---------------------------------------------------------------------------
def _exact_group(case, seed):
    keys, vals = _in_group(case, seed)
    k, order = torch.sort(keys.to(torch.int64), stable=True)
    k, v = k.cpu().numpy(), vals[order].cpu().numpy()
    start = np.flatnonzero(np.concatenate([[True], k[1:] != k[:-1]]))
    f = {"sum": np.add, "min": np.minimum, "max": np.maximum}[case["agg"]]
    wide = v.astype(np.longdouble) if case["agg"] == "sum" else v
    out = np.zeros(case["groups"])
    out[:len(start)] = f.reduceat(wide, start).astype(np.float64)
    return {"keys": None, "vals": out, "counts": None, "n": None}


def _exact_q1(case, seed):
    ship, flag, status, qty, price, disc, tax = _in_q1(case, seed)
    g = flag.to(torch.int64) * 2 + status
    dp = price * (1 - disc)
    cols = [qty.to(torch.float64), price, dp, dp * (1 + tax), disc]
    out = np.zeros((6, 8))
    for i in range(6):
        m = (ship <= Q1_CUTOFF) & (g == i)
        n = int(m.sum())
        s = [float(c[m].sum()) for c in cols]
        out[i, :6] = s + [n]
        if n:
            out[i, 6:] = [s[0] / n, s[1] / n]
    return out.reshape(-1)


def _exact_tbl(case, seed):
    _, v = _tbl_values(case, seed)
    f = {4: v["qty"].to(torch.float64)}
    # On the host: torch divides by a number on the GPU by multiplying.
    f[5], f[6], f[7] = (v[c].cpu().numpy() / 100.0 for c in ("cents", "disc", "tax"))
    kept = [i for i, s in enumerate(loaders.LINEITEM_SPEC) if s != "skip"]
    return [f.get(i) for i in kept] + [None, None]


def _exact_plan(case, seed):
    v = _in_plan(case, seed)
    keep = v["L_SHIPDATE"] <= START_DATE - PLAN_DELTA_DAYS * DAY
    g = v["L_RETURNFLAG"].to(torch.int64) * 2 + v["L_LINESTATUS"]
    dp = v["L_EXTENDEDPRICE"] * (1 - v["L_DISCOUNT"])
    cols = dict(sum_qty=v["L_QUANTITY"], sum_base_price=v["L_EXTENDEDPRICE"],
                avg_disc_adt=v["L_DISCOUNT"], sum_disc_price=dp, sum_charge=dp * (1 + v["L_TAX"]))
    groups = torch.unique(g[keep]).tolist()
    out = {}
    for name in PLAN_SUMS:
        out[name] = [None, None, np.array([float(cols[name][keep & (g == i)].sum())
                                           for i in groups])]
    out["count_order"] = [None, None, None]
    return out


def exact(case, seed):
    f = {"group": _exact_group, "q1": _exact_q1, "tbl": _exact_tbl,
         "plan": _exact_plan}.get(case["op"])
    return f(case, seed) if f else None
