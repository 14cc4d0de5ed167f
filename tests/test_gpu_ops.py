"""GPU parity tests: every operator through the C ABI against the CPU oracle, bit-exact."""
import numpy as np
import pytest

import oracle_lib as O
import q3_reference as Q3
from alenka_amd import _lib as L

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(ctx, a):
    return torch.as_tensor(np.ascontiguousarray(a, np.int64)).to(ctx.device)


def host(t):
    return t.cpu().numpy()


# ---- generators --------------------------------------------------------------------------
def test_generators_match_oracle(ctx):
    from alenka_amd import device as D

    for got, want in zip(D.gen_flat(ctx, 7, 5000), O.gen_flat(7, 5000)):
        assert np.array_equal(host(got), want)
    for got, want in zip(D.gen_dim(ctx, 7, 3000), O.gen_dim(7, 3000)):
        assert np.array_equal(host(got), want)
    for got, want in zip(D.gen_orders(ctx, 7, 4001, 3000), O.gen_orders(7, 4001, 3000)):
        assert np.array_equal(host(got), want)
    for got, want in zip(D.gen_fact(ctx, 7, 4001), O.gen_fact(7, 4001)):
        assert np.array_equal(host(got), want)
    code_of, codes = D.dict_first_seen(ctx, D.gen_dim(ctx, 7, 3000)[1], 5)
    w_code_of, w_codes = O.dict_first_seen(O.gen_dim(7, 3000)[1], 5)
    assert code_of == list(w_code_of)
    assert np.array_equal(host(codes), w_codes)


# ---- codec -------------------------------------------------------------------------------
CODEC_CASES = [
    ("small", lambda r, n: r.integers(0, 11, n)),
    ("dates", lambda r, n: r.integers(19920101, 19981231, n)),
    ("negative", lambda r, n: r.integers(-(1 << 40), 1 << 20, n)),
    ("constant", lambda r, n: np.full(n, -5)),
    ("full64", lambda r, n: r.integers(-(1 << 63), (1 << 63) - 1, n, dtype=np.int64)),
    ("bits33", lambda r, n: r.integers(0, 1 << 33, n)),
]


@pytest.mark.parametrize("name,gen", CODEC_CASES)
@pytest.mark.parametrize("n,seg_rows", [(1, 1000), (10007, 1000), (70000, 65536)])
def test_encode_decode(ctx, name, gen, n, seg_rows):
    from alenka_amd import device as D

    r = np.random.default_rng(n + seg_rows)
    v = np.asarray(gen(r, n), np.int64)
    col = D.Column.encode(ctx, dev(ctx, v), seg_rows)
    assert np.array_equal(host(col.decode(ctx)), v)
    words = host(col.words).view(np.uint32)
    for s in range(col.nsegs):
        sg = col.hsegs[s]
        part = v[s * seg_rows: s * seg_rows + sg.nrows]
        assert sg.vmin == part.min() and sg.vmax == part.max()
        assert sg.bits == O.load().orc_bits_for_range(int(part.min()), int(part.max()))
        if sg.bits:
            nw = (sg.nrows * sg.bits + 31) // 32
            want = O.pack(part, sg.base, sg.bits)[:nw]
            assert np.array_equal(words[sg.word_off: sg.word_off + nw], want)
    rows = np.sort(r.choice(n, size=min(n, 333), replace=False)).astype(np.int32)
    got = D.gather(ctx, col, torch.as_tensor(rows).to(ctx.device))
    assert np.array_equal(host(got), v[rows])


@pytest.mark.parametrize("n,seg_rows", [(7, 7), (2047, 5000), (2049, 2049), (4129, 4096), (6200, 3000),
                                        (2049, 8191), (2049, 8192), (20481, 8192), (18433, 8200)])
def test_codec_every_width(ctx, n, seg_rows):
    """Every code width, natural and forced, at the edges of the 2048-row tiles the codes are
    packed and unpacked in: the words are the oracle's and decode to the values."""
    from alenka_amd import device as D

    r = np.random.default_rng(n)
    for bits in range(1, 65):
        lo = 0 if bits < 63 else -(1 << 62)
        v = (r.integers(0, 1 << min(bits, 62), n) + lo).astype(np.int64)
        if bits == 64:
            v[:: 3], v[1:: 3] = -(1 << 63), (1 << 63) - 1
        for force in (0, bits, 64):
            col = D.Column.encode(ctx, dev(ctx, v), seg_rows, force_bits=force)
            words = host(col.words).view(np.uint32)
            for s in range(col.nsegs):
                sg = col.hsegs[s]
                nw = (sg.nrows * sg.bits + 31) // 32
                if force:
                    assert sg.bits == force
                if nw:
                    part = v[s * seg_rows: s * seg_rows + sg.nrows]
                    assert np.array_equal(words[sg.word_off: sg.word_off + nw], O.pack(part, sg.base, sg.bits)[:nw])
            assert np.array_equal(host(col.decode(ctx)), v), (bits, force)


# ---- scan / filter -----------------------------------------------------------------------
NAME, NUM, CMP, AND, OR = L.RPN_NAME, L.RPN_NUMBER, L.RPN_CMP, L.RPN_AND, L.RPN_OR
PREDICATES = [
    ("date_lt", [(NAME, 1, 0), (NUM, 0, 19950315), (CMP, 1, 0)]),
    ("range_and", [(NAME, 1, 0), (NUM, 0, 19940101), (CMP, 6, 0), (NAME, 1, 0), (NUM, 0, 19950101),
                   (CMP, 1, 0), (AND, 0, 0), (NAME, 3, 0), (NUM, 0, 5), (CMP, 5, 0), (AND, 0, 0)]),
    ("or", [(NAME, 0, 0), (NUM, 0, 1000), (CMP, 1, 0), (NAME, 3, 0), (NUM, 0, 10), (CMP, 4, 0), (OR, 0, 0)]),
    ("neq", [(NAME, 3, 0), (NUM, 0, 0), (CMP, 3, 0)]),
    ("decimal_const", [(NAME, 2, 0), (L.RPN_NUMBER, 2, 50000), (CMP, 2, 0)]),  # price > 500.00
    ("reverse", [(NUM, 0, 19950315), (NAME, 1, 0), (CMP, 2, 0)]),  # 19950315 > date
    ("arith", [(NAME, 2, 0), (NUM, 0, 1), (NAME, 3, 0), (L.RPN_MINUS, 0, 0), (L.RPN_MUL, 0, 0),
               (NUM, 0, 500000000), (CMP, 2, 0)]),
    ("col_col", [(NAME, 3, 0), (NAME, 0, 0), (CMP, 1, 0)]),  # disc*100 < key (scales as cm.cu:2299)
    ("const_const", [(NUM, 0, 3), (NUM, 0, 4), (CMP, 1, 0)]),
]


@pytest.mark.parametrize("name,ops", PREDICATES)
@pytest.mark.parametrize("zone_maps", [False, True])
def test_scan_filter(ctx, name, ops, zone_maps):
    from alenka_amd import device as D

    n, seg_rows = 50000, 8192
    cols = O.gen_flat(11, n)
    # sort a copy of the date column by segment so zone maps classify segments A / N / R
    cols[1] = np.sort(cols[1])
    dec = [0, 0, 2, 2]
    dcols = [D.Column.encode(ctx, dev(ctx, c), seg_rows, decimals=d) for c, d in zip(cols, dec)]
    prog, _ = L.compile_rpn(ops, dec)
    modes = None
    if zone_maps:
        modes = []
        for s in range(dcols[0].nsegs):
            mins = [c.hsegs[s].vmin for c in dcols]
            maxs = [c.hsegs[s].vmax for c in dcols]
            m = L.zone_map_check(ops, mins, maxs, dec)
            assert m == O.zone_map_check(ops, mins, maxs, dec)
            modes.append(m)
    got = host(D.scan_filter(ctx, dcols, prog, modes)).astype(np.uint32)
    if modes is None:
        want = O.compact(O.filter_mask(ops, cols, dec))
    else:
        # the reference's filter_op: 'A' keeps the whole segment, 'N' none, 'R' evaluates
        parts = []
        for s, m in enumerate(modes):
            lo, hi = s * seg_rows, min(n, (s + 1) * seg_rows)
            if m == "A":
                parts.append(np.arange(lo, hi, dtype=np.uint32))
            elif m == "R":
                seg = [c[lo:hi] for c in cols]
                parts.append(O.compact(O.filter_mask(ops, seg, dec), lo))
        want = np.concatenate(parts) if parts else np.zeros(0, np.uint32)
    assert np.array_equal(got, want)


def run_program(prog, cols):
    """A compiled integer program over numpy int64 columns (wrapping arithmetic)."""
    st = []
    for op, a, k in prog:
        if op == L.I_COL:
            st.append(cols[a] * np.int64(k))
        elif op == L.I_CONST:
            st.append(np.full(cols[0].size, k, np.int64))
        else:
            r, l = st.pop(), st.pop()
            if op == L.I_DIV:
                q = np.array([0 if y == 0 else abs(int(x)) // abs(int(y)) * (1 if (x < 0) == (y < 0) else -1)
                              for x, y in zip(l, r)], object)
                v = ((q + (1 << 63)) % (1 << 64) - (1 << 63)).astype(np.int64)
            else:
                v = {L.I_ADD: lambda: l + r, L.I_SUB: lambda: l - r, L.I_MUL: lambda: l * r,
                     L.I_AND: lambda: (l != 0) & (r != 0), L.I_OR: lambda: (l != 0) | (r != 0),
                     L.I_CMP: lambda: [None, l < r, l > r, l != r, l == r, l <= r, l >= r][a]}[op]().astype(np.int64)
            st.append(v)
    assert len(st) == 1
    return st[0]


def random_program(r, ncols, depth, lo, hi):
    """A random integer expression in postfix, `depth` operations deep at most."""
    if depth == 0 or r.random() < 0.2:
        if r.random() < 0.6:
            return [(L.I_COL, int(r.integers(ncols)), int(r.choice([1, 1, 1, 100, -3])))]
        return [(L.I_CONST, 0, int(r.choice([0, 1, 2, -7, 1000, 99999, 1 << 40, int(r.integers(lo, hi))])))]
    op = int(r.choice([L.I_ADD, L.I_SUB, L.I_MUL, L.I_DIV, L.I_CMP, L.I_CMP, L.I_AND, L.I_OR]))
    return (random_program(r, ncols, depth - 1, lo, hi) + random_program(r, ncols, depth - 1, lo, hi) +
            [(op, int(r.integers(1, 7)) if op == L.I_CMP else 0, 0)])


@pytest.mark.parametrize("n,seg_rows", [(1, 1), (63, 64), (4097, 4096), (4096, 5000), (8191, 8191), (9001, 700)])
def test_programs_random(ctx, n, seg_rows):
    """Scans and expressions of random programs (conjunctions of intervals and any shape; one
    to five values on the stack) over columns of every code width class (0, 1 to 32, 33 to 63,
    64 bits, plain), at the edges of the 4096-row tiles and of short segments, against numpy;
    the allocation-free scan gives the same rows."""
    import ctypes as C

    from alenka_amd import device as D

    r = np.random.default_rng(n * 31 + seg_rows)
    cols = [r.integers(0, 2, n), r.integers(-50000, 80000, n), r.integers(0, 1 << 31, n) * 2 + 1,
            r.integers(-(1 << 44), 1 << 44, n), np.full(n, -77), r.integers(-(1 << 63), (1 << 63) - 1, n),
            r.integers(-(1 << 62), 1 << 62, n)]
    cols = [c.astype(np.int64) for c in cols]
    dcols = [D.Column.encode(ctx, dev(ctx, c), seg_rows) for c in cols[:-1]]
    dcols.append(D.Column.plain(ctx, dev(ctx, cols[-1]), seg_rows))
    progs = [[(L.I_COL, c, 1), (L.I_CONST, 0, int(np.median(cols[c])) + d), (L.I_CMP, cmp, 0)]
             for c in range(len(cols)) for cmp in (1, 2, 4, 5, 6) for d in (0, 1)]
    progs += [p + q + [(L.I_AND, 0, 0)] for p, q in zip(progs, reversed(progs))]
    progs += [random_program(r, len(cols), d, -90000, 90000) for d in (1, 2, 3, 3, 4, 4) for _ in range(8)]
    rows = np.sort(r.choice(n, n // 2 + 1, replace=False)).astype(np.int32)
    mixed = r.permutation(rows)  # rows of one wave in several segments
    with np.errstate(over="ignore"):
        for prog in progs:
            if len(prog) > L.MAX_INSN:
                continue
            want = run_program(prog, cols)
            got = host(D.scan_filter(ctx, dcols, prog))
            assert np.array_equal(got, np.nonzero(want)[0]), prog
            out, cnt = ctx.empty(n, torch.int32), C.c_uint64()
            L.check(ctx.lib.aln_scan_filter_noalloc(ctx.h, D._cols_array(dcols), len(dcols), seg_rows,
                                                    L.insn_array(prog), len(prog), None, D._p(out), n, C.byref(cnt)))
            assert np.array_equal(host(out)[: cnt.value], got), prog
            assert np.array_equal(host(D.eval_rows(ctx, dcols, prog)), want), prog
            for sel in (rows, mixed):
                assert np.array_equal(host(D.eval_rows(ctx, dcols, prog, torch.as_tensor(sel).to(ctx.device))),
                                      want[sel]), prog
    for c, dc in zip(cols, dcols):
        assert np.array_equal(host(D.gather(ctx, dc, torch.as_tensor(mixed).to(ctx.device))), c[mixed])
        assert np.array_equal(host(D.gather(ctx, dc)), c)
        for a, b in ((0, n), (n // 3, n - n // 4), (n - 1, n)):
            assert np.array_equal(host(dc.decode(ctx, a, b)), c[a:b])


def test_eval_revenue(ctx):
    from alenka_amd import device as D

    n = 40000
    cols = O.gen_flat(3, n)
    dec = [0, 0, 2, 2]
    dcols = [D.Column.encode(ctx, dev(ctx, c), 4096, decimals=d) for c, d in zip(cols, dec)]
    ops = [(NAME, 2, 0), (NUM, 0, 1), (NAME, 3, 0), (L.RPN_MINUS, 0, 0), (L.RPN_MUL, 0, 0)]
    prog, prec = L.compile_rpn(ops, dec, mode=1)
    want, wprec = O.eval_expr(ops, cols, dec)
    assert prec == wprec == 4
    rows = np.arange(0, n, 3, dtype=np.int32)
    got = host(D.eval_rows(ctx, dcols, prog, torch.as_tensor(rows).to(ctx.device)))
    assert np.array_equal(got, want[rows])
    assert np.array_equal(want, cols[2] * (100 - cols[3]))  # closed form of the trace


# ---- group-by ----------------------------------------------------------------------------
def test_groupby_flat_query(ctx):
    """Flat 1M-row filter + GROUP BY key: SUM(price*(1-discount)), COUNT(key), one segment."""
    from alenka_amd import device as D

    n = 200000
    key, date, price, disc = O.gen_flat(42, n)
    sel = date < 19950315
    rev = price[sel] * (100 - disc[sel])
    k = key[sel]
    ok, ov = D.groupby(ctx, [dev(ctx, k)], [dev(ctx, rev), dev(ctx, rev)], [L.AGG_SUM, L.AGG_COUNT])
    wk, wv = O.groupby([k], [rev, rev], [L.AGG_SUM, L.AGG_COUNT])
    assert np.array_equal(host(ok[0]), wk[0])
    assert np.array_equal(host(ov[0]), wv[0])
    assert np.array_equal(host(ov[1]), wv[1])
    # FP64 check of the exact decimal sums: within 1e-12 of a Kahan-summed float oracle
    g = {int(a): i for i, a in enumerate(wk[0][:50])}
    for kk, i in g.items():
        m = k == kk
        f = O.kahan_sum((price[sel][m] / 100.0) * (1.0 - disc[sel][m] / 100.0))
        assert abs(wv[0][i] / 1e4 - f) <= 1e-12 * abs(f)


@pytest.mark.parametrize("nkeys", [1, 2, 3])
def test_groupby_hash_order(ctx, nkeys):
    """Multi-segment output order: ascending MurmurHash64A of the key tuple (merge.cu)."""
    from alenka_amd import device as D

    r = np.random.default_rng(nkeys)
    n = 30000
    keys = [r.integers(0, 300, n), r.integers(-50, 50, n), r.integers(19920101, 19920131, n)][:nkeys]
    v = r.integers(-1000, 1000, n)
    bounds = [0, 10000, 20000, n]
    aggs = [L.AGG_SUM, L.AGG_COUNT, L.AGG_MIN, L.AGG_MAX]
    ok, ov = D.groupby(ctx, [dev(ctx, x) for x in keys], [dev(ctx, v)] * 4, aggs, order=L.ORDER_HASH,
                       seed=100)
    wk, wv = O.groupby(keys, [v] * 4, aggs, seg_bounds=bounds, seed=100)
    for a, b in zip(ok, wk):
        assert np.array_equal(host(a), b)
    for a, b in zip(ov, wv):
        assert np.array_equal(host(a), b)


def test_groupby_wide_keys(ctx):
    """Key tuples wider than 63 bits take the sort-based path."""
    from alenka_amd import device as D

    r = np.random.default_rng(5)
    n = 20000
    k1 = r.integers(-(1 << 62), 1 << 62, 200)[r.integers(0, 200, n)]
    k2 = r.integers(0, 1 << 20, 50)[r.integers(0, 50, n)]
    v = r.integers(0, 1 << 30, n)
    for order in (L.ORDER_KEYS, L.ORDER_HASH):
        ok, ov = D.groupby(ctx, [dev(ctx, k1), dev(ctx, k2)], [dev(ctx, v), dev(ctx, v)],
                           [L.AGG_SUM, L.AGG_COUNT], order=order)
        wk, wv = O.groupby([k1, k2], [v, v], [L.AGG_SUM, L.AGG_COUNT],
                           seg_bounds=[0, 1, n] if order == L.ORDER_HASH else None)
        for a, b in zip(ok + ov, wk + wv):
            assert np.array_equal(host(a), b)


def _gb_check(ctx, keys, vals, aggs, order=None, bounds=None):
    from alenka_amd import device as D

    order = L.ORDER_KEYS if order is None else order
    ok, ov = D.groupby(ctx, [dev(ctx, x) for x in keys], [dev(ctx, v) for v in vals], aggs, order=order, seed=100)
    wk, wv = O.groupby(keys, vals, aggs, seg_bounds=bounds, seed=100)
    for a, b in zip(ok + ov, wk + wv):
        assert np.array_equal(host(a), b)
    return len(wk[0])


AGGS4 = [L.AGG_SUM, L.AGG_COUNT, L.AGG_MIN, L.AGG_MAX]


@pytest.mark.parametrize("n", [1, 1000, 3_000_007])
def test_groupby_no_keys(ctx, n):
    """No GROUP BY: one group, a reduction over all rows (reduce, select.cu:549), against
    numpy's sum / min / max / len; f64 SUM within 1e-12 of math.fsum, f64 MIN / MAX exact."""
    import math

    from alenka_amd import device as D

    r = np.random.default_rng(n)
    v = r.integers(-(1 << 40), 1 << 40, n)
    ok, ov = D.groupby(ctx, [], [dev(ctx, v)] * 4, AGGS4)
    assert ok == [] and all(x.numel() == 1 for x in ov)
    assert [int(host(x)[0]) for x in ov] == [int(v.sum()), n, int(v.min()), int(v.max())]
    f = r.standard_normal(n) * 1e6
    fb = torch.as_tensor(f.view(np.int64)).to(ctx.device)
    _, fv = D.groupby(ctx, [], [fb] * 3, [L.AGG_FSUM, L.AGG_FMIN, L.AGG_FMAX])
    got = [host(x).view(np.float64)[0] for x in fv]
    want = math.fsum(f)
    assert abs(got[0] - want) <= 1e-12 * max(1.0, np.abs(f).sum())
    assert got[1] == f.min() and got[2] == f.max()


def test_groupby_constant_key(ctx):
    """Keys that never vary: one group with that key."""
    n = 500_001
    r = np.random.default_rng(7)
    assert _gb_check(ctx, [np.full(n, -42, np.int64)], [r.integers(-100, 100, n)] * 4, AGGS4) == 1


@pytest.mark.parametrize("case", ["g10", "g1000_2keys", "dense_2e20", "zipf_sparse", "retry_3m", "clustered"])
def test_groupby_paths(ctx, case):
    """The group-by paths against the oracle: direct-indexed LDS slots (10 groups), hashed
    LDS slots over direct-indexed globals (1000 groups of 2 keys), direct-indexed globals
    (2^20 codes), the hash table with hot keys (Zipf over 40-bit keys), more than 2^20
    groups (the first table overflows; the rows are aggregated again in a 2n table), and
    sorted input (runs of equal keys in adjacent lanes); key order and hash order."""
    r = np.random.default_rng(len(case))
    if case == "g10":
        n = 2_000_003
        keys = [r.integers(0, 10, n) * 7 + 19920101]
    elif case == "g1000_2keys":
        n = 1_000_000
        keys = [r.integers(0, 40, n), r.integers(-12, 13, n)]
    elif case == "dense_2e20":
        n = 1 << 20
        keys = [r.integers(0, 1 << 20, n)]
    elif case == "zipf_sparse":
        n = 2_000_000
        z = np.minimum(r.zipf(1.2, n), 1 << 20)
        keys = [z * 1_000_003 + 5]
    elif case == "retry_3m":
        n = 3_000_000
        keys = [r.integers(0, 1 << 40, n)]
    else:
        n = 1_500_000
        keys = [np.sort(r.integers(0, 100_000, n))]
    v = r.integers(-(1 << 30), 1 << 30, n)
    g = _gb_check(ctx, keys, [v] * 4, AGGS4)
    assert g > 1
    bounds = [0, n // 3, 2 * n // 3, n]
    _gb_check(ctx, keys, [v, v], [L.AGG_SUM, L.AGG_COUNT], order=L.ORDER_HASH, bounds=bounds)


@pytest.mark.parametrize("n", [1, 2047, 2049, 20000, (1 << 20) + 5])
@pytest.mark.parametrize("widths", [(2,), (3, 2), (1000,), (40, 90), (2, 5, 3, 3)])
def test_groupby_few_groups(ctx, n, widths):
    """Accumulators in LDS: one to four keys, every aggregate (with and without a COUNT among
    them, eight at once), both orders, at the edges of the 2048-row blocks, and (from 2^20 rows,
    where the key ranges come from a sample first) with a key the sample misses; f64 columns with
    NaN, infinities and -0.0."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + len(widths))
    keys = [r.integers(0, w, n).astype(np.int64) - w // 2 for w in widths]
    if n > 1 << 20:
        keys[0][12345] = 5000  # in none of the sampled runs
    vals = [r.integers(-(1 << 62), 1 << 62, n).astype(np.int64) for _ in range(4)]
    aggs = [L.AGG_SUM, L.AGG_MIN, L.AGG_MAX, L.AGG_SUM]
    wk, wv = O.groupby(keys, vals, aggs, seed=100)
    hk, hv = O.groupby(keys, vals, aggs, seg_bounds=[0, n // 2, n] if n > 1 else [0, n], seed=100)
    f = r.integers(-1000, 1000, n) / 8.0  # sums of these are exact in any order
    code = np.zeros(n, np.int64)
    for k in keys:
        code = code * 12000 + (k + 6000)
    ucode, inv = np.unique(code, return_inverse=True)
    bits = lambda x: np.ascontiguousarray(x).view(np.int64)  # noqa: E731
    special = f.copy()
    special[:: 5], special[1:: 7], special[2:: 11] = np.nan, np.inf, -0.0
    fmin, fmax = np.full(ucode.size, np.inf), np.full(ucode.size, -np.inf)
    ok = ~np.isnan(special)
    np.minimum.at(fmin, inv[ok], special[ok])
    np.maximum.at(fmax, inv[ok], special[ok])
    fsum = np.bincount(inv, weights=f, minlength=ucode.size)
    cnt = np.bincount(inv, minlength=ucode.size)
    dk, dv = [dev(ctx, k) for k in keys], [dev(ctx, v) for v in vals]
    df, ds = dev(ctx, bits(f)), dev(ctx, bits(special))
    for order, (ek, ev) in ((L.ORDER_KEYS, (wk, wv)), (L.ORDER_HASH, (hk, hv))):
        ok_, ov = D.groupby(ctx, dk, dv, aggs, order=order, seed=100)
        for x, y in zip(ok_ + ov, list(ek) + list(ev)):
            assert np.array_equal(host(x), y)
    ok_, ov = D.groupby(ctx, dk, [df, ds, ds, None, dv[0], dv[1], dv[2], df],
                        [L.AGG_FSUM, L.AGG_FMIN, L.AGG_FMAX, L.AGG_COUNT, L.AGG_SUM, L.AGG_MIN, L.AGG_MAX, L.AGG_FSUM])
    for x, y in zip(ok_, wk):
        assert np.array_equal(host(x), y)
    f64 = lambda t: host(t).view(np.float64)  # noqa: E731
    assert np.array_equal(f64(ov[0]), fsum) and np.array_equal(f64(ov[7]), fsum)
    assert np.array_equal(f64(ov[1]), fmin) and np.array_equal(f64(ov[2]), fmax)
    assert np.array_equal(host(ov[3]), cnt)
    for x, y in zip(ov[4:7], wv[:3]):
        assert np.array_equal(host(x), y)
    if len(wk[0]) > 1:
        with pytest.raises(L.AlnError) as e:
            D.groupby(ctx, dk, dv, aggs, cap=len(wk[0]) - 1)
        assert e.value.code == L.ALN_E_CAPACITY


@pytest.mark.parametrize("n,case", [(n, c) for n in (196607, 196608, 1 << 20, (1 << 20) + 4097)
                                    for c in ("2keys", "wide", "skewed", "hot", "edge")]
                         + [(2047 * 4096, "2keys"), (2047 * 4096 + 1, "hot")])
def test_groupby_parts(ctx, n, case):
    """Rows moved into parts of the code range (from 196608 rows on; from 2048 tiles of 4096 rows on
    eight tiles are counted per block): a few thousand codes of two keys, 2^21 codes, a skewed column (parts of several blocks), one key almost everywhere, and
    the smallest code range; all aggregates over one and several value columns, with and without
    a COUNT, in both orders."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + len(case))
    keys = {"2keys": lambda: [r.integers(-20, 100, n), r.integers(0, 100, n)],
            "wide": lambda: [r.integers(0, 1 << 21, n)],
            "skewed": lambda: [np.minimum(r.zipf(1.15, n), 1 << 17) + 7],
            "hot": lambda: [np.where(r.random(n) < 0.98, 4000, r.integers(0, 1 << 18, n))],
            "edge": lambda: [r.integers(0, 8193, n)]}[case]()
    keys = [k.astype(np.int64) for k in keys]
    v, w = r.integers(-(1 << 40), 1 << 40, n).astype(np.int64), r.integers(-1000, 1000, n).astype(np.int64)
    _gb_check(ctx, keys, [v, v, w, v], AGGS4)
    _gb_check(ctx, keys, [v], [L.AGG_SUM])
    _gb_check(ctx, keys, [v, w], [L.AGG_MIN, L.AGG_COUNT], order=L.ORDER_HASH, bounds=[0, n // 2, n])
    f = r.integers(-1000, 1000, n) / 8.0
    code = keys[0] * 1000 + keys[1] if len(keys) == 2 else keys[0]
    ucode, inv = np.unique(code, return_inverse=True)
    fmin, fmax = np.full(ucode.size, np.inf), np.full(ucode.size, -np.inf)
    np.minimum.at(fmin, inv, f)
    np.maximum.at(fmax, inv, f)
    df = dev(ctx, f.view(np.int64))
    ok, ov = D.groupby(ctx, [dev(ctx, k) for k in keys], [df, df, df], [L.AGG_FSUM, L.AGG_FMIN, L.AGG_FMAX])
    assert ok[0].numel() == ucode.size
    for got, want in zip(ov, (np.bincount(inv, weights=f), fmin, fmax)):
        assert np.array_equal(host(got).view(np.float64), want)


@pytest.mark.parametrize("n,outlier,nv", [((1 << 21) + 4099, (1 << 22) - 1, 8), ((1 << 20) + 5, 1 << 20, 2),
                                          ((1 << 20) + 5, 1 << 27, 2), ((1 << 20) + 5, 1 << 62, 2), ((1 << 20) + 5, 900, 2)])
@pytest.mark.parametrize("order", [L.ORDER_KEYS, L.ORDER_HASH])
def test_groupby_sample_missed(ctx, n, outlier, nv, order):
    """A key that the sample of a few-groups call misses, in each route the call then starts again
    with: direct-indexed tables with atomics (2^22 codes of eight accumulators and the row count are
    too many for parts), parts, the hash table (codes over 2^26 or 2n), sorting (tuples over 63
    bits) and accumulators in LDS again; without a COUNT among the aggregates, whose table would
    tell the groups, and with one."""
    r = np.random.default_rng(n + outlier % 1000)
    for keys in ([r.integers(0, 200, n)], [r.integers(0, 4, n), r.integers(0, 3, n)]):
        keys = [k.astype(np.int64) for k in keys]
        keys[0][[12345, n - 20000]] = outlier, outlier - 1  # in none of the sampled runs
        cols = [r.integers(-(1 << 40), 1 << 40, n).astype(np.int64) for _ in range(nv)]
        bounds = [0, n // 2, n] if order == L.ORDER_HASH else None
        _gb_check(ctx, keys, cols, [L.AGG_SUM, L.AGG_MIN, L.AGG_MAX, L.AGG_SUM] * (nv // 4) or [L.AGG_SUM, L.AGG_MIN],
                  order=order, bounds=bounds)
        _gb_check(ctx, keys, cols[:1] * 2, [L.AGG_SUM, L.AGG_COUNT], order=order, bounds=bounds)


@pytest.mark.parametrize("kind,n,sort", [("blocks", 9_000_000, False), ("sorted", 9_000_000, False),
                                         ("one_row_runs", 2_000_000, True), ("zipf", 2_000_000, False),
                                         ("hot", 2_000_000, False), ("hot_tail", 2_000_000, True),
                                         ("blocks", 200_000, False), ("one_row_runs", 200_000, True)])
def test_groupby_wide_route(ctx, kind, n, sort):
    """Wide keys whose rows come in blocks of a few repeated keys, in order, skewed, with one hot key
    and few or many others, or all different: the groups, and the route a sample chooses for them
    (few global additions: the table, however the rows are clustered; many: sorting)."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + len(kind))
    gid = {"blocks": lambda: np.repeat(r.integers(0, 600, n // 16 + 1), 16)[:n],
           "sorted": lambda: np.sort(r.integers(0, 20000, n)),
           "one_row_runs": lambda: r.integers(0, n, n),
           "zipf": lambda: np.minimum(r.zipf(2.0, n), 1 << 20),
           "hot": lambda: np.where(r.random(n) < 0.99, 0, r.integers(0, n, n)),
           "hot_tail": lambda: np.where(r.random(n) < 0.5, 0, r.integers(0, n, n))}[kind]().astype(np.int64)
    v = r.integers(-1000, 1000, n).astype(np.int64)
    cnt = np.bincount(gid)
    g = np.nonzero(cnt)[0]
    want = [g * 1_000_003 + 5, np.bincount(gid, weights=v)[g].astype(np.int64), cnt[g]]
    dk, dv = dev(ctx, gid * 1_000_003 + 5), dev(ctx, v)
    ctx.profile()
    ctx.profile_reset()
    try:
        k, out = D.groupby(ctx, [dk], [dv, dv], [L.AGG_SUM, L.AGG_COUNT])
        assert ctx.profile_get("groupby_sorted_agg")[1] == int(sort)
    finally:
        ctx.profile(False)
    for x, y in zip(k + out, want):
        assert np.array_equal(host(x), y)


@pytest.mark.parametrize("n,groups", [(1 << 20, 30000), (1_100_000, 34000), (1_100_000, 40000), (300_007, 9000)])
def test_groupby_hash_order_by_key(ctx, n, groups):
    """Hash order of sorted wide keys around 32 rows a group, from where the rows are sorted by key
    and the groups by hash, against the oracle; two keys and one, several aggregates."""
    r = np.random.default_rng(n + groups)
    gid = r.integers(0, groups, n)
    v, w = r.integers(-(1 << 40), 1 << 40, n).astype(np.int64), r.integers(-1000, 1000, n).astype(np.int64)
    for keys in ([gid * 0x12345677 + 5], [gid * 1_000_003 - 77, gid % 5 * 10_000_019]):
        _gb_check(ctx, [k.astype(np.int64) for k in keys], [v, v, w, v], AGGS4, order=L.ORDER_HASH, bounds=[0, n // 2, n])


def gb_raw(ctx, keys, vals, aggs, order, outk, outv, cap):
    """aln_groupby into given output tensors: (status, number of groups)."""
    import ctypes as C

    p = lambda ts: (C.c_void_p * max(1, len(ts)))(*[t.data_ptr() for t in ts])  # noqa: E731
    g = C.c_uint64()
    rc = ctx.lib.aln_groupby(ctx.h, p(keys), len(keys), p(vals), (C.c_int32 * max(1, len(aggs)))(*aggs), len(vals),
                             keys[0].numel(), order, 100, p(outk), p(outv), cap, C.byref(g))
    return rc, g.value


# sizes, key columns: the routes of key codes of at most 63 bits
GB_ROUTES = {"few": (5000, lambda r, n: [r.integers(0, 7, n), r.integers(0, 30, n)]),
             "sampled": ((1 << 20) + 5, lambda r, n: [r.integers(0, 7, n)]),
             "missed": ((1 << 20) + 5, lambda r, n: [np.where(np.arange(n) == 12345, 5000, r.integers(0, 7, n))]),
             "direct": (150000, lambda r, n: [r.integers(0, 30000, n)]),
             "parts": (300000, lambda r, n: [r.integers(0, 30000, n)]),
             "table": (150000, lambda r, n: [r.integers(0, 300, n) * 1000003]),
             "sorted": (300007, lambda r, n: [r.integers(0, n // 2, n) * 1000003])}


@pytest.mark.parametrize("order", [L.ORDER_KEYS, L.ORDER_HASH])
@pytest.mark.parametrize("route", GB_ROUTES)
def test_groupby_in_place_and_short(ctx, route, order):
    """Outputs that lie over the inputs: every row is read before a group is written, also when the
    call starts again; and with too short a capacity nothing is written, the number needed is
    returned, and the inputs are still there for the next call."""
    n, gen = GB_ROUTES[route]
    r = np.random.default_rng(n)
    keys = [k.astype(np.int64) for k in gen(r, n)]
    v = r.integers(-(1 << 40), 1 << 40, n).astype(np.int64)
    bounds = [0, n // 2, n] if order == L.ORDER_HASH else None
    aggs = [L.AGG_SUM, L.AGG_MAX]
    wk, wv = O.groupby(keys, [v, v], aggs, seg_bounds=bounds, seed=100)
    g = len(wk[0])
    dk, dv = [dev(ctx, k) for k in keys], [dev(ctx, v), dev(ctx, v)]
    for cap in (0, 1, g - 1):
        assert gb_raw(ctx, dk, dv, aggs, order, dk, dv, cap) == (L.ALN_E_CAPACITY, g)
        for x, y in zip(dk + dv, keys + [v, v]):
            assert np.array_equal(host(x), y)
    assert gb_raw(ctx, dk, dv, aggs, order, dk, dv, g) == (L.ALN_OK, g)
    for x, y in zip(dk + dv, list(wk) + list(wv)):
        assert np.array_equal(host(x)[:g], y)


@pytest.mark.parametrize("order", [L.ORDER_KEYS, L.ORDER_HASH])
@pytest.mark.parametrize("case,n", [("tuples", 300007), ("codes", 3_000_017), ("parts", 400_003)])
def test_groupby_workspace_limit(ctx, case, n, order):
    """Routes of less workspace where the first choice does not fit: wide tuples sorted without
    packed rows (half the bytes), wide codes of many groups in the table instead of sorted, the
    direct tables without moved rows; the results are the same, and below what any route needs the
    call fails, and a context that has failed goes on working."""
    from alenka_amd import device as D

    r = np.random.default_rng(n)
    keys = {"tuples": lambda: [r.integers(0, n // 3, n) * 0x1234567ABCD1 - (1 << 62),
                               r.integers(0, 2, n) * ((1 << 62) + 5)],
            "codes": lambda: [r.integers(0, 30000, n) * 1_000_003],
            "parts": lambda: [r.integers(0, 60000, n)]}[case]()
    keys = [k.astype(np.int64) for k in keys]
    v, w = r.integers(-(1 << 40), 1 << 40, n).astype(np.int64), r.integers(-1000, 1000, n).astype(np.int64)
    vals, aggs = ([v, v, w, v], AGGS4) if case == "tuples" else ([v, v], [L.AGG_SUM, L.AGG_COUNT])
    bounds = [0, n // 2, n] if order == L.ORDER_HASH else None
    # all routes fit (with what the chunks of a small workspace leave unused); the second only
    full, less = {"tuples": (100 * n, 58 * n), "codes": (80 * n, 110 << 20), "parts": (40 * n, (8 if order == L.ORDER_KEYS else 14) * n)}[case]
    first, second = {"tuples": (("groupby_pack", 1), ("groupby_sorted_agg", 1)),
                     "codes": (("groupby_sorted_agg", 1), ("groupby_insert", 1)),
                     "parts": (("groupby_move", 1), ("groupby_move", 0))}[case]
    for limit, seen in ((full, first), (less, second)):
        c = D.Context(0)
        L.check(c.lib.aln_set_workspace_limit(c.h, limit))
        c.profile()
        _gb_check(c, keys, vals, aggs, order=order, bounds=bounds)
        assert c.profile_get(seen[0])[1] == seen[1], seen
        c.close()
    c = D.Context(0)
    L.check(c.lib.aln_set_workspace_limit(c.h, 1 << 16))
    with pytest.raises(L.AlnError) as e:
        _gb_check(c, keys, vals, aggs, order=order, bounds=bounds)
    assert e.value.code == L.ALN_E_NOMEM
    L.check(c.lib.aln_set_workspace_limit(c.h, 0))
    _gb_check(c, keys, vals, aggs, order=order, bounds=bounds)
    c.close()


M64 = (1 << 64) - 1
MUR = 0xC6A4A7935BD1E995


def murmur_step(k):
    k = k * MUR & M64
    return (k ^ k >> 47) * MUR & M64


def murmur_unstep(x):
    """The k of murmur_step(k) = x (every part of it is a bijection)."""
    inv = pow(MUR, -1, 1 << 64)
    x = x * inv & M64
    return (x ^ x >> 47) * inv & M64


@pytest.mark.parametrize("n,run", [(1 << 17, 2), (300007, 40), (1 << 20, 3), (1_800_001, 3), (1_800_001, 1200)])
def test_groupby_clustered(ctx, n, run):
    """Wide keys whose rows come in runs: few and many groups, and (600001 groups) more than the
    first hash table takes."""
    r = np.random.default_rng(n + run)
    keys = [np.arange(n, dtype=np.int64) // run * 0x1234567ABCD1 - (1 << 61)]
    v = r.integers(-(1 << 40), 1 << 40, n).astype(np.int64)
    _gb_check(ctx, keys, [v, v], [L.AGG_SUM, L.AGG_COUNT])
    _gb_check(ctx, keys, [v], [L.AGG_MAX], order=L.ORDER_HASH, bounds=[0, n // 2, n])


@pytest.mark.parametrize("n", [1, 64, 65, 1023, 1025, 4096, 5121, 70001, (1 << 17) - 1, 1 << 17, 300007, (1 << 20) + 77])
@pytest.mark.parametrize("case", ["unique", "pairs", "runs", "one", "wide_values"])
def test_groupby_sorted(ctx, n, case):
    """GROUP BY by sorting: key tuples of more than 63 bits with every group one row, two rows,
    runs over several 64-row words and 1024-row waves, one group; every aggregate (f64 with NaN),
    one to eight distinct value columns; key and hash order; and (from 2^17 rows) one key of 40 to
    62 bits with many groups, whose rows are sorted instead of hashed."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + len(case))
    groups = {"unique": 4 * n, "pairs": max(1, n // 2), "runs": max(1, n // 1500), "one": 1,
              "wide_values": max(1, n // 3)}[case]
    gid = r.integers(0, groups, n)
    k0 = gid * 0x1234567ABCD1 - (1 << 62)
    k1 = (gid % 7) * ((1 << 60) + 12345) - (1 << 62)
    v, w = r.integers(-(1 << 62), 1 << 62, n).astype(np.int64), r.integers(-1000, 1000, n).astype(np.int64)
    bounds = [0, n // 2, n] if n > 1 else [0, n]
    keys = [k0.astype(np.int64), k1.astype(np.int64)]
    if case == "one":  # two rows of other keys make the tuples wide
        for i, x in zip(range(min(n, 2)), (-(1 << 63), (1 << 63) - 1)):
            keys[0][i] = x
    _gb_check(ctx, keys, [v, v, w, v], AGGS4)
    _gb_check(ctx, keys, [v, v, w], [L.AGG_MAX, L.AGG_COUNT, L.AGG_MIN], order=L.ORDER_HASH, bounds=bounds)
    if case == "wide_values":
        cols = [r.integers(-1000, 1000, n).astype(np.int64) for _ in range(8)]
        _gb_check(ctx, keys, cols, [L.AGG_SUM] * 8)
        _gb_check(ctx, keys, cols[:5], [L.AGG_SUM] * 5, order=L.ORDER_HASH, bounds=bounds)
    if n >= (1 << 17) - 1 and case != "one":
        one = [(gid * 0x1234567 + 5).astype(np.int64)]
        _gb_check(ctx, one, [v, w], [L.AGG_SUM, L.AGG_COUNT])
        _gb_check(ctx, one, [v, w], [L.AGG_SUM, L.AGG_MIN], order=L.ORDER_HASH, bounds=bounds)
    f = r.integers(-1000, 1000, n) / 8.0
    nan = f.copy()
    nan[r.random(n) < 0.3] = np.nan
    _, inv = np.unique(keys[0], return_inverse=True)
    g = inv.max() + 1
    fmin, fmax = np.full(g, np.inf), np.full(g, -np.inf)
    ok = ~np.isnan(nan)
    np.minimum.at(fmin, inv[ok], nan[ok])
    np.maximum.at(fmax, inv[ok], nan[ok])
    bits = [dev(ctx, x.view(np.int64)) for x in (f, nan, nan)]
    gk, gv = D.groupby(ctx, [dev(ctx, k) for k in keys], bits, [L.AGG_FSUM, L.AGG_FMIN, L.AGG_FMAX])
    for got, want in zip(gv, (np.bincount(inv, weights=f, minlength=g), fmin, fmax)):
        assert np.array_equal(host(got).view(np.float64), want)
    if g > 1:
        for order in (L.ORDER_KEYS, L.ORDER_HASH):
            with pytest.raises(L.AlnError) as e:
                D.groupby(ctx, [dev(ctx, k) for k in keys], [dev(ctx, v)], [L.AGG_SUM], order=order, cap=int(g) - 1)
            assert e.value.code == L.ALN_E_CAPACITY


def test_results_complete_on_return(ctx):
    """What a call returns is whole for every stream, not only the context's: groups of the
    few-groups kernels (which hand the host their number themselves) read at once on another
    stream, and a join counted on one stream whose pairs are written on another."""
    import ctypes as C

    from alenka_amd import device as D

    r = np.random.default_rng(3)
    other = torch.cuda.Stream()
    n = 3000
    key, v = r.integers(0, 1000, n).astype(np.int64), r.integers(-1000, 1000, n).astype(np.int64)
    uk, inv = np.unique(key, return_inverse=True)
    want = [np.bincount(inv, weights=v).astype(np.int64), np.bincount(inv)]
    build, probe = r.permutation(4000)[:2000].astype(np.int64), r.integers(0, 4000, 50000).astype(np.int64)
    row = np.full(4000, -1)
    row[build] = np.arange(2000)
    dk, dv, db, dp = (dev(ctx, x) for x in (key, v, build, probe))
    torch.cuda.synchronize()
    for _ in range(20):
        (gk,), gv = D.groupby(ctx, [dk], [dv, dv], [L.AGG_SUM, L.AGG_COUNT])
        with torch.cuda.stream(other):
            got = [x.clone() for x in (gk, *gv)]
        cnt = C.c_uint64()
        L.check(ctx.lib.aln_hash_join_count(ctx.h, D._p(db), 2000, D._p(dp), 50000, C.byref(cnt)))
        pi, bi = ctx.empty(cnt.value, torch.int32), ctx.empty(cnt.value, torch.int32)
        L.check(ctx.lib.aln_set_stream(ctx.h, C.c_void_p(other.cuda_stream)))
        try:
            L.check(ctx.lib.aln_hash_join_pairs(ctx.h, D._p(pi), D._p(bi), cnt.value, C.byref(cnt)))
        finally:
            L.check(ctx.lib.aln_set_stream(ctx.h, C.c_void_p(ctx.stream.cuda_stream)))
        torch.cuda.synchronize()
        for x, y in zip(got, [uk] + want):
            assert np.array_equal(host(x), y)
        hit = np.nonzero(row[probe] >= 0)[0]
        assert np.array_equal(host(pi), hit) and np.array_equal(host(bi), row[probe[hit]])


def test_groupby_hash_clash(ctx):
    """Key tuples made to share a MurmurHash64A stay groups of their own in hash order: by hash,
    then by key tuple."""
    from alenka_amd import device as D

    seed, r = 100, np.random.default_rng(5)
    h0 = seed ^ (16 * MUR & M64)
    after = lambda k: (h0 ^ murmur_step(k)) * MUR & M64  # noqa: E731
    sgn = lambda x: x - (1 << 64) if x >> 63 else x  # noqa: E731
    tuples = []
    for _ in range(50):
        a, b, c = (int(x) for x in r.integers(0, 1 << 63, 3))
        d = murmur_unstep(after(a) ^ after(c) ^ murmur_step(b))
        tuples += [(a, b), (c, d)]
        ha, hc = (L.murmur64a(np.array([sgn(x) for x in t], np.int64).tobytes(), seed) for t in ((a, b), (c, d)))
        assert ha == hc
    pick = r.integers(0, len(tuples), 5000)
    keys = [np.array([sgn(tuples[i][j]) for i in pick], np.int64) for j in range(2)]
    v = r.integers(-1000, 1000, 5000).astype(np.int64)
    (g0, g1), (s, cnt) = D.groupby(ctx, [dev(ctx, k) for k in keys], [dev(ctx, v)] * 2, [L.AGG_SUM, L.AGG_COUNT],
                                   order=L.ORDER_HASH, seed=seed)
    want = {}
    for x, y, z in zip(*keys, v):
        t = want.setdefault((int(x), int(y)), [0, 0])
        t[0] += int(z)
        t[1] += 1
    order = sorted(want, key=lambda t: (L.murmur64a(np.array(t, np.int64).tobytes(), seed), t))
    assert list(zip(host(g0).tolist(), host(g1).tolist())) == order
    assert host(s).tolist() == [want[t][0] for t in order] and host(cnt).tolist() == [want[t][1] for t in order]


# ---- join --------------------------------------------------------------------------------
@pytest.mark.parametrize("case", ["dense", "dups", "sparse", "wide", "dense_big"])
def test_hash_join(ctx, case):
    """dense: unique keys over a range of <= 64 per build row (bitmap + rank index); dups:
    repeated keys (sorted runs in the hash table); sparse / wide: unique keys over a range
    too wide for the bitmap (hash table), the second beyond 2^32; dense_big: 2M probe rows."""
    from alenka_amd import device as D

    r = np.random.default_rng(9 + len(case))
    nb, npb = 20000, 50000
    dups = case == "dups"
    if dups:
        build = r.integers(0, 5000, nb)
    elif case == "sparse":
        build = r.permutation(1 << 24)[:nb].astype(np.int64) * 7 - 300000
    elif case == "wide":
        build = r.integers(-(1 << 40), 1 << 40, nb)
        build = np.unique(build)[:nb]
        nb = build.size
    else:
        if case == "dense_big":
            nb, npb = 500000, 2000000
        build = r.permutation(1 << 20 if nb < 100000 else 1 << 22)[:nb].astype(np.int64) - 300000
    lo, hi = int(build.min()) - 1000, int(build.max()) + 1000
    probe = np.concatenate([build[r.integers(0, nb, npb // 2)], r.integers(lo, hi, npb - npb // 2)])
    probe = r.permutation(probe)
    pi, bi = D.hash_join(ctx, dev(ctx, build), dev(ctx, probe))
    pi, bi = host(pi).astype(np.uint32), host(bi).astype(np.uint32)
    # expected: probe-row order, then ascending build row
    if not dups:  # unique build keys: one pair per probe row whose key is a build key
        pos = {int(b): j for j, b in enumerate(build)}
        want_p = np.array([i for i, p in enumerate(probe) if int(p) in pos], np.uint32)
        want_b = np.array([pos[int(probe[i])] for i in want_p], np.uint32)
        assert np.array_equal(pi, want_p) and np.array_equal(bi, want_b)
    else:
        exp = []
        where = {}
        for j, b in enumerate(build):
            where.setdefault(int(b), []).append(j)
        for i, p in enumerate(probe):
            for j in where.get(int(p), []):
                exp.append((i, j))
        exp = np.array(exp, np.uint32).reshape(-1, 2)
        assert np.array_equal(np.stack([pi, bi], 1), exp)
    if case != "dense_big":  # same multiset as the reference's sort-merge join
        ol, orr = O.join_sortmerge(probe, build)
        assert sorted(zip(ol.tolist(), orr.tolist())) == sorted(zip(pi.tolist(), bi.tolist()))


@pytest.mark.parametrize("ntiles", [1, 2, 64, 65, 1023, 1025, 16383, 16384, 16385])
def test_scan_tile_counts(ctx, ntiles):
    """Row ids of a scan whose tile counts are scanned by one wave row, one block (up to 16384
    tiles) or the tile scan: one-row segments, of which about a third pass."""
    from alenka_amd import device as D

    r = np.random.default_rng(ntiles)
    v = r.integers(0, 3, ntiles).astype(np.int64)
    col = D.Column.plain(ctx, dev(ctx, v), 1)
    got = host(D.scan_filter(ctx, [col], [(L.I_COL, 0, 1), (L.I_CONST, 0, 1), (L.I_CMP, 4, 0)]))
    assert np.array_equal(got, np.nonzero(v == 1)[0])


J_NOKEY = 0x9A7C0F53D1B24E86 - (1 << 64)  # the join table's mark of a free entry


@pytest.mark.parametrize("nb,npb,distinct", [(1, 1, 1), (3, 2049, 1), (2048, 2047, 300), (70001, 6145, 9000),
                                             (5000, 100003, 2)])
def test_hash_join_sparse_keys(ctx, nb, npb, distinct):
    """Build keys spread over the int64 range, repeated (runs of 1 to nb rows, more pairs than
    probe rows) and unique, with the extremes and the free-entry mark among them, at the edges
    of the 2048-row probe tiles; in one call with a short capacity, and in two."""
    import ctypes as C

    from alenka_amd import device as D

    r = np.random.default_rng(nb + npb)
    pool = np.unique(np.concatenate([r.integers(-(1 << 62), 1 << 62, max(distinct, nb)),
                                     [J_NOKEY, 0, -(1 << 63), (1 << 63) - 1]]))
    pool = r.permutation(pool)[-max(distinct, nb):]
    pool[0] = J_NOKEY if J_NOKEY not in pool else pool[0]
    for build in (pool[r.integers(0, distinct, nb)], pool[:nb]):
        probe = np.concatenate([pool, r.integers(-(1 << 62), 1 << 62, 8), [J_NOKEY]])[r.integers(0, distinct + 9, npb)]
        order = np.argsort(build, kind="stable")
        lo, hi = (np.searchsorted(build[order], probe, side=x) for x in ("left", "right"))
        want_p = np.repeat(np.arange(npb), hi - lo)
        want_b = np.concatenate([order[a:b] for a, b in zip(lo, hi)]) if npb else order[:0]
        db, dp = dev(ctx, build), dev(ctx, probe)
        for cap in (None, 1):
            pi, bi = D.hash_join(ctx, db, dp, cap=cap)
            assert np.array_equal(host(pi), want_p) and np.array_equal(host(bi), want_b)
    D.join_rows(ctx, pi, npb, False)  # takes the workspace: the counted join is over
    n = C.c_uint64()
    assert ctx.lib.aln_hash_join_pairs(ctx.h, D._p(pi), D._p(bi), pi.numel(), C.byref(n)) == L.ALN_E_ARG


@pytest.mark.parametrize("width", [3, 8, 25])
def test_like_dict_matches_oracle(ctx, width):
    """LIKE over a dictionary on the device against the oracle's restatement of gpu_regex
    (filter.cu:67-129), with entries that fill the width (where the position budget binds)."""
    from alenka_amd import device as D

    r = np.random.default_rng(width)
    alpha = list("ab.")
    entries = ["".join(r.choice(alpha, size=int(r.integers(0, width + 1)))) for _ in range(777)]
    entries += ["BUILDING"[:width], "aaab"[:width], ""]
    pats = ["%", "", "a%", "%b", "%a%b%", "a?b", "?%", "%.%", "%ab", "a.b%", "%%a", "b?%?a"]
    for pat in pats:
        bits = D.like_dict(ctx, entries, width, pat)
        got = [(int(bits[i >> 5]) >> (i & 31)) & 1 == 1 for i in range(len(entries))]
        want = [O.like(e, width, pat) for e in entries]
        assert got == want, pat


@pytest.mark.parametrize("nrows,nidx", [(1, 0), (31, 5), (32, 64), (100003, 250000), (5000, 0)])
def test_join_rows(ctx, nrows, nidx):
    """Semi/anti reduction: rows that occur among a join side's pair indices (with
    duplicates), or do not, in ascending order - the oracle's sort + unique and set
    difference (operators.cu:1357-1399)."""
    from alenka_amd import device as D

    r = np.random.default_rng(nrows + nidx)
    idx = r.integers(0, nrows, nidx).astype(np.int32)
    t = torch.as_tensor(idx if nidx else np.zeros(1, np.int32)).to(ctx.device)[:nidx]
    semi = np.unique(idx)
    anti = np.setdiff1d(np.arange(nrows), semi)
    assert np.array_equal(host(D.join_rows(ctx, t, nrows, False)), semi.astype(np.int32))
    assert np.array_equal(host(D.join_rows(ctx, t, nrows, True)), anti.astype(np.int32))
    if len(anti) > 1:
        with pytest.raises(L.AlnError) as e:
            D.join_rows(ctx, t, nrows, True, cap=len(anti) - 1)
        assert e.value.code == L.ALN_E_CAPACITY


@pytest.mark.parametrize("nrows,nidx", [(1, 1), (8192, 2048), (8193, 2049), (70000, 5000), (1 << 22, 30000)])
@pytest.mark.parametrize("order", ["sorted", "shuffled", "mixed"])
def test_join_rows_windows(ctx, nrows, nidx, order):
    """Row marks through the LDS window (indices in order, duplicates, both ends of the table),
    directly (indices all over it), and both in one call; entries that are no row are left out."""
    from alenka_amd import device as D

    r = np.random.default_rng(nrows + nidx)
    idx = np.sort(r.integers(0, nrows, nidx)).astype(np.int64)
    idx[0], idx[-1] = 0, nrows - 1
    if order == "shuffled":
        idx = r.permutation(idx)
    elif order == "mixed" and nidx > 3000:
        idx[2048:] = r.permutation(idx[2048:])
        idx[100:110] = nrows  # not a row
    t = torch.as_tensor(idx.astype(np.uint32).view(np.int32)).to(ctx.device)
    semi = np.unique(idx[idx < nrows])
    assert np.array_equal(host(D.join_rows(ctx, t, nrows, False)), semi)
    assert np.array_equal(host(D.join_rows(ctx, t, nrows, True)), np.setdiff1d(np.arange(nrows), semi))


# ---- sort / top-k ------------------------------------------------------------------------
@pytest.mark.parametrize("wide", [False, True])
def test_sort_and_topk(ctx, wide):
    from alenka_amd import device as D

    r = np.random.default_rng(21 + wide)
    n = 60000
    if wide:
        keys = [r.integers(-(1 << 62), 1 << 62, n), r.integers(0, 1 << 40, n)]
    else:
        keys = [r.integers(0, 1000, n), r.integers(19920101, 19981231, n)]
    desc = [1, 0]
    perm = host(D.sort_keys(ctx, [dev(ctx, k) for k in keys], desc)).astype(np.uint32)
    want = O.order(keys, desc)
    assert np.array_equal(perm, want)
    for k in (1, 10, 100):
        top = host(D.topk(ctx, [dev(ctx, x) for x in keys], desc, k)).astype(np.uint32)
        assert np.array_equal(top, want[:k])


@pytest.mark.parametrize("n,k", [(1, 1), (2048, 512), (2049, 32), (2049, 40), (4099, 64), (70001, 100),
                                 (70001, 512), (600000, 3), (1500000, 100)])
@pytest.mark.parametrize("kind", ["spread", "ties", "sorted", "one", "wide"])
def test_topk_candidates(ctx, n, k, kind):
    """ORDER BY .. LIMIT k at the edges of its routes (all rows in one block; chunks of 64 to
    1024 rows; few, many and too many candidates) against the stable multi-key sort: spread
    first keys with the int64 extremes among them, few distinct ones, rows already in (and
    against) the order, one value everywhere, and keys of more than 64 bits together."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + k)
    k0 = {"spread": lambda: r.integers(-(1 << 62), 1 << 62, n), "ties": lambda: r.integers(0, 7, n),
          "sorted": lambda: np.arange(n) * 3 - 50, "one": lambda: np.full(n, -5),
          "wide": lambda: r.integers(-(1 << 40), 1 << 40, n)}[kind]().astype(np.int64)
    if kind == "spread" and n > 8:
        k0[3], k0[n - 2], k0[n // 2] = -(1 << 63), (1 << 63) - 1, -(1 << 63)
    k1 = r.integers(0, 5, n).astype(np.int64)
    k2 = r.integers(-(1 << 30), 1 << 30, n).astype(np.int64)
    for keys, desc in (([k0], [0]), ([k0], [1]), ([k0, k1], [1, 0]), ([k0, k1, k2], [0, 1, 1]),
                       ([k0, k1, k2, k0], [1, 1, 0, 0])):
        got = host(D.topk(ctx, [dev(ctx, x) for x in keys], desc, k)).astype(np.int64)
        cols = [(~x if d else x) for x, d in zip(keys, desc)]  # ~x reverses the int64 order
        want = np.lexsort([np.arange(n)] + cols[::-1])[:k]
        assert np.array_equal(got, want), (len(keys), desc)


@pytest.mark.parametrize("n", [1_600_000, 3_145_728, 3_145_729, 4_000_003])
@pytest.mark.parametrize("kind", ["copies64", "half", "long", "few_long", "heavy_low"])
def test_sort_crowded_windows(ctx, n, kind):
    """ORDER BY of codes that crowd the bucket path's bins (64 copies of every code, of half of
    them), or overflow its windows (one code of 5000 rows, several, a crowd of codes in one bucket),
    with more windows than are resident at once and at the sizes where wide windows begin; the
    permutation is the stable one, also in the GROUP BY that sorts by codes."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + len(kind))
    spread = lambda ids: ids * np.int64(0x1234567ABCDEF)  # noqa: E731  (wraps)
    with np.errstate(over="ignore"):
        key = spread(r.integers(0, n * 4, n))
        if kind == "copies64":
            key = spread(r.integers(0, n // 64, n))
        elif kind == "half":
            key[: n // 2] = spread(r.integers(0, n // 128, n // 2))
        elif kind == "long":
            key[r.choice(n, 5000, replace=False)] = key[7]
        elif kind == "few_long":
            for i in range(20):
                key[r.choice(n, 3000, replace=False)] = key[i]
        else:
            key[r.choice(n, 30000, replace=False)] = key[7] + r.integers(0, 1000, 30000)
    got = host(D.sort_keys(ctx, [dev(ctx, key)], [0]))
    assert np.array_equal(got, np.argsort(key, kind="stable"))
    ucode, cnt = np.unique(key, return_counts=True)
    (k,), (c,) = D.groupby(ctx, [dev(ctx, key)], [None], [L.AGG_COUNT])
    assert np.array_equal(host(k), ucode) and np.array_equal(host(c), cnt)


def test_radix_sort_pairs(ctx):
    from alenka_amd import device as D

    r = np.random.default_rng(3)
    n = 100003
    k = r.integers(0, 1 << 63, n, dtype=np.int64).astype(np.uint64) | np.uint64(1 << 63)
    kt = torch.as_tensor(k.view(np.int64)).to(ctx.device)
    vt = torch.arange(n, dtype=torch.int32, device=ctx.device)
    D.radix_sort_pairs(ctx, kt, vt, 64)
    order = np.argsort(k, kind="stable")
    assert np.array_equal(host(kt).view(np.uint64), k[order])
    assert np.array_equal(host(vt), order.astype(np.int32))


RADIX_CASES = [(1, 64, "u"), (2, 64, "u"), (4095, 64, "u"), (4096, 17, "u"), (4097, 8, "u"), (100003, 5, "u"),
               ((1 << 20) + 3, 64, "u"), ((1 << 20) + 3, 40, "few"), (1 << 20, 64, "const"), ((1 << 20) + 5, 64, "hi"),
               (300001, 64, "hi")]


@pytest.mark.parametrize("n,bits,kind", RADIX_CASES)
def test_radix_sort_pairs_shapes(ctx, n, bits, kind):
    """Stable sort by the low `bits` bits: tile-boundary sizes, one-pass sorts (sorted through
    a temporary), digits that every item shares (skipped passes at 2^20 items and up), all
    keys equal, and bits above `bits` that must not take part."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + bits)
    if kind == "u":
        k = r.integers(0, 1 << 63, n, dtype=np.int64).astype(np.uint64) * np.uint64(2) + r.integers(0, 2, n).astype(np.uint64)
    elif kind == "few":  # 16 values, digits 0-1 and 3-4 shared by every key
        k = r.integers(0, 16, n).astype(np.uint64) << np.uint64(20)
    elif kind == "const":
        k = np.full(n, 0x0123456789ABCDEF, np.uint64)
    else:  # only the top digit varies
        k = r.integers(0, 256, n).astype(np.uint64) << np.uint64(56)
    kt = torch.as_tensor(k.view(np.int64)).to(ctx.device)
    vt = torch.arange(n, dtype=torch.int32, device=ctx.device)
    D.radix_sort_pairs(ctx, kt, vt, bits)
    low = k & np.uint64((1 << bits) - 1 if bits < 64 else 0xFFFFFFFFFFFFFFFF)
    order = np.argsort(low, kind="stable")
    assert np.array_equal(host(vt), order.astype(np.int32))
    assert np.array_equal(host(kt).view(np.uint64), k[order])


@pytest.mark.parametrize("n,shape", [(60000, "wide_small_last"), (60000, "small_first_wide"),
                                     ((1 << 20) + 7, "wide_small_last"), ((1 << 20) + 7, "three")])
def test_sort_keys_lsd_shapes(ctx, n, shape):
    """ORDER BY keys whose codes exceed 64 bits: one sort per key, last key first, each one
    reading its key through the permutation so far; a key of at most 8 bits is a one-pass
    sort whose permutation is both read and written."""
    from alenka_amd import device as D

    r = np.random.default_rng(n + len(shape))
    full = r.integers(-(1 << 63), (1 << 63) - 1, n, dtype=np.int64)
    small = r.integers(-100, 100, n)
    if shape == "wide_small_last":
        keys, desc = [full, small], [0, 1]
    elif shape == "small_first_wide":
        keys, desc = [small, full], [1, 0]
    else:
        keys, desc = [small, full, r.integers(0, 1 << 40, n)], [0, 1, 1]
    perm = host(D.sort_keys(ctx, [dev(ctx, k) for k in keys], desc)).astype(np.uint32)
    assert np.array_equal(perm, O.order(keys, desc))


@pytest.mark.parametrize("case", ["uniform_desc", "u32_keys", "u28_keys", "tiny_buckets", "overflow", "dups", "two_keys"])
def test_sort_keys_bucket_path(ctx, case):
    """ORDER BY of 2^20 rows and more with at least four varying digits: two passes on the
    top two digits, then each bucket sorted in LDS; buckets too large for a block fall back
    to the digit passes.  Cases: uniform 64-bit keys DESC; 32- and 28-bit keys (many small
    buckets per block); >256 buckets in some blocks (two ordinal passes); buckets of 4096
    rows (fallback); 300 distinct values (fallback); two keys packed into one code."""
    from alenka_amd import device as D

    r = np.random.default_rng(len(case) * 7)
    desc = [0]
    if case == "uniform_desc":
        n = 3_000_001
        keys, desc = [r.integers(-(1 << 63), (1 << 63) - 1, n, dtype=np.int64)], [1]
    elif case == "u32_keys":
        n = 2_000_003
        keys = [r.integers(0, 1 << 32, n)]
    elif case == "u28_keys":
        n = 1_500_000
        keys = [r.integers(0, 1 << 28, n) - (1 << 27)]
    elif case == "tiny_buckets":
        n = 1_100_000
        top = np.concatenate([r.integers(0, 60000, 100_000), 60000 + r.integers(0, 5536, n - 100_000)])
        keys = [(top << 24) | r.integers(0, 1 << 24, n)]
    elif case == "overflow":
        n = 4_000_000
        keys = [(r.integers(0, 4, n) << 40) | r.integers(0, 1 << 32, n)]
    elif case == "dups":
        n = 2_000_000
        keys = [r.integers(-(1 << 62), 1 << 62, 300)[r.integers(0, 300, n)]]
    else:
        n = 1_200_000
        keys, desc = [r.integers(0, 1 << 20, n), r.integers(-(1 << 30), 1 << 30, n)], [1, 0]
    perm = host(D.sort_keys(ctx, [dev(ctx, k) for k in keys], desc)).astype(np.uint32)
    assert np.array_equal(perm, O.order(keys, desc))


def test_hash_rows(ctx):
    from alenka_amd import device as D

    r = np.random.default_rng(4)
    a, b = r.integers(-(1 << 62), 1 << 62, 1000), r.integers(0, 100, 1000)
    h = host(D.hash_rows(ctx, [dev(ctx, a), dev(ctx, b)], 100)).view(np.uint64)
    for i in range(0, 1000, 37):
        tup = np.array([a[i], b[i]], np.int64).tobytes()
        assert int(h[i]) == O.murmur64a(tup, 100)


# ---- fused q3 pipeline -------------------------------------------------------------------
def encode_q3(ctx, t, seg_rows):
    from alenka_amd import device as D

    enc = lambda a, d=0: D.Column.encode(ctx, dev(ctx, a), seg_rows, decimals=d)
    dim = [enc(t["c_key"]), enc(t["c_seg"])]
    mid = [enc(t["o_key"]), enc(t["o_cust"]), enc(t["o_date"]), enc(t["o_prio"])]
    fact = [enc(t["l_okey"]), enc(t["l_price"], 2), enc(t["l_disc"], 2), enc(t["l_ship"])]
    return dim, mid, fact


def q3_args(t, dim, mid, fact):
    building = int(t["code_of"][Q3.SEGMENTS.index("BUILDING")])
    D_ = dict(cols=dim, ranges=[(1, building, building)])
    M_ = dict(cols=mid, ranges=[(2, -(1 << 63), Q3.DATE - 1)])
    F_ = dict(cols=fact, ranges=[(3, Q3.DATE + 1, (1 << 63) - 1)])
    spec = dict(d_key=0, m_key=0, m_fk=1, m_g1=2, m_g2=3, f_fk=0, f_x=1, f_y=2, a0=0, a1=1, b0=100, b1=-1)
    return D_, M_, F_, spec


@pytest.mark.parametrize("join", ["bitmap", "hash"])
@pytest.mark.parametrize("scale,seg_rows", [(0.02, 4096), (0.1, 65536)])
def test_star_q3(ctx, scale, seg_rows, join):
    from alenka_amd import device as D

    ndim, norders = int(150000 * scale), int(1500000 * scale)
    t = Q3.tables(1234, ndim, norders)
    top, groups, stats = Q3.run(t)
    dim, mid, fact = encode_q3(ctx, t, seg_rows)
    D_, M_, F_, spec = q3_args(t, dim, mid, fact)
    rows, g, st = D.star_agg(ctx, D_, M_, F_, spec, limit=10, want_groups=True, force_hash=join == "hash")
    assert rows == top
    if join == "bitmap":  # a prepared query gives the same answer on every run
        q = D.StarQuery(ctx, D_, M_, F_, spec, limit=10)
        for _ in range(2):
            r2, _, st2 = q.run()
            assert r2 == top and st2.fact_pass == stats["fact_pass"]
    assert st.dim_pass == stats["dim_pass"] and st.mid_pass == stats["mid_pass"]
    assert st.fact_pass == stats["fact_pass"] and st.groups == stats["groups"]
    assert np.array_equal(host(g), groups)


def star_expected(t, dr, mr, fr, limit=10, coef=(0, 1, 100, -1)):
    """Oracle answer of a star query with range lists (col, lo, hi) on the q3 tables: the same
    sort-merge joins and sort-based group-by as the q3 reference run, SUM((a0 + a1 price) *
    (b0 + b1 disc)) with coef = (a0, a1, b0, b1) (q3: price * (100 - disc))."""
    cols = dict(d=[t["c_key"], t["c_seg"]], m=[t["o_key"], t["o_cust"], t["o_date"], t["o_prio"]],
                f=[t["l_okey"], t["l_price"], t["l_disc"], t["l_ship"]])

    def ids(k, ranges):
        m = np.ones(len(cols[k][0]), bool)
        for c, lo, hi in ranges:
            m &= (cols[k][c] >= lo) & (cols[k][c] <= hi)
        return O.compact(m)

    c_ids, o_ids, l_ids = ids("d", dr), ids("m", mr), ids("f", fr)
    pl, _ = O.join_sortmerge(t["o_cust"][o_ids], t["c_key"][c_ids])
    olc1 = o_ids[pl]
    ql, qr = O.join_sortmerge(t["l_okey"][l_ids], t["o_key"][olc1])
    lrow, orow = l_ids[ql], olc1[qr]
    a0, a1, b0, b1 = coef
    rev = (a0 + a1 * t["l_price"][lrow]) * (b0 + b1 * t["l_disc"][lrow])
    gk, gv = O.groupby([t["o_key"][orow], t["o_date"][orow], t["o_prio"][orow]], [rev, rev],
                       [L.AGG_SUM, L.AGG_COUNT])
    perm = O.order([gv[0], gk[1]], [1, 0])
    top = [(int(gk[0][i]), int(gk[1][i]), int(gk[2][i]), int(gv[0][i]), int(gv[1][i])) for i in perm[:limit]]
    groups = np.stack([gk[0], gk[1], gk[2], gv[0], gv[1]], axis=1) if len(gk[0]) else np.zeros((0, 5), np.int64)
    return top, groups, len(c_ids), len(olc1), len(lrow)


@pytest.mark.parametrize("join", ["bitmap", "hash"])
@pytest.mark.parametrize("case", ["wide", "multi", "zone", "dense"])
def test_star_scan_shapes(ctx, case, join):
    """Segments the scans' fast decoder cannot take (codes wider than 31 bits, several ranges
    on a table) run the generic staged decoder, zone maps skip ('N') or pass ('A') whole
    segments, and with no filter every fact row joins (more joined rows per wave than its
    deferred slots hold, so the scan adds the rest itself); every shape gives the oracle's
    answer."""
    from alenka_amd import device as D

    t = Q3.tables(77, 3000, 30000)
    seg_rows = 4096
    enc = lambda a, d=0, fb=0: D.Column.encode(ctx, dev(ctx, a), seg_rows, decimals=d, force_bits=fb)
    wide = case == "wide"
    dim = [enc(t["c_key"], fb=36 if wide else 0), enc(t["c_seg"])]
    mid = [enc(t["o_key"], fb=40 if wide else 0), enc(t["o_cust"], fb=36 if wide else 0), enc(t["o_date"]),
           enc(t["o_prio"])]
    fact = [enc(t["l_okey"], fb=40 if wide else 0), enc(t["l_price"], 2), enc(t["l_disc"], 2), enc(t["l_ship"])]
    building = int(t["code_of"][Q3.SEGMENTS.index("BUILDING")])
    lo, hi = -(1 << 63), (1 << 63) - 1
    if case == "multi":
        dr = [(1, building, building), (0, lo, 2400)]
        mr = [(2, lo, Q3.DATE - 1), (2, 19930101, hi)]
        fr = [(3, Q3.DATE + 1, hi), (2, 2, 8)]
    elif case == "dense":  # every row of every table passes
        dr, mr, fr = [(1, lo, hi)], [(2, lo, hi)], [(3, lo, hi)]
    elif case == "zone":  # fact and mid ranges on the (clustered) order key itself
        kmid = int(np.median(t["o_key"]))
        dr = [(1, building, building)]
        mr = [(0, lo, kmid)]
        fr = [(0, int(t["l_okey"][len(t["l_okey"]) // 5]), kmid)]
    else:
        dr, mr, fr = [(1, building, building)], [(2, lo, Q3.DATE - 1)], [(3, Q3.DATE + 1, hi)]
    top, groups, dpass, mpass, fpass = star_expected(t, dr, mr, fr)
    spec = dict(d_key=0, m_key=0, m_fk=1, m_g1=2, m_g2=3, f_fk=0, f_x=1, f_y=2, a0=0, a1=1, b0=100, b1=-1)
    rows, g, st = D.star_agg(ctx, dict(cols=dim, ranges=dr), dict(cols=mid, ranges=mr), dict(cols=fact, ranges=fr),
                             spec, limit=10, want_groups=True, force_hash=join == "hash")
    assert rows == top
    assert (st.dim_pass, st.mid_pass, st.fact_pass) == (dpass, mpass, fpass)
    assert np.array_equal(host(g), groups)


@pytest.mark.parametrize("join", ["bitmap", "hash"])
def test_star_q3_orders_shuffled(ctx, join):
    """The orders table's rows in random order (the answer does not depend on it): every
    mid tile's passing keys then span most of the key range, so the top-k reads the rows of
    its candidate groups from every tile instead of the few a key-ordered table leaves."""
    from alenka_amd import device as D

    t = Q3.tables(4321, 3000, 30000)
    perm = np.random.default_rng(5).permutation(len(t["o_key"]))
    t2 = dict(t)
    for k in ("o_key", "o_cust", "o_date", "o_prio"):
        t2[k] = t[k][perm]
    top, groups, stats = Q3.run(t)
    assert Q3.run(t2)[0] == top
    dim, mid, fact = encode_q3(ctx, t2, 4096)
    D_, M_, F_, spec = q3_args(t2, dim, mid, fact)
    rows, g, st = D.star_agg(ctx, D_, M_, F_, spec, limit=10, want_groups=True, force_hash=join == "hash")
    assert rows == top
    assert (st.dim_pass, st.mid_pass, st.fact_pass) == (stats["dim_pass"], stats["mid_pass"], stats["fact_pass"])
    assert np.array_equal(host(g), groups)


@pytest.mark.parametrize("join", ["bitmap", "hash"])
@pytest.mark.parametrize("case", ["dense", "filtered"])
def test_star_topk_ties(ctx, case, join):
    """SUM(1) per joined row: a group's sum is its row count (1 to 7), so many groups tie at
    the top-k threshold and the order falls to (o_date, o_key).  Every row passing gives
    thousands of candidate groups at the threshold (the top-k then looks up every group's mid
    row); the q3 filters give fewer (each candidate's row found by its code)."""
    from alenka_amd import device as D

    t = Q3.tables(91, 3000, 30000)
    seg_rows = 4096
    dim, mid, fact = encode_q3(ctx, t, seg_rows)
    lo, hi = -(1 << 63), (1 << 63) - 1
    building = int(t["code_of"][Q3.SEGMENTS.index("BUILDING")])
    if case == "dense":
        dr, mr, fr = [(1, lo, hi)], [(2, lo, hi)], [(3, lo, hi)]
    else:
        dr, mr, fr = [(1, building, building)], [(2, lo, Q3.DATE - 1)], [(3, Q3.DATE + 1, hi)]
    top, groups, dpass, mpass, fpass = star_expected(t, dr, mr, fr, coef=(1, 0, 1, 0))
    kth = np.sort(groups[:, 3])[::-1][9]  # the 10th largest sum: groups at or above it are candidates
    assert int((groups[:, 3] >= kth).sum()) > (2048 if case == "dense" else 10)
    spec = dict(d_key=0, m_key=0, m_fk=1, m_g1=2, m_g2=3, f_fk=0, f_x=1, f_y=2, a0=1, a1=0, b0=1, b1=0)
    for want in (False, True):  # the top-k alone, and with the group list
        rows, g, st = D.star_agg(ctx, dict(cols=dim, ranges=dr), dict(cols=mid, ranges=mr),
                                 dict(cols=fact, ranges=fr), spec, limit=10, want_groups=want,
                                 force_hash=join == "hash")
        assert rows == top
        assert (st.dim_pass, st.mid_pass, st.fact_pass) == (dpass, mpass, fpass)
        if want:
            assert np.array_equal(host(g), groups)


@pytest.mark.parametrize("join", ["bitmap", "hash"])
def test_star_ranges_reused_then_changed(ctx, join):
    """A call on the same key columns as the last one reuses their key ranges and checks them
    on the device.  Here the dimension key and the orders' foreign key are rewritten in place
    (same buffers and segment count, keys moved up by 100000, new zone maps): the reused
    ranges are stale (with them no key would fall in the dimension bitmap), so the query must
    run again with fresh ranges and give the oracle's answer for the new contents."""
    import ctypes

    import torch
    from alenka_amd import device as D

    t = Q3.tables(1234, 3000, 30000)
    seg_rows = 4096
    t2 = dict(t)
    t2["c_key"] = t["c_key"] + 100000
    t2["o_cust"] = t["o_cust"] + 100000
    enc = lambda a, d=0, fb=0: D.Column.encode(ctx, dev(ctx, a), seg_rows, decimals=d, force_bits=fb)
    dim = [enc(t["c_key"], fb=20), enc(t["c_seg"])]
    mid = [enc(t["o_key"]), enc(t["o_cust"], fb=20), enc(t["o_date"]), enc(t["o_prio"])]
    fact = [enc(t["l_okey"]), enc(t["l_price"], 2), enc(t["l_disc"], 2), enc(t["l_ship"])]
    D_, M_, F_, spec = q3_args(t, dim, mid, fact)
    force = join == "hash"
    for tab in (t, t2):
        if tab is t2:  # the new contents into the same buffers
            for old, new in ((dim[0], enc(t2["c_key"], fb=20)), (mid[1], enc(t2["o_cust"], fb=20))):
                assert old.words.numel() == new.words.numel() and old.nsegs == new.nsegs
                old.words.copy_(new.words)
                old.dsegs.copy_(new.dsegs)
                ctypes.memmove(old.hsegs, new.hsegs, ctypes.sizeof(old.hsegs))
            torch.cuda.synchronize()
        top, groups, stats = Q3.run(tab)
        for _ in range(2):  # the first call after the change, and one reusing its ranges
            rows, g, st = D.star_agg(ctx, D_, M_, F_, spec, limit=10, want_groups=True, force_hash=force)
            assert rows == top
            assert (st.dim_pass, st.mid_pass, st.fact_pass) == (stats["dim_pass"], stats["mid_pass"],
                                                                 stats["fact_pass"])
            assert np.array_equal(host(g), groups)


@pytest.mark.parametrize("scale,seg_rows", [(0.02, 4096), (0.1, 65536)])
def test_star_q3_batch(ctx, scale, seg_rows):
    """q3 with different substitution parameters (segment, date) answered by one pass of each
    table: every query equals its own oracle run and its own single-query star_agg."""
    from alenka_amd import device as D

    ndim, norders = int(150000 * scale), int(1500000 * scale)
    t = Q3.tables(4321, ndim, norders)
    dim, mid, fact = encode_q3(ctx, t, seg_rows)
    params = [("BUILDING", 19950315), ("MACHINERY", 19950301), ("AUTOMOBILE", 19950331),
              ("BUILDING", 19920201), ("HOUSEHOLD", 19980801)]
    qs = []
    for seg_name, date in params:
        code = int(t["code_of"][Q3.SEGMENTS.index(seg_name)])
        qs.append((dict(cols=dim, ranges=[(1, code, code)]), dict(cols=mid, ranges=[(2, -(1 << 63), date - 1)]),
                   dict(cols=fact, ranges=[(3, date + 1, (1 << 63) - 1)]),
                   dict(d_key=0, m_key=0, m_fk=1, m_g1=2, m_g2=3, f_fk=0, f_x=1, f_y=2, a0=0, a1=1, b0=100, b1=-1)))
    got = D.star_agg_batch(ctx, qs, limit=10)
    for (seg_name, date), q, (rows, st) in zip(params, qs, got):
        top, groups, stats = Q3.run(t, segment=seg_name, date=date)
        assert rows == top, (seg_name, date)
        assert st.dim_pass == stats["dim_pass"] and st.mid_pass == stats["mid_pass"]
        assert st.fact_pass == stats["fact_pass"]
        alone, _, st1 = D.star_agg(ctx, *q, limit=10)
        assert alone == rows
        assert (st1.mid_probe, st1.fact_probe) == (st.mid_probe, st.fact_probe)


@pytest.mark.parametrize("force_hash", [False, True])
def test_star_duplicate_keys_rejected(ctx, force_hash):
    """A build side with a repeated key is not a star join: the fused pipeline refuses it
    (ALN_E_UNSUPPORTED) so the caller falls back to the unfused operators."""
    from alenka_amd import device as D

    t = Q3.tables(55, 3000, 30000)
    o_key = t["o_key"].copy()
    passing = np.nonzero(t["o_date"] < Q3.DATE)[0]
    o_key[passing[1]] = o_key[passing[0]]  # two passing orders share a key
    t2 = dict(t, o_key=o_key)
    dim, mid, fact = encode_q3(ctx, t2, 4096)
    D_, M_, F_, spec = q3_args(t2, dim, mid, fact)
    # every dimension row passes, so both orders reach the mid bitmap
    D_ = dict(cols=dim, ranges=[])
    with pytest.raises(L.AlnError) as e:
        D.star_agg(ctx, D_, M_, F_, spec, limit=10, force_hash=force_hash)
    assert e.value.code == L.ALN_E_UNSUPPORTED


# ---- the benchmark's segment layout: 1,000,000-row segments ------------------------------
@pytest.mark.parametrize("join", ["bitmap", "hash"])
def test_star_q3_million_row_segments(ctx, join):
    """q3 at the 6M-row base size (dimension 150k, orders 1.5M, fact ~6M rows) in the
    benchmark's 1,000,000-row segments: six fact segments, each 244 full 4096-row tiles and
    a 576-row tail tile, and the resolve grid built from that shape; groups, pass counts and
    top-10 against the oracle, then three runs of a prepared query as the benchmark loop
    makes them."""
    from alenka_amd import device as D

    t = Q3.tables(2024, 150000, 1500000)
    top, groups, stats = Q3.run(t)
    assert len(t["l_okey"]) > 5_000_000 and stats["fact_pass"] > 10_000
    dim, mid, fact = encode_q3(ctx, t, 1_000_000)
    assert fact[0].nsegs == 6 and all(fact[0].hsegs[s].nrows % 4096 == 576 for s in range(5))
    D_, M_, F_, spec = q3_args(t, dim, mid, fact)
    rows, g, st = D.star_agg(ctx, D_, M_, F_, spec, limit=10, want_groups=True, force_hash=join == "hash")
    assert rows == top
    assert (st.dim_pass, st.mid_pass, st.fact_pass, st.groups) == (
        stats["dim_pass"], stats["mid_pass"], stats["fact_pass"], stats["groups"])
    assert np.array_equal(host(g), groups)
    if join == "bitmap":
        q = D.StarQuery(ctx, D_, M_, F_, spec, limit=10)
        for _ in range(3):
            r2, _, st2 = q.run()
            assert r2 == top and (st2.mid_pass, st2.fact_pass) == (stats["mid_pass"], stats["fact_pass"])


@pytest.mark.parametrize("name,ops", [PREDICATES[0], PREDICATES[1], PREDICATES[2], PREDICATES[6]])
@pytest.mark.parametrize("zone_maps", [False, True])
def test_scan_filter_million_row_segments(ctx, name, ops, zone_maps):
    """aln_scan_filter over 3.5 segments of 1,000,000 rows (the benchmark's segment size):
    exact row ids against the oracle's compaction, with and without zone-map skipping."""
    from alenka_amd import device as D

    n, seg_rows = 3_500_000, 1_000_000
    cols = O.gen_flat(12, n)
    cols[1] = np.sort(cols[1])  # date sorted, so zone maps give A / N / R segments
    dec = [0, 0, 2, 2]
    dcols = [D.Column.encode(ctx, dev(ctx, c), seg_rows, decimals=d) for c, d in zip(cols, dec)]
    assert dcols[0].nsegs == 4
    prog, _ = L.compile_rpn(ops, dec)
    modes = None
    if zone_maps:
        modes = [L.zone_map_check(ops, [c.hsegs[s].vmin for c in dcols], [c.hsegs[s].vmax for c in dcols], dec)
                 for s in range(4)]
    got = host(D.scan_filter(ctx, dcols, prog, modes)).astype(np.uint32)
    parts = []
    for s in range(4):
        lo, hi = s * seg_rows, min(n, (s + 1) * seg_rows)
        m = "R" if modes is None else modes[s]
        if m == "A":
            parts.append(np.arange(lo, hi, dtype=np.uint32))
        elif m == "R":
            parts.append(O.compact(O.filter_mask(ops, [c[lo:hi] for c in cols], dec), lo))
    want = np.concatenate(parts)
    assert np.array_equal(got, want)
    if modes is None:  # the whole-table mask gives the same ids
        assert np.array_equal(got, O.compact(O.filter_mask(ops, cols, dec)))
