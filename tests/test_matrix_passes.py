"""The 753-bit matrix passes (gpusnarks_amd/csrc/matrix753_kernels.h) restated
in Python, CPU only: their arithmetic with whole numbers at the ends of its
ranges, and their digits, twiddle factors and addresses over a small prime
field against the O(n^2) DFT, and the addresses of every schedule in use."""
import random

import numpy as np
import pytest

import gpusnarks_amd as g

FIELDS = [g.FIELD_MNT4753_FR, g.FIELD_MNT6753_FR]
TOP = 1 << 768
OFFSET = int("80" * 96, 16)
BIAS, BIAS_ROW0 = (1 << 22) - (1 << 14), 1 << 14
LIFT = 12400


def digits(x):
    """The signed byte digits of x from its offset form."""
    return [b - 128 for b in ((x + OFFSET) % TOP).to_bytes(96, "little")]


def columns(w, p):
    cols = []
    for k in range(96):
        c = (w << (8 * k)) % p
        # the kernel centres by the top limb alone
        cols.append(c - p if (c >> 736) > (p >> 736) // 2 else c)
    return cols


def product(y, w, p):
    """mat753_mul: column sums from BIAS, four to a limb, one carry chain."""
    cols, dy = columns(w, p), digits(y)
    m = np.array([digits(c) for c in cols], dtype=np.int64).T
    sums = m @ np.array(dy, dtype=np.int64) + BIAS
    assert sums.min() >= 0 and sums.max() < 1 << 23
    t = carry = prev = 0
    for l in range(24):
        n0, n1 = int(sums[4 * l] + (sums[4 * l + 1] << 8)), int(sums[4 * l + 2] + (sums[4 * l + 3] << 8))
        assert n0 < 1 << 31 and n1 < 1 << 31
        n0 += BIAS_ROW0 if l == 0 else 0
        v = n0 + (((n1 << 16) | (prev >> 16)) & 0xFFFFFFFF) + carry
        t |= (v & 0xFFFFFFFF) << (32 * l)
        carry, prev = v >> 32, n1
    return t - TOP if t >> 767 else t


def reduced(x, p):
    """Mat753::reduce: the quotient from the top limb in single precision."""
    top = np.float32((p >> 736) + ((p >> 704) & 0xFFFFFFFF) / 2.0 ** 32)
    xt = (((x + OFFSET) % TOP) >> 736) - 0x80808080
    q = int(np.rint(np.float32(xt) * np.float32(1.0 / float(top))))
    return x - q * p


@pytest.mark.parametrize("field", FIELDS)
def test_products_and_bounds(field):
    p = g.MODULI[field]
    bound = 6144 * p
    limit = 2 * bound + 6 * p
    # the digits' range, the lift and the top limb cover every value
    assert -OFFSET <= -limit and limit <= (TOP - 1) - OFFSET
    assert LIFT * p > limit and LIFT * p + limit < TOP
    rng = random.Random(field)
    ws = [0, 1, p - 1, p // 2, p // 2 + 1] + [rng.randrange(p) for _ in range(6)]
    ys = [0, 1, -1, limit, -limit, 2 * bound, -2 * bound] + [rng.randrange(-limit, limit) for _ in range(6)]
    # digits all at one end against the signs of the columns' own extremes
    for w in ws:
        cols = columns(w, p)
        assert all(abs(c) <= p // 2 + (p >> 15) for c in cols)
        for y in ys + [sum((-128 if c > 0 else 127) << (8 * k) for k, c in enumerate(cols[:95]))]:
            t = product(y, w, p)
            assert (t - y * w) % p == 0 and abs(t) <= bound + (96 * 128 * p >> 15)
    for x in ys + [k * p // 2 + d for k in range(-24000, 24000, 997) for d in (-1, 0, 1)]:
        if abs(x) <= limit:
            assert abs(reduced(x, p)) <= 0.52 * p


# ------------------------------------------------------------ the passes

P, G = 3 * 2 ** 30 + 1, 5


def column_dft(col, r, log_g, kap, table):
    """Steps of one column: in-place decimation in time over positions, the
    twiddle of step s from entry ((2^s - 1) << log_g) + (kap << s) + kk."""
    R = 1 << r
    v = [col[int(format(i, "0%db" % r)[::-1], 2)] for i in range(R)]
    for s in range(r):
        for i in range(R):
            if not i & (1 << s):
                kk = i & ((1 << s) - 1)
                t = v[i | (1 << s)] * table[((1 << s) - 1 << log_g) + (kap << s) + kk] % P
                v[i], v[i | (1 << s)] = (v[i] + t) % P, (v[i] - t) % P
    return v


def fold_table(w, n, r, log_g):
    out = []
    for i in range(((1 << r) - 1) << log_g):
        s = ((i >> log_g) + 1).bit_length() - 1
        rest = i - (((1 << s) - 1) << log_g)
        gi, kk = rest >> s, rest & ((1 << s) - 1)
        out.append(pow(w, (gi + (kk << log_g)) * (n >> (log_g + s + 1)), P))
    return out


@pytest.mark.parametrize("radices", [(2, 2, 2), (1, 3, 2), (3, 2, 3), (2, 1, 2, 2), (2, 2, 1, 3), (1, 2, 3, 1)])
def test_passes_match_dft(radices):
    log_n, num = sum(radices), len(radices)
    n = 1 << log_n
    w = pow(G, (P - 1) >> log_n, P)
    rng = random.Random(log_n * num)
    a = [rng.randrange(P) for _ in range(n)]
    want = [sum(x * pow(w, j * k, P) for j, x in enumerate(a)) % P for k in range(n)]
    buf, rp, n1 = list(a), radices[-1], radices[0]
    out = [None] * n
    log_ns = 0
    for i, r in enumerate(radices):
        R, log_g = 1 << r, radices[i - 1] if i else 0
        fold = fold_table(w, n, r, log_g)
        if i < num - 1:
            log_s = log_n - log_ns - r
            for blk in range(n >> r):  # one column at a time
                log_hi = log_n - r - log_s - log_g
                p, lo = blk >> log_s, blk & ((1 << log_s) - 1)
                kap = p >> log_hi if i else 0
                pre = ((p & ((1 << log_hi) - 1)) << log_g) | kap if i else 0
                base = (pre << (log_s + r)) + lo
                col = [buf[base + (row << log_s)] for row in range(R)]
                if i and i == num - 3:  # the pair (1, 3), on both halves of step 0
                    e = kap * (lo >> rp) << rp
                    col = [x * pow(w, e, P) % P for x in col]
                v = column_dft(col, r, log_g, kap, fold)
                if i:  # the column factor of jP
                    e = (lo & ((1 << rp) - 1)) * kap << (log_ns - log_g)
                    v = [x * pow(w, e, P) % P for x in v]
                for row in range(R):
                    buf[base + (row << log_s)] = v[row]
        else:
            for blk in range(n >> r):
                rev, k1 = blk >> n1, blk & ((1 << n1) - 1)
                log_k = log_n - n1 - r - log_g
                kap = rev >> log_k
                mid = ((rev & ((1 << log_k) - 1)) << log_g) | kap if log_k else rev
                at = k1 * (n >> n1) + (mid << r)
                v = column_dft(buf[at:at + R], r, log_g, kap, fold)
                for row in range(R):
                    assert out[(row << (log_n - r)) + (rev << n1) + k1] is None
                    out[(row << (log_n - r)) + (rev << n1) + k1] = v[row]
        log_ns += r
    assert out == want


@pytest.mark.parametrize("field", FIELDS)
def test_dense_sums_and_bounds(field):
    """dense753.hip: column sums of up to 32 terms from 2^18 255, 25 limbs, the
    quotient from the top two in single precision, four such parts plus 3 p."""
    p = g.MODULI[field]
    bias, row0 = 255 << 18, 1 << 18
    top = np.float32((p >> 736) + ((p >> 704) & 0xFFFFFFFF) / 2.0 ** 32)
    inv = np.float32(1.0 / float(top))
    assert 32 * 96 * 2 ** 14 < bias and 2 * p < OFFSET and -2 * p > -OFFSET
    rng = random.Random(field + 100)
    for case in range(8):
        parts, exact = [], 0
        for _ in range(4):
            sums, want = np.full(96, bias, dtype=np.int64), 0
            for _ in range(32):
                w = rng.choice([0, 1, p - 1, p // 2, p // 2 + 1, rng.randrange(p)])
                cols = columns(w, p)
                y = rng.choice([0, 4 * p, -2 * p, 2 * p - 1, rng.randrange(-2 * p, 4 * p)])
                if case < 2:  # every digit at the end that makes its column largest
                    y = sum((-128 if (c > 0) != (case == 1) else 127) << (8 * k) for k, c in enumerate(cols[:95]))
                sums += np.array([digits(c) for c in cols], dtype=np.int64).T @ np.array(digits(y), dtype=np.int64)
                want += y * w
            assert sums.min() >= 0 and sums.max() < 1 << 31
            total = sum(int(s) << (8 * r) for r, s in enumerate(sums)) + row0
            low, high = total % TOP, (total >> 768) - row0
            f = np.float32(np.float32(high) * np.float32(2.0 ** 32) + np.float32(low >> 736)) * inv
            q = int(np.rint(f))
            part = high * TOP + low - q * p
            assert abs(part) <= 0.51 * p and (part - want) % p == 0
            parts.append(part)
            exact += want
        y = sum(parts) + 3 * p
        assert 0 < y < TOP and (y - exact) % p == 0


SCHEDULES = {15: (5, 5, 5), 16: (5, 6, 5), 17: (6, 5, 6), 18: (6, 6, 6), 19: (5, 5, 4, 5), 20: (5, 5, 5, 5),
             21: (6, 5, 5, 5), 22: (6, 5, 5, 6), 23: (6, 6, 5, 6), 24: (6, 6, 6, 6)}


@pytest.mark.parametrize("log_n", sorted(SCHEDULES))
def test_addresses_and_entries_of_every_schedule(log_n):
    """MatTile's addresses of every tile, row and column: each pass reads and
    writes every element once, the ones between the first and the last where
    they read, with matrix entries inside the tables built for the pass and
    32-bit arithmetic where the kernel has it."""
    radices = SCHEDULES[log_n]
    n, num, rp, n1 = 1 << log_n, len(radices), radices[-1], radices[0]
    assert sum(radices) == log_n
    W, u32 = 32, 1 << 32

    def covers(at):
        assert at.min() >= 0 and at.max() < n and at.size == n
        seen = np.zeros(n, dtype=bool)
        seen[at.reshape(-1)] = True
        return seen.all()

    log_ns = 0
    for i, r in enumerate(radices):
        R, log_g, log_s = 1 << r, radices[i - 1] if i else 0, log_n - log_ns - r
        blk = np.arange(n >> (r + 5), dtype=np.int64)
        row, col = np.arange(R)[None, :, None], np.arange(W)[None, None, :]
        if i == 0:
            kap = np.zeros_like(blk)
            at = (blk * W)[:, None, None] + row * (n >> r) + col
            assert covers(at)
        elif i < num - 1:
            log_hi = log_n - r - log_s - log_g
            assert log_hi >= 0 and log_s >= rp >= 5
            p, lo = blk >> (log_s - 5), (blk << 5) & ((1 << log_s) - 1)
            assert (blk << 5).max() < u32
            kap = p >> log_hi
            pre = ((p & ((1 << log_hi) - 1)) << log_g) | kap
            top, nxt = lo & ((1 << rp) - 1), lo >> rp
            at = ((pre << (log_s + r)) + lo)[:, None, None] + (row << log_s) + col
            assert covers(at)
            # column factors: entry (kap << rp) + top + column of 2^(g + rp)
            assert ((kap << rp) + top + W - 1).max() < 1 << (log_g + rp)
            if i == num - 3:  # the pair (1, 3): 2 entries of 2^(g + r3)
                assert log_s - rp == radices[2]
                assert (2 * ((kap << (log_s - rp)) + nxt) + 1).max() < 2 << (log_g + radices[2])
            else:
                assert num == 3 or i == 2
        else:
            rev, k1 = blk >> (n1 - 5), (blk << 5) & ((1 << n1) - 1)
            log_k = log_n - n1 - r - log_g
            kap = rev >> log_k
            mid = ((rev & ((1 << log_k) - 1)) << log_g) | kap if log_k else rev
            assert covers((k1 * (n >> n1) + (mid << r))[:, None, None] + row + col * (n >> n1))
            assert covers(((rev << n1) + k1)[:, None, None] + row * (n >> r) + col)
        # step s takes entry ((2^s - 1) << g) + (kap << s) + kk, kk < 2^s
        s = r - 1
        assert kap.min() >= 0 and kap.max() < 1 << log_g
        assert (((1 << s) - 1) << log_g) + (kap.max() << s) + (1 << s) - 1 < ((1 << r) - 1) << log_g
        log_ns += r


@pytest.mark.parametrize("field", FIELDS)
def test_columns_in_runs_of_eight(field):
    """write_matrices: twelve lanes with eight columns each, the first one
    256^(8 t) w mod p and every next one 256 times the one before it, which
    canon takes below 2^761."""
    p = g.MODULI[field]
    rng = random.Random(field + 200)
    for w in [0, 1, p - 1, p // 2] + [rng.randrange(p) for _ in range(4)]:
        got = []
        for t in range(12):
            c = (w << (64 * t)) % p
            for k in range(8):
                got.append(c - p if (c >> 736) > (p >> 736) // 2 else c)
                assert c << 8 < 1 << 761
                c = (c << 8) % p
        assert got == columns(w, p)


VALUE_MAX, LIFTED_MAX = 18434, 12290  # in units of p
DIGITS_MAX = int("7f" * 96, 16)


def magnitudes(kind, r, start):
    """Largest value met in a pass of 2^r rows whose inputs are below `start`,
    and what it leaves, in units of p."""
    B = 6144 * (1 + 2.0 ** -15)
    v = seen = start
    for s in range(r):
        if kind == "first" and s < 2:  # sums, and at step 1 products by w_4
            v = 2 * v if s == 0 else max(2 * v, v + B)
        elif kind == "mid2" and s == 0:  # both halves are products
            v = 2 * B
        else:
            reduced = {"first": s % 2 == 1, "mid": s % 2 == 0, "mid2": s % 2 == 0}.get(kind, s % 2 == 1)
            v = (0.51 if reduced else v) + B
        seen = max(seen, v)
    return seen, v


def test_values_of_every_schedule_stay_in_range():
    """The bounds that the passes are built on, followed through every schedule
    and every pair of column passes; 3 B is reached in MAT_MID2 and COL_LAST."""
    B = 6144 * (1 + 2.0 ** -15)
    most = {}
    for radices in SCHEDULES.values():
        num, v = len(radices), 1.0
        for i, r in enumerate(radices):
            kind = "first" if i == 0 else "last" if i == num - 1 else "mid2" if i == num - 3 else "mid"
            seen, left = magnitudes(kind, r, v)
            most[kind] = max(most.get(kind, 0), seen)
            v = left if kind in ("first", "last") else B  # a column factor ends the passes between
        assert v <= LIFTED_MAX
    for log_n in range(8, 13):
        r1, r2 = (log_n + 1) // 2, log_n // 2
        seen, v = magnitudes("first", r1, 1.0)
        assert seen <= 2 * B + 6
        seen, v = magnitudes("col_last", r2, v)
        most["col_last"] = max(most.get("col_last", 0), seen)
        assert v <= LIFTED_MAX
    assert most["first"] <= 2 * B + 6 and most["mid"] <= 2 * B + 6 and most["last"] <= 2 * B + 6
    assert 3 * B <= most["mid2"] <= VALUE_MAX and 3 * B <= most["col_last"] <= VALUE_MAX


@pytest.mark.parametrize("field", FIELDS)
def test_products_and_reductions_at_the_largest_values(field):
    p = g.MODULI[field]
    limit = VALUE_MAX * p
    assert DIGITS_MAX == (TOP - 1) - OFFSET and limit <= DIGITS_MAX
    assert sum(d << (8 * k) for k, d in enumerate(digits(limit))) == limit
    assert sum(d << (8 * k) for k, d in enumerate(digits(-limit))) == -limit
    assert LIFT > LIFTED_MAX and (LIFT + LIFTED_MAX) * p < TOP
    rng = random.Random(field + 300)
    for y in [limit, -limit, limit - 1, 3 * 6144 * p, -3 * 6144 * p] + [rng.randrange(limit // 2, limit) for _ in range(4)]:
        assert abs(reduced(y, p)) <= 0.52 * p and (reduced(y, p) - y) % p == 0
        for w in (1, p - 1, p // 2, p // 2 + 1, rng.randrange(p)):
            t = product(y, w, p)
            assert (t - y * w) % p == 0 and abs(t) <= 6144 * p + (96 * 128 * p >> 15)


@pytest.mark.parametrize("field", FIELDS)
def test_canon_covers_every_768_bit_value(field):
    """F753::canon: the quotient estimate in double precision is the quotient
    or one less, up to the lifted values of the last passes and to 2^768."""
    p = g.MODULI[field]
    two32 = 4294967296.0
    limb = lambda v, i: float((v >> (32 * i)) & 0xFFFFFFFF)
    top = lambda v: (limb(v, 23) * two32 + limb(v, 22)) * two32 + limb(v, 21)
    factor = (1.0 - 2.0 ** -40) / top(p)
    rng = random.Random(field + 400)
    xs = [TOP - 1, TOP - 2, (LIFT + LIFTED_MAX) * p, 1 << 767, (1 << 767) - 1]
    for _ in range(4000):
        k = rng.randrange(1, TOP // p + 1)
        xs += [k * p - 1, k * p, k * p + 1]
    for k in list(range(1, 40)) + list(range(TOP // p - 40, TOP // p + 1)):
        xs += [k * p - 1, k * p, k * p + 1]
    for x in xs:
        q = int(top(x) * factor)
        assert x // p - 1 <= q <= x // p, x
