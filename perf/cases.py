"""Work that users of this library have it do, as cases to time.

Each case goes through the public entry points: plans on device tensors, a
batch, domain helpers between transforms, the inner product and the
host-buffer call.  Operands are uniform residues (a uniform residue is also
a uniform Montgomery form), as little-endian 32-bit limbs in int32 tensors of
shape (n, limbs).
"""
import numpy as np
import torch

import gpusnarks_amd as g

FIELDS = {"fp32": g.FIELD_FP32, "mnt4": g.FIELD_MNT4753_FR, "mnt6": g.FIELD_MNT6753_FR}
TWO_ADICITY = {"fp32": 30, "mnt4": 15, "mnt6": 30}
# the smallest quadratic non-residue: the base of the standard roots of unity
NON_RESIDUE = {"fp32": 5, "mnt4": 13, "mnt6": 11}
VECTOR_OPS = ("inner_product", "pointwise_mul", "to_montgomery", "coset_shift", "vec_sub")
# 32x32 -> 64 bit multiply-adds of one 24-limb Montgomery product, and the
# multiplies of one 32-bit one; each counts as two operations
MADS = {"fp32": 3, "mnt4": 2 * 24 * 24 + 24, "mnt6": 2 * 24 * 24 + 24}


def listed():
    return [
        # the smallest transforms of a proof's sub-circuits: latency and launches
        {"name": "mnt4_2e10", "kind": "plan", "field": "mnt4", "log_n": 10, "inverse": False},
        # the largest plain domain of the reference's field, interpolation
        {"name": "mnt4_2e15_inverse", "kind": "plan", "field": "mnt4", "log_n": 15, "inverse": True},
        # the size that the reference quotes, over the field that has the root
        {"name": "mnt6_2e18", "kind": "plan", "field": "mnt6", "log_n": 18, "inverse": False},
        # a large circuit's interpolation
        {"name": "mnt6_2e20_inverse", "kind": "plan", "field": "mnt6", "log_n": 20, "inverse": True},
        # 32-bit field: an ordinary trace column, and the size bound by memory
        {"name": "fp32_2e16_inverse", "kind": "plan", "field": "fp32", "log_n": 16, "inverse": True},
        {"name": "fp32_2e26", "kind": "plan", "field": "fp32", "log_n": 26, "inverse": False},
        # many provers' transforms of mixed fields, sizes and directions at once
        {"name": "batch_ragged_64", "kind": "batch", "count": 64, "mix": 1, "low": 10, "high": 18},
        # the reference's own size over its own field, one past the 2-adicity
        {"name": "mnt4_2e16_extended", "kind": "extended", "field": "mnt4", "log_n": 16, "inverse": False},
        # a domain far past the 2-adicity: odd factors of p - 1
        {"name": "mnt4_525x2e12", "kind": "mixed", "field": "mnt4", "odd": 525, "log_n": 12, "inverse": False},
        # the quotient polynomial of a proof: (A B - C) / Z through a coset
        {"name": "quotient_mnt6_2e16", "kind": "quotient", "field": "mnt6", "log_n": 16},
        # the reference's multiexp over field elements, a ragged length
        {"name": "inner_product_262143", "kind": "vector", "field": "mnt4", "op": "inner_product", "n": 262143},
        # best_fft on a host vector, copies included
        {"name": "host_mnt6_2e14", "kind": "host", "field": "mnt6", "log_n": 14, "inverse": False},
    ]


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "plan32", "batch", "extended", "mixed", "quotient", "vector", "host"])
    inverse = rng.random() < 0.5
    if kind == "plan":
        field = rng.choice(["mnt4", "mnt6", "mnt6"])
        return {"kind": "plan", "field": field, "log_n": rng.randint(10, 15 if field == "mnt4" else 20),
                "inverse": inverse}
    if kind == "plan32":
        return {"kind": "plan", "field": "fp32", "log_n": rng.randint(10, 26), "inverse": inverse}
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(9, 64), "mix": rng.randint(1, 10 ** 6), "low": 10,
                "high": rng.randint(12, 18)}
    if kind == "extended":
        return {"kind": "extended", "field": "mnt4", "log_n": rng.randint(10, 16), "inverse": inverse}
    if kind == "mixed":
        return {"kind": "mixed", "field": "mnt4", "odd": rng.choice([3, 5, 7, 15, 21, 35, 75, 105, 175, 525]),
                "log_n": rng.randint(6, 12), "inverse": inverse}
    if kind == "quotient":
        return {"kind": "quotient", "field": "mnt6", "log_n": rng.randint(10, 16)}
    if kind == "vector":
        op = rng.choice(VECTOR_OPS)
        n = int(2 ** rng.uniform(10, 19)) | 1
        return {"kind": "vector", "field": rng.choice(["fp32", "mnt4", "mnt6"]), "op": op,
                "n": 1 << (n.bit_length() - 1) if op == "coset_shift" else n}
    field = rng.choice(["fp32", "mnt4", "mnt6"])
    return {"kind": "host", "field": field, "log_n": rng.randint(10, 20 if field == "fp32" else 15),
            "inverse": inverse}


# ------------------------------------------------------------------ inputs

def _residues(field, n, seed):
    """n uniform residues: random limbs with the top one below the modulus'."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if field == "fp32":
        v = torch.randint(0, g.MODULI[g.FIELD_FP32], (n, 1), generator=gen, device="cuda", dtype=torch.int64)
        return (v - ((v >> 31) << 32)).to(torch.int32)
    x = torch.randint(-2 ** 31, 2 ** 31, (n, 24), generator=gen, device="cuda", dtype=torch.int64).to(torch.int32)
    x[:, 23] = torch.randint(0, g.MODULI[FIELDS[field]] >> (32 * 23), (n,), generator=gen, device="cuda",
                             dtype=torch.int64).to(torch.int32)
    return x


def _constant(field, value):
    """The Montgomery form of an integer as limbs on the host."""
    f = FIELDS[field]
    limbs = g.NLIMBS[f]
    v = value * (1 << (32 * limbs)) % g.MODULI[f]
    return np.array([(v >> (32 * i)) & 0xFFFFFFFF for i in range(limbs)], dtype=np.uint32)


def _batch_items(case):
    """(field, log_n, inverse) of each transform: 3 of 4 over the 753-bit field."""
    rng = np.random.RandomState(case["mix"])
    return [("mnt6" if rng.rand() < 0.75 else "fp32", int(rng.randint(case["low"], case["high"] + 1)),
             bool(rng.rand() < 0.5)) for _ in range(case["count"])]


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind in ("plan", "extended", "mixed"):
        field, f = case["field"], FIELDS[case["field"]]
        if kind == "plan":
            st["plan"] = g.Plan(f, case["log_n"], inverse=case["inverse"])
        elif kind == "extended":
            st["plan"] = g.Plan.extended(f, case["log_n"], inverse=case["inverse"])
        else:
            st["plan"] = g.Plan.mixed(f, case["odd"] << case["log_n"], inverse=case["inverse"])
        st["x"] = _residues(field, st["plan"].n, seed)
        st["out"] = torch.empty_like(st["x"])
    elif kind == "batch":
        items = _batch_items(case)
        totals = {fd: sum(1 << l for fi, l, _ in items if fi == fd) for fd in ("mnt6", "fp32")}
        st["x"] = {fd: _residues(fd, max(t, 1), seed + i) for i, (fd, t) in enumerate(totals.items())}
        st["out"] = {fd: torch.zeros_like(x) for fd, x in st["x"].items()}
        at = dict.fromkeys(totals, 0)
        rows = []
        for fd, log_n, inverse in items:
            off = at[fd] * g.ELEMENT_BYTES[FIELDS[fd]]
            rows.append((FIELDS[fd], log_n, inverse, st["x"][fd].data_ptr() + off, st["out"][fd].data_ptr() + off))
            at[fd] += 1 << log_n
        st["batch"] = g.Batch(rows)
    elif kind == "quotient":
        field, f, n = case["field"], FIELDS[case["field"]], 1 << case["log_n"]
        st["forward"] = g.Plan(f, case["log_n"])
        st["inverse"] = g.Plan(f, case["log_n"], inverse=True)
        st["abc"] = [_residues(field, n, 3 * seed + i) for i in range(3)]
        st["tmp"] = [torch.empty_like(v) for v in st["abc"]]
        q = NON_RESIDUE[field]
        st["shift"] = _constant(field, q)
        st["z_inv"] = _constant(field, pow(pow(q, n, g.MODULI[f]) - 1, -1, g.MODULI[f]))
    elif kind == "vector":
        st["a"] = _residues(case["field"], case["n"], 2 * seed)
        st["b"] = _residues(case["field"], case["n"], 2 * seed + 1)
        st["out"] = torch.empty_like(st["a"][:1] if case["op"] == "inner_product" else st["a"])
        st["shift"] = _constant(case["field"], NON_RESIDUE[case["field"]])
    else:
        st["x"] = _residues(case["field"], 1 << case["log_n"], seed).cpu().numpy().view(np.uint32)
    return st


# -------------------------------------------------------------------- runs

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("plan", "extended", "mixed"):
        return st["plan"].execute_tensor(st["x"], st["out"])
    f = FIELDS.get(case.get("field"))
    if kind == "host":
        return g.best_fft(st["x"], None, f, inverse=case["inverse"])
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "batch":
        st["batch"].launch(stream)
        return st["out"]
    if kind == "vector":
        out, a, b, n, op = st["out"], st["a"].data_ptr(), st["b"].data_ptr(), case["n"], case["op"]
        if op == "to_montgomery":
            g.to_montgomery(f, out.data_ptr(), a, n, stream)
        elif op == "coset_shift":
            g.coset_shift(f, out.data_ptr(), a, n, st["shift"], False, stream)
        else:
            getattr(g, op)(f, out.data_ptr(), a, b, n, stream)
        return out
    # quotient: values of A, B, C on H -> coefficients -> values on the coset
    # -> (A B - C) / Z there -> coefficients
    n = 1 << case["log_n"]
    a, b, c = st["tmp"]
    for v, t in zip(st["abc"], st["tmp"]):
        st["inverse"].execute_tensor(v, t)
        g.coset_shift(f, t.data_ptr(), t.data_ptr(), n, st["shift"], False, stream)
        st["forward"].execute_tensor(t)
    g.pointwise_mul(f, a.data_ptr(), a.data_ptr(), b.data_ptr(), n, stream)
    g.vec_sub(f, a.data_ptr(), a.data_ptr(), c.data_ptr(), n, stream)
    g.scale(f, a.data_ptr(), a.data_ptr(), n, st["z_inv"], stream)
    st["inverse"].execute_tensor(a)
    g.coset_shift(f, a.data_ptr(), a.data_ptr(), n, st["shift"], True, stream)
    return a


# ---------------------------------------------------------- what they need

def work(case):
    kind = case["kind"]
    if kind == "batch":
        parts = [work({"kind": "plan", "field": fd, "log_n": l}) for fd, l, _ in _batch_items(case)]
        return {k: sum(p[k] for p in parts) for k in ("bytes", "flops")}
    field = case["field"]
    eb, op = g.ELEMENT_BYTES[FIELDS[field]], 2 * MADS[field]
    if kind == "vector":
        inputs = 1 if case["op"] in ("to_montgomery", "coset_shift") else 2
        outputs = 1 if case["op"] == "inner_product" else case["n"]
        return {"bytes": (inputs * case["n"] + outputs) * eb, "flops": op * case["n"] if case["op"] != "vec_sub" else 0}
    n = (case["odd"] if kind == "mixed" else 1) << case["log_n"]
    butterflies = n / 2 * np.log2(n)
    if kind == "quotient":  # three inputs, one output, 7 transforms, 4 shifts, a product and a scaling
        return {"bytes": 4.0 * n * eb, "flops": float(op * (7 * butterflies + 6 * n))}
    return {"bytes": 2.0 * n * eb, "flops": float(op * butterflies)}


# ----------------------------------------------------------- exact outputs

def _ints(x):
    """The values of an (n, limbs) array as Python integers."""
    raw = np.ascontiguousarray(x.cpu().numpy() if torch.is_tensor(x) else x).view(np.uint32)
    size = 4 * raw.shape[1]
    data = raw.tobytes()
    return [int.from_bytes(data[i:i + size], "little") for i in range(0, len(data), size)]


def _limbs(v, field):
    size = 4 * g.NLIMBS[FIELDS[field]]
    return np.frombuffer(b"".join(e.to_bytes(size, "little") for e in v), dtype=np.int32).reshape(len(v), -1)


def _root(field, log_n, inverse):
    p = g.MODULI[FIELDS[field]]
    w = pow(NON_RESIDUE[field], (p - 1) >> log_n, p)
    return pow(w, -1, p) if inverse else w


def _transform(v, field, inverse):
    """X_k = sum_j v_j w^(j k), n^-1 for the inverse; radix-2 self-sorting."""
    p, n = g.MODULI[FIELDS[field]], len(v)
    log_n = n.bit_length() - 1
    w = _root(field, log_n, inverse)
    scale = pow(n, -1, p) if inverse else 1
    if field == "fp32":  # the same steps on arrays: every product fits 64 bits
        a, q = np.array(v, dtype=np.uint64), np.uint64(p)
        powers = np.ones(1, dtype=np.uint64)
        for i in range(log_n - 1):  # w^0 .. w^(n/2 - 1) by doubling
            powers = np.concatenate([powers, powers * np.uint64(pow(w, 1 << i, p)) % q])
        for s in range(log_n):
            lo, hi = a[:n // 2].reshape(-1, 1 << s), a[n // 2:].reshape(-1, 1 << s)
            t = powers[::1 << s][:, None]
            a = np.stack([(lo + hi) % q, (lo + q - hi) % q * t % q], axis=1).reshape(-1)
        return [int(e) for e in a * np.uint64(scale) % q]
    powers = [1] * (n // 2)
    for i in range(1, n // 2):
        powers[i] = powers[i - 1] * w % p
    for s in range(log_n):
        m, nxt = 1 << s, [0] * n
        for b in range(n // 2 >> s):
            t = powers[b << s]
            for k in range(m):
                x, y = v[b * m + k], v[b * m + k + n // 2]
                nxt[2 * b * m + k] = (x + y) % p
                nxt[(2 * b + 1) * m + k] = (x - y) * t % p
        v = nxt
    return [e * scale % p for e in v]


def exact(case, seed):
    kind, field = case["kind"], case.get("field")
    if kind in ("batch", "mixed") or (field != "fp32" and case.get("log_n", 0) > 17):
        return None  # minutes of whole-number arithmetic
    if field == "fp32" and (case.get("log_n", 0) > 22):
        return None
    p = g.MODULI[FIELDS[field]]
    r_inv = pow(1 << (32 * g.NLIMBS[FIELDS[field]]), -1, p)
    if kind == "plan" or kind == "host":
        v = _transform(_ints(_residues(field, 1 << case["log_n"], seed)), field, case["inverse"])
        return _limbs(v, field).view(np.uint32 if kind == "host" else np.int32)
    if kind == "vector":
        n, op = case["n"], case["op"]
        a, b = _ints(_residues(field, n, 2 * seed)), _ints(_residues(field, n, 2 * seed + 1))
        if op == "inner_product":
            return _limbs([sum(x * y for x, y in zip(a, b)) * r_inv % p], field)
        if op == "pointwise_mul":
            return _limbs([x * y * r_inv % p for x, y in zip(a, b)], field)
        if op == "vec_sub":
            return _limbs([(x - y) % p for x, y in zip(a, b)], field)
        if op == "to_montgomery":
            return _limbs([(x << (32 * g.NLIMBS[FIELDS[field]])) % p for x in a], field)
        return _limbs(_coset(a, field, False), field)
    if kind == "extended":
        m, q = 1 << (case["log_n"] - 1), NON_RESIDUE[field]
        v = _ints(_residues(field, 2 * m, seed))
        G = pow(q, m, p)
        if not case["inverse"]:
            shifted = _coset([(x + G * y) % p for x, y in zip(v[:m], v[m:])], field, False)
            return _limbs(_transform([(x + y) % p for x, y in zip(v[:m], v[m:])], field, False) +
                          _transform(shifted, field, False), field)
        u, s = _transform(v[:m], field, True), _coset(_transform(v[m:], field, True), field, True)
        k = pow(1 - G, -1, p)
        high = [(x - y) * k % p for x, y in zip(u, s)]
        return _limbs([(x - y) % p for x, y in zip(u, high)] + high, field)
    n = 1 << case["log_n"]
    values = []
    for i in range(3):
        v = _transform(_ints(_residues(field, n, 3 * seed + i)), field, True)
        values.append(_transform(_coset(v, field, False), field, False))
    z_inv = pow(pow(NON_RESIDUE[field], n, p) - 1, -1, p)
    v = [(x * y * r_inv - z) * z_inv % p for x, y, z in zip(*values)]
    return _limbs(_coset(_transform(v, field, True), field, True), field)


def _coset(v, field, inverse):
    p = g.MODULI[FIELDS[field]]
    step = pow(NON_RESIDUE[field], -1, p) if inverse else NON_RESIDUE[field]
    out, e = [], 1
    for x in v:
        out.append(x * e % p)
        e = e * step % p
    return out
