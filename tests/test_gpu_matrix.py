"""GPU: the 753-bit matrix passes against the vector kernels, bit for bit, at
every schedule they have (three and four passes, 2^15 to 2^24), forward and
inverse, in place, with operands at the ends of the field, alone and (from
2^15) in a batch; which calls take them."""
import os
import sys

import numpy as np
import pytest

import gpusnarks_amd as g
from gpusnarks_amd import synth

pytestmark = pytest.mark.gpu


def operands(field, log_n, seed):
    n, p = 1 << log_n, g.MODULI[field]
    x = synth.uniform_residues(seed, min(n, 1 << 15), p, 24)
    x = np.concatenate([x] * (n // len(x)))
    ends = np.array([[(v >> (32 * k)) & 0xFFFFFFFF for k in range(24)] for v in (p - 1, 0, 1, p // 2)], np.uint32)
    x[:n // 4] = ends[np.random.RandomState(seed).randint(0, 4, n // 4)]
    x[n // 2:n // 2 + n // 8] = ends[0]
    return x


def run(plan, x, in_place):
    d_in = g.DeviceArray.from_numpy(x)
    d_out = d_in if in_place else g.DeviceArray(x.nbytes)
    plan.execute(d_in.ptr, d_out.ptr, 0)
    g.synchronize()
    return d_out.download(x.shape)


@pytest.mark.parametrize("field,log_n", [(g.FIELD_MNT4753_FR, 15)] +
                         [(g.FIELD_MNT6753_FR, l) for l in (15, 16, 17, 18, 19, 20, 21, 22)])
def test_matrix_passes_match_vector_kernels(field, log_n):
    x = operands(field, log_n, 0x3A7 + log_n)
    vector = [(7, 0, 1)] * (log_n // 7) + ([(log_n % 7, 2, 1)] if log_n % 7 else [])
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")
    for inverse in (False, True):
        print("matrix passes", field, log_n, inverse, flush=True)
        sys.stdout.flush()
        plan = g.Plan(field, log_n, inverse=inverse)
        got = run(plan, x, in_place=inverse)
        d_in, d_out = g.DeviceArray.from_numpy(x), g.DeviceArray(2 * x.nbytes)
        batch = g.Batch([(field, log_n, inverse, d_in.ptr, d_out.ptr),
                         (field, log_n, inverse, d_in.ptr, d_out.ptr + x.nbytes)])
        batch.launch()
        g.synchronize()
        both = d_out.download((2,) + x.shape)
        batch.close()
        plan.close()
        try:
            g.tuning_set(field, log_n, vector)
            plan = g.Plan(field, log_n, inverse=inverse)
            assert plan.num_passes == len(vector)
            want = run(plan, x, in_place=False)
            plan.close()
        finally:
            g.tuning_clear()
            g.tuning_load(shipped)  # the default routes again
        assert np.array_equal(got, want), (field, log_n, inverse)
        assert np.array_equal(both[0], want) and np.array_equal(both[1], want), (field, log_n, inverse)


@pytest.mark.parametrize("field,log_n", [(f, l) for f in (g.FIELD_MNT4753_FR, g.FIELD_MNT6753_FR)
                                         for l in (10, 11, 12, 13, 14, 15)])
def test_dense_passes_match_vector_kernels(field, log_n):
    """Every schedule of the dense passes (2^10 to 2^15 alone), out of place
    and in place, two executions of one plan back to back."""
    x = operands(field, log_n, 0xDE5 + log_n)
    vector = [(7, 0, 1)] * (log_n // 7) + ([(log_n % 7, 2, 1)] if log_n % 7 else [])
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")
    for inverse in (False, True):
        print("dense passes", field, log_n, inverse, flush=True)
        plan = g.Plan(field, log_n, inverse=inverse)
        got, again = run(plan, x, in_place=False), run(plan, x[::-1].copy(), in_place=True)
        plan.close()
        try:
            g.tuning_set(field, log_n, vector)
            plan = g.Plan(field, log_n, inverse=inverse)
            assert plan.num_passes == len(vector)
            want, want_again = run(plan, x, in_place=False), run(plan, x[::-1].copy(), in_place=False)
            plan.close()
        finally:
            g.tuning_clear()
            g.tuning_load(shipped)  # the default routes again
        assert np.array_equal(got, want) and np.array_equal(again, want_again), (field, log_n, inverse)


# launches of a batch: two passes on the vector kernels; on the matrix cores
# three passes, each with a launch per radix
@pytest.mark.parametrize("sizes,launches", [((16,), 2), ((17,), 2), ((16, 16), 2), ((15, 16), 2), ((15, 15, 16), 2),
                                            ((16, 17), 2), ((15, 16, 17), 2), ((16, 16, 17), 2),
                                            ((15, 15, 16, 16, 16, 17), 2), ((15,), 3), ((15, 15, 15, 15), 3),
                                            ((16, 16, 16), 3), ((17, 17), 3), ((18,), 3), ((15, 16, 16), 4),
                                            ((15, 15, 16, 16, 17, 17), 6), ((16, 17, 18), 6)])
def test_small_batches_take_the_faster_kernels(sizes, launches):
    """Batches on both sides of the line between vector kernels and matrix
    passes, every transform bit-identical to its plan alone."""
    field = g.FIELD_MNT6753_FR
    print("small batch", sizes, flush=True)
    xs = [operands(field, l, 0xBA7 + 31 * i + l) for i, l in enumerate(sizes)]
    d_in = [g.DeviceArray.from_numpy(x) for x in xs]
    d_out = [g.DeviceArray(x.nbytes) for x in xs]
    batch = g.Batch([(field, l, i % 2 == 1, a.ptr, b.ptr) for i, (l, a, b) in enumerate(zip(sizes, d_in, d_out))])
    assert batch.num_launches == launches
    batch.launch()
    g.synchronize()
    for i, (l, x, d) in enumerate(zip(sizes, xs, d_out)):
        plan = g.Plan(field, l, inverse=i % 2 == 1)
        assert np.array_equal(d.download(x.shape), run(plan, x, in_place=False)), (sizes, i)
        plan.close()
    batch.close()


def test_schedules_go_back_to_the_library():
    """A schedule that is read, replaced and put back leaves the size on the
    library's own choice, and so does a table that repeats the shipped lines
    beside others; a schedule of the program's own stands."""
    field = g.FIELD_MNT6753_FR
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")

    def passes(f, log_n):
        plan = g.Plan(f, log_n)
        try:
            return plan.num_passes
        finally:
            plan.close()

    try:
        g.tuning_clear()
        g.tuning_load(shipped)
        vector = [(9, 1, 1), (9, 1, 1)]
        own = {(field, 18): 3, (field, 20): 4, (g.FIELD_MNT4753_FR, 13): 3}
        for (f, l), p in own.items():
            assert passes(f, l) == p
        # the program's own schedule, even the vector kernels' shipped one
        g.tuning_set(field, 18, vector)
        assert passes(field, 18) == 2
        g.tuning_clear()
        g.tuning_load(shipped)
        for (f, l), p in own.items():
            before = g.tuning_get(f, l)
            g.tuning_set(f, l, before)
            assert passes(f, l) == p and g.tuning_get(f, l) == before
            g.tuning_set(f, l, [(7, 0, 1)] * (l // 7) + [(l % 7, 2, 1)])
            assert passes(f, l) == l // 7 + 1
            g.tuning_set(f, l, before)
            assert passes(f, l) == p and g.tuning_get(f, l) == before
    finally:
        g.tuning_clear()
        g.tuning_load(shipped)


def test_tables_that_repeat_shipped_lines(tmp_path):
    field = g.FIELD_MNT6753_FR
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")
    lines = open(shipped).read().splitlines()
    copy, mine = tmp_path / "copy.txt", tmp_path / "mine.txt"
    copy.write_text("\n".join("0 20 10,4,4 10,4,4" if l.startswith("0 20 ") else l for l in lines) + "\n")
    mine.write_text("2 18 9,0,1 9,0,1\nbatch 2 15 8,0,1 7,0,1\n")
    x = g.DeviceArray(96 << 18)

    def passes():
        plan, batch = g.Plan(field, 18), g.Batch([(field, 15, False, x.ptr, x.ptr)])
        out = plan.num_passes, batch.num_launches
        plan.close()
        batch.close()
        return out

    try:
        g.tuning_clear()
        g.tuning_load(shipped)
        assert passes() == (3, 3)
        g.tuning_load(str(copy))
        assert g.tuning_get(g.FIELD_FP32, 20) == [(10, 4, 4), (10, 4, 4)]
        assert passes() == (3, 3) and g.tuning_get(field, 18) == [(9, 1, 1), (9, 1, 1)]
        g.tuning_load(str(mine))
        assert passes() == (2, 2)
        g.tuning_load(str(copy))  # the shipped lines again
        assert passes() == (3, 3)
    finally:
        g.tuning_clear()
        g.tuning_load(shipped)


def test_autotuner_leaves_faster_choices_to_the_library(tmp_path):
    """At MNT6 2^10 no schedule of the vector kernels is near the matrix cores:
    the tuner writes no line, and its table keeps the library's choice."""
    from gpusnarks_amd import autotune as at
    field = g.FIELD_MNT6753_FR
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")
    table = tmp_path / "t.txt"
    try:
        results = at.tune(["mnt6"], [10], budget_s=2.0, log=lambda *a: print(*a, flush=True))
        sched, ms, ms_default = results[(field, 10)]
        assert sched is None and ms == ms_default
        at.write_table(results, str(table), keep_from=shipped)
        assert not any(l.startswith("2 10 ") for l in table.read_text().splitlines())
        g.tuning_clear()
        g.tuning_load(shipped)
        g.tuning_load(str(table))
        for l, p in ((10, 2), (15, 3), (18, 3), (20, 4)):
            plan = g.Plan(field, l)
            assert plan.num_passes == p
            plan.close()
    finally:
        g.tuning_clear()
        g.tuning_load(shipped)


@pytest.mark.parametrize("log_n", [23, 24])
def test_largest_matrix_passes_match_vector_kernels(log_n):
    """The two largest schedules, in place, and out of place in a batch."""
    field = g.FIELD_MNT6753_FR
    x = operands(field, log_n, 0x3A7 + log_n)
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")
    for inverse in (False, True):
        print("largest matrix passes", log_n, inverse, flush=True)
        plan = g.Plan(field, log_n, inverse=inverse)
        assert plan.num_passes == 4
        got = run(plan, x, in_place=True)
        plan.close()
        d_in, d_out = g.DeviceArray.from_numpy(x), g.DeviceArray(x.nbytes)
        batch = g.Batch([(field, log_n, inverse, d_in.ptr, d_out.ptr)])
        batch.launch()
        g.synchronize()
        assert np.array_equal(d_out.download(x.shape), got), (log_n, inverse)
        batch.close()
        print("vector kernels", log_n, inverse, flush=True)
        try:
            g.tuning_set(field, log_n, [(5, 2, 1)] * 4 + [(log_n - 20, 2, 1)])
            plan = g.Plan(field, log_n, inverse=inverse)
            assert plan.num_passes == 5
            want = run(plan, x, in_place=False)
            plan.close()
        finally:
            g.tuning_clear()
            g.tuning_load(shipped)  # the default routes again
        assert np.array_equal(got, want), (log_n, inverse)
        del got, want


def test_table_lines_on_the_vector_kernels():
    """Every 753-bit line of the shipped table, of transforms alone and in
    batches, set explicitly: the vector kernels run it, bit-identical to the
    library's own choice (elsewhere against the oracle)."""
    shipped = os.path.join(os.path.dirname(g.library_path), "tuning.txt")
    lines = []
    for line in open(shipped):
        tok = [t for t in line.split("#", 1)[0].split() if t != "batch"]
        if tok and int(tok[0]) != g.FIELD_FP32:
            lines.append((int(tok[0]), int(tok[1]), [tuple(map(int, t.split(","))) for t in tok[2:]]))
    assert len(lines) >= 25
    for field, log_n, sched in sorted(lines):
        print("vector schedule", field, log_n, sched, flush=True)
        x = operands(field, log_n, 0x7AB + log_n)
        want = {}
        try:
            g.tuning_clear()
            g.tuning_load(shipped)
            for inverse in (False, True):
                plan = g.Plan(field, log_n, inverse=inverse)
                want[inverse] = run(plan, x, in_place=False)
                plan.close()
            g.tuning_set(field, log_n, sched)
            for inverse in (False, True):
                plan = g.Plan(field, log_n, inverse=inverse)
                assert plan.num_passes == len(sched)
                assert np.array_equal(run(plan, x, in_place=False), want[inverse]), (field, log_n, sched, inverse)
                plan.close()
        finally:
            g.tuning_clear()
            g.tuning_load(shipped)
