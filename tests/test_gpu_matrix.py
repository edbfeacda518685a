"""GPU: the 753-bit matrix passes against the vector kernels, bit for bit, at
every schedule they have (three and four passes, 2^15 to 2^22), forward and
inverse, in place, with operands at the ends of the field, alone and (from
2^15) in a batch."""
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
