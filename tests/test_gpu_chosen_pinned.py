"""The chosen form gives the amplitudes, <Z>, spectra, ranks and weights it
always gave.  Its FP32 sweeps put 1e-6 to 1e-4 into the amplitudes, and a
last bit changed in any gate before one draws that error anew, so a kernel
that rounds differently shows up here at 1e-6 and more; the bound is that of
64-bit results, 1e-9 of the norm."""
import os
import sys

import numpy as np
import pytest

from qaintensor import FORM_PLAIN

GOLD = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
sys.path.insert(0, GOLD)

import make_chosen as M  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("i", range(len(M.CASES)))
def test_chosen_results_are_kept(gpu_ctx, i):
    want = np.load(os.path.join(GOLD, "chosen_form.npz"), allow_pickle=False)
    got = M.run(gpu_ctx, *M.CASES[i])
    plain = M.run(gpu_ctx, *M.CASES[i], form=FORM_PLAIN)
    assert np.array_equal(got["kept"], want["%d_kept" % i])
    for k in ("amplitudes", "z", "spectra", "weight"):
        w = want["%d_%s" % (i, k)]
        assert got[k].shape == w.shape
        assert np.linalg.norm(got[k] - w) <= 1e-9 * np.linalg.norm(w), k
    # the case does reach the FP32 sweeps
    a = plain["amplitudes"]
    assert np.linalg.norm(got["amplitudes"] - a) > 1e-8 * np.linalg.norm(a)
