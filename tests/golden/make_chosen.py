"""Writes tests/golden/chosen_form.npz: what the chosen form gives for the
circuits of tests/test_gpu_chosen_pinned.py, from the library itself on an
MI355X.  The fixture pins the FP32 sweeps' rounding, so it is only written
again when the chosen form is meant to give other results.  Run from the
repo root:
    python tests/golden/make_chosen.py OUT.npz
"""
import os
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(
    os.path.abspath(__file__))))
sys.path.insert(0, os.path.join(ROOT, "qaintensor.jl_amd"))

from qaintensor import (DeviceMPS, FORM_CHOSEN, circuits as C,  # noqa: E402
                        default_context)

# (qubits, depth, cap, a layer per call, gates): an FP32 solve of one block
# pair, two block pairs, three launches a round, the LDS-resident round, one
# gate at a time, and a weakly entangled circuit whose gates alternate
# between FP32 and FP64
CASES = [(12, 10, 16, True, "haar"), (14, 10, 48, True, "haar"),
         (16, 10, 100, True, "haar"), (18, 11, 170, True, "haar"),
         (13, 9, 30, False, "haar"), (16, 24, 40, True, "weak")]


def run(ctx, n, depth, chi, batched, gates, form=FORM_CHOSEN):
    make = C.weak_brickwall_layers if gates == "weak" else C.brickwall_layers
    dev = DeviceMPS(n, chi, ctx)
    rec = []
    dev.run_layers(make(n, depth, 7 * n + chi), 1e-8, chi, form=form,
                   batched=batched, record=rec)
    out = {"amplitudes": dev.amplitudes(C.random_bitstrings(n, 64, chi)),
           "z": dev.expect_z(),
           "spectra": np.concatenate([dev.bond_spectrum(b)
                                      for b in range(1, n)]),
           "kept": np.array([k for _, k, _ in rec]),
           "weight": 1.0 - np.array([d for _, _, d in rec])}
    dev.free()
    return out


def main():
    ctx = default_context()
    out = {}
    for i, case in enumerate(CASES):
        for k, v in run(ctx, *case).items():
            out["%d_%s" % (i, k)] = v
    np.savez_compressed(sys.argv[1], **out)


if __name__ == "__main__":
    main()
