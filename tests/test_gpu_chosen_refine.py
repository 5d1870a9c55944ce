"""One capped layer in the chosen form on random states of square, wide and
tall two-site matrices, flat and steeply decaying spectra (columns below the
FP32 floor), caps next to the full rank and well below it, against the FP64
layer.  The FP32 vectors mix kept and discarded directions by at most some
1e-5: states within 1e-10 infidelity, spectra within 1e-6; values below the
floor (2e-5 |X|, 4e-10 of the weight each) count as zeros, so weights agree
within 1e-8; Newton-Schulz leaves the vectors orthonormal to 1e-12."""
import numpy as np
import pytest

from qaintensor import DeviceMPS, FORM_CHOSEN, circuits as C

pytestmark = pytest.mark.gpu


def state(ctx, n, dims, fall, seed, cap):
    rng = np.random.default_rng(seed)
    sites = []
    for j in range(n):
        t = rng.standard_normal((dims[j], 2, dims[j + 1])) + \
            1j * rng.standard_normal((dims[j], 2, dims[j + 1]))
        sites.append(np.asfortranarray(
            t * np.exp(-fall * np.arange(dims[j + 1]) / dims[j + 1])))
    dev = DeviceMPS(n, cap, ctx)
    dev.set_sites(sites)
    return dev


@pytest.mark.parametrize("dims,cap", [
    # (chi_{i-1}, chi_i, chi_{i+1}) of the gate's bond: square, wide
    # (M < N), tall (M > N), rank one above the cap, 64-column solve
    ((64, 100, 64), 100), ((40, 70, 64), 70), ((64, 70, 40), 70),
    ((50, 99, 50), 99), ((30, 40, 30), 40), ((128, 160, 128), 160)])
@pytest.mark.parametrize("fall", [0.0, 12.0])
def test_refined_layer_matches_fp64(gpu_ctx, dims, cap, fall):
    a, m, b = dims
    n, i = 14, 7
    chis = [min(2 ** j, 2 ** (n - j)) for j in range(n + 1)]
    chis[i - 1], chis[i], chis[i + 1] = a, m, b
    for j in range(i - 2, -1, -1):
        chis[j] = min(chis[j], 2 ** j, 2 * chis[j + 1])
    for j in range(i + 2, n + 1):
        chis[j] = min(chis[j], 2 ** (n - j))
    cap_state = max(max(chis), cap)
    ref = state(gpu_ctx, n, chis, fall, 3, cap_state)
    dev = DeviceMPS(n, cap_state, gpu_ctx)
    dev.copy_from(ref)
    g = C.haar_unitary(np.random.default_rng(a + m), 4)
    k0, d0 = ref.apply_layer([i], [g], 1e-8, cap)
    k1, d1 = dev.apply_layer([i], [g], 1e-8, cap, FORM_CHOSEN)
    assert k0[0] == k1[0]
    assert abs(d0[0] - d1[0]) <= 1e-8
    f = abs(ref.overlap(dev)) ** 2 / (ref.norm2() * dev.norm2())
    assert 1.0 - f <= 1e-10
    assert np.abs(ref.bond_spectrum(i) - dev.bond_spectrum(i)).max() <= 1e-6
    B = dev.site(i + 1)
    v = B.reshape((B.shape[0], -1), order="F")
    assert np.abs(v @ v.conj().T - np.eye(B.shape[0])).max() <= 1e-12
