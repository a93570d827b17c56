"""The dipolar FFT convolution at transform lengths that are no power of two, against the oracle's
field: every radix (2 to 13) on every axis, lengths of one point, odd row counts (the last row pair
has one row), partly filled column tiles, narrow tiles of long lines and wide ones of many columns,
unpadded periodic lengths, two basis atoms and lattices of one plane.  Tolerance 1e-12 of the largest gradient: the transforms' rounding, eps log2(n) with the
sums over a lattice, stays below 1e-14."""
import numpy as np
import pytest

from test_gpu_parity import engine  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu

CASES = [
    # cells, boundary conditions, padding, basis atoms
    ([45, 50, 4], "000", 1, 1),    # 90 x 100 x 8: radices 9 and 10
    ([13, 11, 7], "000", 1, 1),    # 26 x 22 x 14: radices 13 and 11
    ([21, 33, 15], "000", 1, 1),   # 42 x 66 x 30
    ([3, 2, 3], "000", 1, 1),      # single-stage lengths 6 x 4 x 6
    ([1, 9, 5], "000", 1, 1),      # one point along a
    ([9, 1, 5], "000", 1, 1),      # one point along b, one row a pair
    ([121, 5, 3], "000", 1, 1),    # 242 = 11 11 2, odd row count
    ([5, 169, 2], "000", 1, 1),    # 338 = 13 13 2
    ([7, 6, 150], "000", 1, 1),    # 300 along c: three stages, narrow column tile
    ([4, 250, 3], "000", 1, 1),    # 500 along b
    ([250, 3, 2], "000", 1, 1),    # 500 along a
    ([27, 35, 12], "110", 0, 1),   # periodic without padding: odd lengths 27 x 35, images
    ([6, 10, 5], "000", 1, 2),     # two basis atoms: complex spectrum
    ([11, 13, 3], "100", 1, 2),
    ([20, 500, 1], "000", 1, 1),   # one plane: 1000 points along b
    ([50, 45, 1], "110", 1, 1),
    ([32, 64, 1], "000", 1, 1),    # one plane, powers of two
    ([22, 26, 1], "110", 0, 2),
    ([1, 7, 1], "000", 1, 1),
    ([7, 1, 1], "000", 1, 1),
    # tiles that more than a block's threads could serve: few columns or row pairs a tile
    ([200, 520, 4], "000", 1, 1),  # 1040 along b
    ([128, 560, 8], "000", 1, 1),  # 1120 along b
    ([6, 864, 2], "000", 1, 1),    # 1728 along b
    ([6, 1008, 2], "000", 1, 1),   # 2016 along b
    ([864, 16, 35], "000", 1, 1),  # 1728 along a, 840 row pairs
    ([1008, 16, 35], "000", 1, 1), # 2016 along a
    # the tiles of films: 16 columns of 300 points, 8 of 400, 4 row pairs
    ([64, 150, 32], "000", 1, 1),
    ([100, 200, 20], "000", 1, 1),
    # lines of the kernel spectrum's set-up longer than one pass over a block's threads
    ([4, 3, 264], "000", 1, 1),    # 528 along c
    ([3, 4, 512], "000", 1, 1),    # 1024 along c
    ([3, 2, 700], "000", 1, 1),    # 1400 along c
    ([3, 2, 300], "000", 1, 2),    # 600 along c, two basis atoms
    ([2, 3, 735], "000", 1, 2),    # 1470 along c, two atoms: the twiddles do not fit behind the tile
    ([2, 3, 210], "000", 1, 8),    # 420 along c, eight atoms
    ([1500, 4, 2], "000", 1, 1),   # 3000 along a
    ([3, 1430, 2], "000", 1, 1),   # 2860 along b
    ([3, 2000, 1], "000", 1, 1),   # 4000 along b, one plane
    ([2048, 3, 2], "000", 1, 1),   # 4096 along a
]


@pytest.mark.parametrize("cells,bc,padding,basis", CASES)
def test_ddi_field_of_any_length(engine, oracle, cells, bc, padding, basis):  # noqa: F811
    print("CASE ddi lengths", cells, bc, padding, basis, flush=True)
    cfg = dict(bravais_lattice="sc", n_basis_cells=cells, boundary_conditions=[int(c) for c in bc],
               mu_s=[2.0 - 0.5 * k / max(1, basis - 1) for k in range(basis)], ddi_method="fft", ddi_n_periodic_images=[2, 1, 0], ddi_pb_zero_padding=padding)
    if basis > 1:
        cfg["basis"] = [[0, 0, 0], [0.5, 0.4, 0.3], [0.5, 0, 0], [0, 0.5, 0], [0, 0, 0.6], [0.3, 0.7, 0.8], [0.7, 0.2, 0.1],
                        [0.9, 0.8, 0.4]][:basis]
    e = engine(cfg)
    S = oracle.System(cfg)
    s = oracle.random_spins(S.nos, 77)
    e.set_spins(s)
    g, E = e.gradient()
    g0, E0 = S.gradient_and_energy(s)
    assert np.abs(g - g0).max() <= 1e-12 * np.abs(g0).max()
    assert abs(E - E0) <= 1e-11 * max(abs(E0), np.abs(g0).max())


@pytest.mark.parametrize("passes", ["one kernel", "generic"])
@pytest.mark.parametrize("cells,basis", [([20, 500, 1], 1), ([22, 26, 1], 2), ([10, 128, 1], 4), ([9, 25, 1], 8)])
def test_ddi_field_of_one_plane_both_ways(engine, oracle, monkeypatch, cells, basis, passes):  # noqa: F811
    """One kernel along b, and the passes B, C and B^-1 that it takes the place of (plans of several
    atoms time the two)."""
    if passes == "generic":
        monkeypatch.setenv("SPIRIT_HIP_DDI_PASS_C", "generic")
    test_ddi_field_of_any_length(engine, oracle, cells, "000", 1, basis)
