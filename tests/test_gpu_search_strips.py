"""The search's matrix-core form against the column passes (the same particles
scored in one call of many units, which takes the strips, and one particle at a
time, under 2,048 units, which takes the passes) at boxes whose last ky tile, kz
step and table region differ, to FP32 summation order; and against the FP64 oracle."""
import numpy as np
import pytest

from emclarity_amd import synthetic as S
from emclarity_amd.batched import BatchAligner
from emclarity_amd.device import Context
from emclarity_amd.geometry import eulerSearch
from emclarity_amd.workload import local_matrix, random_rotation
from oracle import emc_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,radius,peak_radius,table", [
    (8, 3.0, 4, "c64"), (16, 7.4, 6, "c64"), (31, 14.9, 6, "f16"), (33, 16.4, 4, "c64"), (40, 15.2, 6, "c64"),
    (64, 14.9, 6, "f16"), (96, 16.4, 6, "f16"),
])
def test_strips_match_passes(ctx, n, radius, peak_radius, table):
    rng = np.random.default_rng(n)
    ax = np.arange(n) - n // 2
    z, y, x = np.meshgrid(ax, ax, ax, indexing="ij")
    ref = np.exp(-((x - 0.1 * n) ** 2 + y ** 2 + 2 * z ** 2) / (2 * (0.12 * n) ** 2))
    ref += 0.6 * np.exp(-((x + 0.2 * n) ** 2 + (y - 0.1 * n) ** 2 + z ** 2) / (2 * (0.05 * n) ** 2))
    grid = eulerSearch("C1", 15, 5, 15, 5)
    parts = [(np.roll(ref, tuple(rng.integers(-2, 3, 3)), (0, 1, 2)) + 0.2 * rng.standard_normal((n, n, n)))
             .astype(np.float32) for _ in range(-(-2048 // len(grid)) + 1)]
    _compare(n, radius, peak_radius, table, rng, grid, ref, parts)


@pytest.mark.parametrize("n,radius,peak_radius,table", [(9, 4.4, 4, "c64"), (31, 15.4, 6, "c64"), (41, 20.4, 4, "f16")])
def test_odd_boxes_keep_their_last_x_plane(ctx, n, radius, peak_radius, table):
    """An odd box has a plane kx = (n - 1) / 2 inside supports past it (white volumes)."""
    rng = np.random.default_rng(n)
    ref = rng.standard_normal((n, n, n))
    grid = eulerSearch("C1", 15, 5, 15, 5)
    parts = [rng.standard_normal((n, n, n)).astype(np.float32) for _ in range(-(-2048 // len(grid)))]
    _compare(n, radius, peak_radius, table, rng, grid, ref, parts)


def _compare(n, radius, peak_radius, table, rng, grid, ref, parts):
    P = len(parts)
    starts = [random_rotation(rng) for _ in range(P)]
    al = BatchAligner(n, ref.astype(np.float32), np.ones((n, n, n), np.float32), support_radius=radius,
                      peak_radius=peak_radius, table=table)
    assert P * len(grid) >= 2048
    al.set_particles(parts, [None] * P, starts)
    score, shift = al.search(grid)
    one = BatchAligner(n, ref.astype(np.float32), np.ones((n, n, n), np.float32), support_radius=radius,
                       peak_radius=peak_radius, table=table)
    for i in range(P):
        one.set_particles(parts[i:i + 1], [None], starts[i:i + 1])
        s1, d1 = one.search(grid)
        assert np.max(np.abs(score[i] - s1[0])) < 1e-5 * np.max(np.abs(s1))
        # the peak's parabola; a tie of two voxels may fall to either
        assert np.mean(np.max(np.abs(shift[i] - d1[0]), axis=1) < 1e-3) > 0.99


def test_radii_that_print_alike_are_kept_apart(ctx):
    """radius^2 = 3.9999998 and 4.0 print the same and differ by the frequencies at |k| = 2."""
    rng = np.random.default_rng(1)
    n, P, grid = 8, 147, eulerSearch("C1", 15, 10, 15, 10)[:14]
    vol = rng.standard_normal((n, n, n)).astype(np.float32)
    part = rng.standard_normal((n, n, n)).astype(np.float32)
    starts = [random_rotation(rng) for _ in range(P)]
    score = []
    for before in (None, float(np.sqrt(3.9999998))):
        own = Context(0)
        al = BatchAligner(n, vol, np.ones((n, n, n), np.float32), support_radius=2.0, peak_radius=4, ctx=own)
        al.set_particles([part] * P, [None] * P, starts)
        if before:
            al.search(grid, before)
        score.append(al.search(grid, 2.0)[0])
    assert score[0].size >= 2048
    np.testing.assert_array_equal(score[0], score[1])


@pytest.mark.parametrize("table", ["c64", "f16"])
def test_strips_match_the_oracle(ctx, table):
    """One particle from 128 start orientations over 16 grid points: 2,048 units, every
    85th against the full-grid FP64 restatement, to the bounds of the passes' test."""
    n, P = 32, 128
    bp = O.bandpass3d((n, n, n), 1e-3, 40.0, 8.0, 2.5)
    truth = (40.0, 30.0, 20.0)
    c = S.make_align_case(11, n=n, euler=truth, snr=1.0, n_blobs=16, blob_radius=0.22 * n)
    rng = np.random.default_rng(2)
    starts = [np.eye(3) if i % 2 else local_matrix(*rng.uniform(-20, 20, 3)) for i in range(P)]
    al = BatchAligner(n, c.ref, bp.astype(np.float32), peak_radius=6, table=table)
    al.set_particles([c.particle] * P, [None] * P, starts)
    pts = np.array([truth] + [tuple(rng.uniform(0, 180, 3)) for _ in range(15)])
    score, shift = al.search(pts)
    assert score.size >= 2048
    F2 = O.batch_reference_spectrum(c.ref, table)
    bpp = O.batch_prepare(c.particle, bp, np.ones((n, n, n), np.float32), al.support)
    for unit in range(0, P * len(pts), 85):
        i, k = divmod(unit, len(pts))
        sc, sh = O.batch_score_map(F2, n, bpp, starts[i] @ local_matrix(*pts[k]), 6)
        assert abs(score[i, k] - sc) < 1e-4 * abs(sc), (i, k, score[i, k], sc)
        assert np.max(np.abs(shift[i, k] - sh)) < 2e-3, (i, k, shift[i, k], sh)
