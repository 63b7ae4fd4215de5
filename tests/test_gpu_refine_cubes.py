"""The refinement's evaluation by cubes and table bricks against the adjoint
entry (emc_align_eval_grad, support-list order): scores and the steps taken
from the gradients, at the smallest and largest supports, odd boxes, both
table formats, few and many particles, and poses that are not rotations
(gathered from the table instead of the staged bricks)."""
import ctypes

import numpy as np
import pytest

from emclarity_amd import _lib
from emclarity_amd.batched import BatchAligner
from emclarity_amd.device import Context, DeviceArray
from emclarity_amd.workload import random_rotation

from test_gpu_batched import _host_refine

pytestmark = pytest.mark.gpu


def _aligner(n, count, radius, table, seed):
    rng = np.random.default_rng(seed)
    ax = np.arange(n) - n // 2
    z, y, x = np.meshgrid(ax, ax, ax, indexing="ij")
    ref = np.exp(-((x - 0.1 * n) ** 2 + (y + 0.05 * n) ** 2 + 2 * z ** 2) / (2 * (0.12 * n) ** 2))
    ref += 0.5 * np.exp(-((x + 0.2 * n) ** 2 + y ** 2 + (z - 0.1 * n) ** 2) / (2 * (0.05 * n) ** 2))
    al = BatchAligner(n, ref.astype(np.float32), np.ones((n, n, n), np.float32), support_radius=radius, table=table,
                      tuning={"params": {table: {str(n): {"grad_kernel": 0}}}})
    parts = [(ref + 0.3 * rng.standard_normal((n, n, n))).astype(np.float32) for _ in range(count)]
    weights = [rng.uniform(0.2, 1.0, (n, n, n)).astype(np.float32) if i % 2 else None for i in range(count)]
    al.set_particles(parts, weights, [np.eye(3)] * count)
    R = np.stack([random_rotation(rng) for _ in range(count)])
    return al, R, rng.uniform(-2.0, 2.0, (count, 3))


def _score64(al, R, s):
    """Scores in 64 bits from the aligner's own table (c64), spectra and norms."""
    n, r = al.n, al.support
    a = np.fft.fftfreq(n) * n
    kz, kx, ky = np.meshgrid(a, np.arange(n // 2 + 1.0), a, indexing="ij")
    k2 = kx ** 2 + ky ** 2 + kz ** 2
    m = (k2 <= r * r) & (k2 > 0)
    k = np.stack([kx[m], ky[m], kz[m]], 1)
    mult = np.where(k[:, 0] > 0, 2.0, 1.0)
    T = al.F2.get().reshape(-1, 4)
    Q = al.Q.get().reshape(al.n_part, *m.shape)[:, m]
    N = al.N.get().reshape(al.n_part, *m.shape)[:, m]
    A = al.A.get()
    out = []
    for p in range(al.n_part):
        j = k @ (2.0 * R[p])
        neg = j[:, 0] < 0
        j = np.where(neg[:, None], -j, j)
        i = np.floor(j).astype(np.int64)
        w = j - i
        e = ((i[:, 2] + n) * (2 * n + 1) + i[:, 1] + n) * (n + 2) + i[:, 0]
        f = 0.0
        for c in range(4):      # texel (y + c % 2, z + c // 2) of entries x and x + 1
            t = T[e, c].astype(np.complex128) * (1 - w[:, 0]) + T[e + 1, c].astype(np.complex128) * w[:, 0]
            f = f + t * (w[:, 1] if c & 1 else 1 - w[:, 1]) * (w[:, 2] if c >> 1 else 1 - w[:, 2])
        f = np.where(neg, f.conj(), f)
        num = np.sum(mult * (Q[p].astype(np.complex128) * f.conj() * np.exp(2j * np.pi / n * (k @ s[p]))).real)
        out.append(num / np.sqrt(A[p] * np.sum(mult * np.abs(f) ** 2 * N[p].astype(np.float64))))
    return np.array(out)


def _scores(al, R, s):
    cc = al.refine_device(DeviceArray.from_numpy(np.ascontiguousarray(R.reshape(-1, 9))),
                          DeviceArray.from_numpy(s.copy()), iters=0).get()
    return cc, al._eval_local(R, s)[0]


@pytest.mark.parametrize("n,count,radius,table", [
    (8, 3, 1.2, "c64"),        # the three axes' first frequencies only (below 1 both forms divide 0 by 0)
    (12, 1, 5.4, "f16"),
    (33, 17, 15.9, "c64"),     # odd box, one particle past a workgroup's waves
    (64, 70, 14.0, "c64"),     # several runs of particles per brick
    (75, 5, 28.7, "f16"),
    (128, 2, 63.5, "c64"),     # 9,405 cubes in 2,160 bricks
    (128, 5, 63.99, "c64"),    # the most of both: 9,598 in 2,316
    (8, 5, 3.4, "f16"),        # the fewest particles whose bricks are staged, the most that are gathered
    (75, 4, 36.0, "c64"),
])
def test_steps_match_the_adjoint_entry(ctx, n, count, radius, table):
    al, R, s = _aligner(n, count, radius, table, n)
    cc, ref = _scores(al, R, s)
    # FP32 samples and sums of up to 4e5 terms in another order
    assert np.max(np.abs(cc - ref)) <= 2e-6 * max(1.0, np.max(np.abs(ref)))
    Rd, sd, cd = al.refine(R, s, iters=1)
    Rh, sh, ch = _host_refine(al, R, s, iters=1)
    # the first step moves by 0.02 rad and 0.3 px along gradients that agree to ~1e-5; a refused step leaves the start
    same = (np.max(np.abs(Rd - R), axis=(1, 2)) > 0) == (np.max(np.abs(Rh - R), axis=(1, 2)) > 0)
    assert same.mean() > 0.9
    assert np.max(np.abs(Rd - Rh)[same]) < 2e-5 and np.max(np.abs(sd - sh)[same]) < 3e-4
    al.ctx.synchronize()


@pytest.mark.parametrize("table", ["c64", "f16"])
def test_poses_that_are_not_rotations_are_gathered(ctx, table):
    al, R, s = _aligner(36, 6, 12.3, table, 4)
    R[1] *= 1.3                                   # stretched: leaves the bricks' halo
    R[2] *= 0.4
    R[3] = np.diag([1.0, 1.0, -1.0]) @ R[3]       # a reflection keeps lengths
    R[4] = R[4] @ np.array([[1.0, 0.6, 0], [0, 1, 0], [0, 0, 1]])
    cc, ref = _scores(al, R, s)
    assert np.max(np.abs(cc - ref)) <= 2e-6


@pytest.mark.parametrize("n,radius", [(32, 14.5), (64, 18.3), (75, 21.0)])
def test_score_error_is_that_of_samples_taken_one_by_one(ctx, n, radius):
    """The cubes share images and phases and the waves add up 64 lanes: against 64
    bits that may cost no more than the adjoint entry's own FP32 samples, each
    positioned by itself and summed in FP64 from the thread up. A quarter is
    allowed for the two rms over 48 particles (10 % each)."""
    al, _, s = _aligner(n, 48, radius, "c64", 5)
    rng = np.random.default_rng(n)
    R = []
    for _ in range(48):           # within a few degrees of the particles' pose: the sums have a signal
        w = 0.05 * rng.standard_normal(3)
        K = np.array([[0, -w[2], w[1]], [w[2], 0, -w[0]], [-w[1], w[0], 0]])
        t = np.linalg.norm(w)
        R.append(np.eye(3) + np.sin(t) / t * K + (1 - np.cos(t)) / t ** 2 * K @ K)
    R = np.stack(R)
    cc, ref = _scores(al, R, s)
    exact = _score64(al, R, s)
    rms = lambda v: np.sqrt(np.mean(v ** 2))  # noqa: E731
    print(f"score error: refinement {rms(cc - exact):.2e}, adjoint entry {rms(ref - exact):.2e}")
    assert rms(cc - exact) < 1.25 * rms(ref - exact)


@pytest.mark.parametrize("n,radius,table", [(8, 3.9, "c64"), (16, 7.9, "f16"), (33, 16.4, "c64"), (64, 31.9, "c64"),
                                            (75, 37.4, "f16"), (128, 63.7, "c64")])
def test_samples_at_the_tables_edge(ctx, n, radius, table):
    """Supports past (n - 1) / 2 reach the table's last plane on every axis: white
    particles whose spectra are zero but in that last shell, so that one wrong texel
    of its ~100 n samples shows."""
    al, R, s = _aligner(n, 12, radius, table, n)
    rng = np.random.default_rng(n)
    ref = rng.standard_normal((n, n, n)).astype(np.float32)
    al = BatchAligner(n, ref, np.ones((n, n, n), np.float32), support_radius=radius, table=table,
                      tuning={"params": {table: {str(n): {"grad_kernel": 0}}}})
    al.set_particles([rng.standard_normal((n, n, n)).astype(np.float32) for _ in R], [None] * len(R),
                     [np.eye(3)] * len(R))
    a = np.fft.fftfreq(n) * n
    kz, kx, ky = np.meshgrid(a, np.arange(n // 2 + 1.0), a, indexing="ij")
    shell = (kx ** 2 + ky ** 2 + kz ** 2 > ((n - 1) / 2) ** 2).ravel()
    al.Q = DeviceArray.from_numpy(np.where(shell, al.Q.get(), 0).astype(np.complex64), ctx=al.ctx)
    al.N = DeviceArray.from_numpy(np.where(shell, al.N.get(), 0).astype(np.float32), ctx=al.ctx)
    cc, ref_cc = _scores(al, R, s)
    assert np.max(np.abs(cc - ref_cc)) <= 2e-6 * max(1.0, np.max(np.abs(ref_cc)))
    Rd, sd, _ = al.refine(R, s, iters=1)
    Rh, sh, _ = _host_refine(al, R, s, iters=1)
    same = (np.max(np.abs(Rd - R), axis=(1, 2)) > 0) == (np.max(np.abs(Rh - R), axis=(1, 2)) > 0)
    assert np.max(np.abs(Rd - Rh)[same], initial=0.0) < 2e-5 and np.max(np.abs(sd - sh)[same], initial=0.0) < 3e-4


def test_supports_that_print_alike_are_kept_apart(ctx):
    """4.9999999 and 5.0 differ by the frequencies at |k| = 5, some of them in cubes
    of their own: the call with the larger may not meet the smaller's cubes."""
    cc = []
    for before in (None, 4.9999999):
        al, R, s = _aligner(16, 4, 5.0, "c64", 1)
        own = Context(0)
        al.ctx = own
        al.ctx.wait_for(ctx)
        args = lambda: (DeviceArray.from_numpy(np.ascontiguousarray(R.reshape(-1, 9)), ctx=own),  # noqa: E731
                        DeviceArray.from_numpy(s.copy(), ctx=own))
        if before:
            al.refine_device(*args(), iters=0, support_radius=before).get()
        cc.append(al.refine_device(*args(), iters=0).get())
    np.testing.assert_array_equal(cc[0], cc[1])


@pytest.mark.parametrize("table,count", [("c64", 6), ("f16", 6), ("c64", 4)])
def test_steps_from_poses_that_are_not_rotations(ctx, table, count):
    """Stretched, sheared and singular start matrices (a projection maps the table
    onto a plane): the shift's gradient sums k itself, as no inverse gives it back."""
    al, R, s = _aligner(36, count, 12.3, table, 4)
    change = [lambda A: A, lambda A: 1.3 * A, lambda A: A @ np.array([[1.0, 0.6, 0], [0, 1, 0], [0, 0, 1]]),
              lambda A: A @ np.diag([1.0, 1.0, 0.0]), lambda A: np.outer(A[:, 0], A[0]),
              lambda A: 1.0001 * A]             # the last within the bricks' halo: staged
    R = np.stack([f(A) for f, A in zip(change[-count:], R)])
    Rd, sd, cd = al.refine(R, s, iters=1)
    Rh, sh, ch = _host_refine(al, R, s, iters=1)
    assert np.max(np.abs(cd - ch)) <= 2e-6
    # as above; both forms decide alike on all but ties
    same = (np.max(np.abs(Rd - R), axis=(1, 2)) > 0) == (np.max(np.abs(Rh - R), axis=(1, 2)) > 0)
    assert same.sum() >= count - 1 and np.max(np.abs(sd - s)[-3:-1]) > 0
    assert np.max(np.abs(Rd - Rh)[same]) < 4e-5 and np.max(np.abs(sd - sh)[same]) < 3e-4


def test_runs_of_particles_within_the_scratch_bound(ctx):
    """200 particles of 128^3 over their whole support take two runs within 1 GiB of
    scratch: as many bytes as that, and the poses of the particles refined by themselves."""
    n, count = 128, 200
    al, R, s = _aligner(n, 2, 62.9, "c64", 3)
    rng = np.random.default_rng(1)
    own = Context(0)
    own.wait_for(ctx)
    al.ctx, al.n_part = own, count
    for name in ("Q", "N", "A"):
        a = getattr(al, name).get()
        setattr(al, name, DeviceArray.from_numpy(np.ascontiguousarray(np.tile(a, (count // 2,) + (1,) * (a.ndim - 1))),
                                                 ctx=own))
    R = R[np.arange(count) % 2]
    s = rng.uniform(-2.0, 2.0, (count, 3))
    dev = lambda v: DeviceArray.from_numpy(np.ascontiguousarray(v), ctx=own)  # noqa: E731
    Rd, sd = dev(R.reshape(-1, 9)), dev(s)
    own.synchronize()

    def free():
        f, total = ctypes.c_size_t(), ctypes.c_size_t()
        assert _lib.load().hipMemGetInfo(ctypes.byref(f), ctypes.byref(total)) == 0
        return f.value
    before = free()
    cc = al.refine_device(Rd, sd, iters=2).get()
    assert before - free() < 1.1 * 2 ** 30
    al.n_part = 8
    for p0 in (0, 96, 192):
        q = slice(p0, p0 + 8)
        R8, s8 = dev(R[q].reshape(-1, 9)), dev(s[q])
        c8 = al.refine_device(R8, s8, iters=2).get()   # particles repeat with period 2
        np.testing.assert_array_equal(c8, cc[q])
        np.testing.assert_array_equal(R8.get(), Rd.get()[q])
        np.testing.assert_array_equal(s8.get(), sd.get()[q])


def test_pose_updates_of_more_particles_than_cus(ctx):
    """Past 256 particles the pose update runs on fewer threads: another order of its
    FP64 fold and nothing else."""
    al, R, s = _aligner(12, 260, 5.2, "c64", 12)
    Rd, sd, cd = al.refine(R, s, iters=2)
    al.n_part = 8
    R8, s8, c8 = al.refine(R[:8], s[:8], iters=2)
    assert np.max(np.abs(Rd[:8] - R8)) < 1e-9 and np.max(np.abs(sd[:8] - s8)) < 1e-9
    assert np.max(np.abs(cd[:8] - c8)) < 1e-12
