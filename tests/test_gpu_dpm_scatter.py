"""The differentiable model's tile lists where a lattice block's particles have
left one another (its clouds reach many tiles, and each tile they reach lists
it once), and where a tile's list runs over: every particle of the box in one
tile, which more lattice blocks reach than a list has entries for.

Against the FP64 twin.  A displacement of D cells is held to D 2^-24, and a
density that is linear in it to some 2^-20 of a cell's weight: 1e-4 with room.
The gradient jumps where rounding moves a particle over a cell edge: 3/sqrt(N)
for a few of N particles scattered over the box, 1e-3 where none is near one."""
import time

import numpy as np
import pytest

from cafproject_amd import dpm
from tests.dpm_ref import Ref
from tests.helpers import rel_l2

STEPS = np.array([[0.05, 0.4, 0.04], [0.06, 0.3, 0.05]])


def _box(ng, nf, ic, steps, w, dbar, passes=2):
    import torch
    box = dpm.DPM(ng, nf, len(steps))
    box.set_amplitude(np.ones((ng, ng, ng // 2 + 1), np.float32))
    box.set_schedule(ic, steps)
    wt, dt = torch.from_numpy(w).cuda(), torch.from_numpy(dbar).cuda()
    d, g = torch.empty(nf ** 3, device="cuda"), torch.empty(ng ** 3, device="cuda")
    torch.cuda.synchronize()
    s = []
    for _ in range(passes):
        t = time.perf_counter()
        box.forward(wt.data_ptr(), d.data_ptr())
        box.adjoint(dt.data_ptr(), g.data_ptr())
        box.sync()
        s.append(time.perf_counter() - t)
    box.close()
    return d.cpu().numpy(), g.cpu().numpy(), sorted(s)[len(s) // 2]


def _scattered(ng, nf, rms):
    """White noise with a flat amplitude, and ICs of that rms displacement in cells."""
    rng = np.random.default_rng(ng + nf)
    w = rng.standard_normal(ng ** 3).astype(np.float32)
    dbar = (rng.standard_normal(nf ** 3) / nf ** 3).astype(np.float32)
    one = Ref(ng, nf, np.ones((ng, ng, ng // 2 + 1)), np.array([1.0, 1.0]), np.zeros((1, 3)))
    return w, dbar, rms / np.std(one.ics(w.astype(np.float64))[1])


def _reached(x, ng, nf, T):
    """Distinct (lattice block, tile) pairs of particles at x."""
    nt, nb = (nf + T - 1) // T, (ng + 3) // 4
    l = np.stack(np.meshgrid(*[np.arange(ng)] * 3, indexing="ij"), -1).reshape(-1, 3)[:, ::-1] // 4
    blk = (l[:, 2] * nb + l[:, 1]) * nb + l[:, 0]
    c = np.floor(x).astype(np.int64) % nf
    pairs = []
    for k in range(8):
        t = (c + [k & 1, k >> 1 & 1, k >> 2]) % nf // T
        pairs.append(np.stack([blk, (t[:, 2] * nt + t[:, 1]) * nt + t[:, 0]], 1))
    return np.unique(np.concatenate(pairs), axis=0), nb ** 3, nt ** 3


def _cap(ng, nf, T, nblk, nt3):
    """Entries per list (cube_dpm_create)."""
    per = (4.0 * (nf // ng) + 4.0) / T + 1.0
    return int(min(nblk, max(64.0, 24.0 * nblk * per ** 3 / nt3)))


@pytest.mark.gpu
@pytest.mark.parametrize("ng,nf", [(20, 80), (18, 144), (48, 144), (64, 128)])
@pytest.mark.parametrize("rms", [6.0, 24.0])
def test_scattered_blocks(ng, nf, rms):
    w, dbar, cx = _scattered(ng, nf, rms)
    ic = np.array([cx, 0.3 * cx])
    ref = Ref(ng, nf, np.ones((ng, ng, ng // 2 + 1)), ic, STEPS)
    want = ref.forward(w.astype(np.float64)).ravel()
    wantg = ref.adjoint(dbar.astype(np.float64).reshape(nf, nf, nf))
    d, g, _ = _box(ng, nf, ic, STEPS, w, dbar)
    ed, eg = rel_l2(d, want), rel_l2(g, wantg)
    print(f"ng {ng} nf {nf} rms {rms}: delta {ed:.2e} gradient {eg:.2e}")
    assert ed < 1e-4
    assert eg < 3 / np.sqrt(ng ** 3)


def _collapse(ng, nf, T):
    """Noise whose displacements (ic = 1) take the particles to within r cells
    of one point: sawtooths along the axes.  Two lattice planes of each axis go
    elsewhere, which moves the others by 0.3 of a cell (displacements have no
    mean) off the mesh."""
    r = nf // ng
    at = T * (nf // T // 2) + T // 2
    l = np.arange(ng)
    saw = np.mod(at - r * l + nf / 2, nf) - nf / 2
    saw[4:6] -= 0.15 * ng
    k = 2 * np.pi * np.fft.fftfreq(ng)
    line = np.fft.ifft(-1j * k * np.fft.fft(saw / r)).real  # minus its derivative
    w = line[None, None, :] + line[None, :, None] + line[:, None, None]
    return w.astype(np.float32).ravel()


@pytest.mark.parametrize("ng,nf,T", [(32, 64, 8), (24, 144, 16)])
def test_collapsed_box_runs_a_list_over(ng, nf, T):
    x = Ref(ng, nf, np.ones((ng, ng, ng // 2 + 1)), np.array([1.0, 0.0]), STEPS).ics(
        _collapse(ng, nf, T).astype(np.float64))[0]
    pairs, nblk, nt3 = _reached(x, ng, nf, T)
    assert np.bincount(pairs[:, 1], minlength=nt3).max() > _cap(ng, nf, T, nblk, nt3)
    # and no cell edge is near a particle, so the twin's gradient has no jumps
    assert np.abs(x - np.round(x)).min() > 0.1


@pytest.mark.gpu
@pytest.mark.parametrize("ng,nf,T", [(32, 64, 8), (24, 144, 16)])
def test_collapsed_box(ng, nf, T):
    w = _collapse(ng, nf, T)
    dbar = (np.random.default_rng(4).standard_normal(nf ** 3) / nf ** 3).astype(np.float32)
    ic, steps = np.array([1.0, 0.0]), np.array([[1e-5, 1e-3, 1e-5], [1e-5, 1e-3, 1e-5]])
    ref = Ref(ng, nf, np.ones((ng, ng, ng // 2 + 1)), ic, steps)
    want = ref.forward(w.astype(np.float64)).ravel()
    wantg = ref.adjoint(dbar.astype(np.float64).reshape(nf, nf, nf))
    d, g, _ = _box(ng, nf, ic, steps, w, dbar)
    ed, eg = rel_l2(d, want), rel_l2(g, wantg)
    print(f"ng {ng} nf {nf}: delta {ed:.2e} gradient {eg:.2e}")
    assert ed < 1e-4
    assert eg < 1e-3


@pytest.mark.gpu
def test_scattered_blocks_cost():
    """A block reaches at most 64 (9/8)^3 = 91 8-cell tiles where it reached
    2.5^3 = 16: six times the deposits' work if they were all of it.  (Listed in
    all tiles of the box around them, such blocks took 18 times as long.)"""
    ng, nf = 64, 128
    still = np.array([[0.0, 1e-6, 0.0]] * 3)
    took = []
    for rms in (0.3, 24.0):
        w, dbar, cx = _scattered(ng, nf, rms)
        took.append(_box(ng, nf, np.array([cx, 0.0]), still, w, dbar, passes=15)[2])
    print(f"{took[0] * 1e3:.2f} and {took[1] * 1e3:.2f} ms")
    assert took[1] < 6 * took[0]
