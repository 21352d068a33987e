"""The segmented z kernels (csrc/sparc_zseg.hip) at the sizes where their
indexing can go wrong: the shortest and longest segments, both segment
counts (16 up to nz = 160, 32 above), a last segment of three rows, the
first nz the one-lane sweeps take (513, and 337, which no cut fits), column
counts that are not multiples of a block's 16 or 32, PML layers wider than a
segment.  Against the oracles, tolerances as in the operator and one-step
tests (segmented solves differ from the Thomas sweeps by rounding).  The
oracle takes the library's own vertical stretch: both invert dbyd2 of
z = 1 + height / R_sun, whose rounding (a few parts in 1e16 of 1 against a row
spacing of 1e-4) differs between them and would drown what is compared here."""
import numpy as np
import pytest

from tests.cases import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from oracle.oracle3d import _dbyd2  # noqa: E402
from tests.test_gpu_3d import case, pair  # noqa: E402


def share_stretch(o, s):
    """The library's stretch, from its z-derivative of the row number, in the oracle."""
    p = o.p
    ramp = np.arange(p.nz, dtype=np.float64)
    f = np.broadcast_to(ramp[:, None, None], (p.nz, p.ny, p.nx))
    lib = s.ddz(torch.as_tensor(np.ascontiguousarray(f), device="cuda"), 1).cpu().numpy()[:, 0, 0]
    ratio = lib / (_dbyd2(ramp, 1)[:, 0] * o.stretch)
    o.stretch = o.stretch * ratio
    o.gp0 = o.gp0 * ratio[:, None, None]
    o.gr0 = o.gr0 * ratio[:, None, None]


@pytest.mark.parametrize("nx,ny,nz,npml", [
    (18, 17, 16, 5), (16, 16, 35, 6), (18, 17, 63, 12), (100, 96, 43, 6), (16, 17, 160, 12), (16, 17, 161, 12),
    (18, 17, 300, 30), (16, 16, 323, 8), (16, 17, 337, 8), (16, 16, 512, 12), (16, 16, 513, 12)])
def test_two_steps_match_oracle(nx, ny, nz, npml):
    """Two STEPs from a seeded state (the second with the z filter), with the
    PML variables and the last stage's accelerations."""
    p, bg, c3d, fl = case(nx=nx, ny=ny, nz=nz, npml=npml)
    o, s = pair(p, bg, c3d, fl)
    share_stretch(o, s)
    o.set_forward_source(3.0, -2.0, 50)
    s.set_forward_source(3.0, -2.0, 50)
    a0 = 1e-8 * np.random.default_rng(2).standard_normal((6, nz, ny, nx))
    o.a = a0.copy()
    s.set_state(torch.as_tensor(a0, device="cuda"))
    for t in (0, 1):
        o.step(t)
        s.step(t)
    got, scr = s.state().cpu().numpy(), s.scr().cpu().numpy()
    for f in range(6):
        assert rel_l2(got[f], o.a[f]) < 1e-11, f
    assert rel_l2(s.pml().cpu().numpy(), o.pmlvars) < 1e-11
    for f in range(6):
        assert rel_l2(scr[f], o.scr[f]) < 1e-11, f
