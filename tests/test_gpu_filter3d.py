"""FILTER_VARS_3D_HORIZ_PML (csrc/sparc_3d.hip, k3_filter) with one and with eight rows in
flight per lane (launch_filter): layer thicknesses from the narrowest that is accepted,
filtered row counts that are and are not multiples of eight.  The filtered step of a seeded
state against the 3D oracle, 1e-11 as the one-step test."""
import numpy as np
import pytest

from tests.cases import rel_l2

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from tests.test_gpu_3d import case, pair  # noqa: E402


# eight rows up to 58 240 columns; one row at 256 x 240 (0.70 of a round of blocks)
@pytest.mark.parametrize("nx,ny,nz,npml", [(32, 16, 16, 5), (32, 17, 27, 5), (64, 64, 33, 6), (256, 240, 19, 5),
                                           (256, 240, 28, 6), (256, 228, 18, 5)])
def test_filtered_step_matches_oracle(nx, ny, nz, npml):
    p, bg, c3d, fl = case(nx=nx, ny=ny, nz=nz, npml=npml)
    o, s = pair(p, bg, c3d, fl)
    o.set_forward_source(3.0, -2.0, 50)
    s.set_forward_source(3.0, -2.0, 50)
    a0 = 1e-8 * np.random.default_rng(nz).standard_normal((6, nz, ny, nx))
    o.a = a0.copy()
    s.set_state(torch.as_tensor(a0, device="cuda"))
    o.step(1)
    s.step(1)
    got = s.state().cpu().numpy()
    for f in range(6):
        assert rel_l2(got[f], o.a[f]) < 1e-11, f
