"""The row pass of an nx that is not a power of two with more than 1024 rows, where rows
of up to 128 points run on 64 lanes (csrc/sparc_kernels.hip, any_row_lanes): both sides of
the line in rows and in nx, both parities, one and two values a lane, horizontal PMLs
wider than a lane's stride.  12 steps with flow and bump against the oracle, 1e-11."""
import numpy as np
import pytest

from tests.cases import rel_l2, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import oracle  # noqa: E402
from sparc_flows_amd.solver import Sparc  # noqa: E402


@pytest.mark.parametrize("nx,nz,nsrc,nph", [(17, 33, 32, 3), (62, 40, 26, 5), (63, 33, 32, 20), (65, 41, 25, 7),
                                            (100, 35, 30, 49), (127, 33, 32, 9), (126, 60, 18, 5), (129, 33, 32, 9),
                                            (100, 32, 32, 5)])
def test_steps_match_oracle(nx, nz, nsrc, nph):
    p, bg, c2d, psi = small_case(nx=nx, nz=nz, npml=6, nph=nph)
    maxtime = 12
    xs = list(np.linspace(-60.0, 55.0, nsrc))
    s = Sparc(p, bg, nsrc=nsrc, c2d=c2d, psi=psi)
    vz, sn = s.forward(xs, maxtime, snapshots=True)
    st = s.state()
    for b in (0, nsrc // 2, nsrc - 1):
        o = oracle.Oracle(p, bg, c2d=c2d, psi=psi)
        o.set_forward_source(xs[b], maxtime)
        _, osn = o.run(maxtime, snapshots=True)
        assert np.abs(osn).max() > 0
        assert rel_l2(st[:, b].cpu().numpy(), o.state()) < 1e-11
        assert rel_l2(sn[b].cpu().numpy(), osn) < 1e-11
