"""The discrete adjoint's stages where their indexing can go wrong: odd sizes and
sources (row pairs that straddle two fields), segments of the recompute whose last
one is short, an nz beyond the segmented z-derivative (dense matrices, column sum),
every z row count modulo the filter's eight.  Against the oracle, to the 1e-9 of the
discrete-gradient tests; the segment length does not change the result beyond 1e-13
(the same operations on recomputed states)."""
import numpy as np
import pytest

from tests.cases import rel_l2, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import oracle  # noqa: E402
from sparc_flows_amd.solver import Sparc  # noqa: E402


@pytest.mark.parametrize("nx,nz,nsrc,maxtime", [(64, 33, 1, 11), (75, 37, 3, 12), (64, 40, 2, 8), (48, 39, 5, 9),
                                                (16, 1030, 1, 5)])
def test_gradient_sizes_and_segments(nx, nz, nsrc, maxtime):
    npml = 6 if nz > 40 else 4
    p, bg, c2d, psi = small_case(nx=nx, nz=nz, npml=npml, nph=3, flow=True, dc=True)
    xs = list(np.linspace(-20.0, 15.0, nsrc))
    gvz = np.random.default_rng(nx).standard_normal((nsrc, p.nt_out(maxtime), nx))
    s = Sparc(p, bg, nsrc=nsrc, c2d=c2d, psi=psi)
    s.set_forward_sources(xs, maxtime)
    g = torch.as_tensor(gvz, device="cuda")
    ref = s.discrete_gradient(g, interval=0, psi=True)[2].cpu().numpy()
    for interval in (1, 4):
        got = s.discrete_gradient(g, interval=interval, psi=True)[2].cpu().numpy()
        assert rel_l2(got, ref) < 1e-13
    for b in {0, nsrc - 1}:
        o = oracle.Oracle(p, bg, c2d=c2d, psi=psi)
        o.set_forward_source(xs[b], maxtime)
        for k, want in enumerate(o.discrete_gradient(maxtime, gvz[b])[:3]):
            assert rel_l2(ref[k, b], want) < 1e-9, (b, k)
