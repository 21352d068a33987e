"""The batched circulant derivative (csrc/sparc_kernels.hip, k_circ) on both sides of the
line where blocks hold fewer pairs of lines and split their sums (csrc/sparc_circ.h,
circ_batch): few lines (up to four groups of lanes a pair), the last count that splits and
the first that does not, odd counts.  Against the oracle's direct DFT, 1e-12 as the
operator tests."""
import numpy as np
import pytest

from tests.cases import rel_l2, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import oracle  # noqa: E402
from sparc_flows_amd.solver import Sparc  # noqa: E402
from tests import test_gpu_3d as t3  # noqa: E402


# split up to 512 x (pairs a full block holds / 2) lines: 16384 at 17, 3072 at 96, 2560 at
# 121, 1024 at 250, 512 at 511, never at 999
@pytest.mark.parametrize("nx,rows", [(17, 1), (17, 513), (17, 16384), (17, 16385), (31, 3075), (96, 1), (96, 1026),
                                     (96, 3072), (96, 3073), (121, 515), (121, 2560), (121, 2563), (250, 1023),
                                     (250, 1025), (511, 512), (511, 513), (640, 33), (999, 3)])
def test_ddx(nx, rows):
    nz = 20
    p, bg, _, _ = small_case(nx=nx, nz=nz, npml=4, flow=False, dc=False)
    s, o = Sparc(p, bg), oracle.Oracle(p, bg)
    f = np.random.default_rng(nx + rows).standard_normal((rows, nx))
    got = s.ddx(torch.as_tensor(f, device="cuda")).cpu().numpy()
    assert rel_l2(got, o.ddx(f)) < 1e-12


@pytest.mark.parametrize("nx,ny,nz", [(16, 17, 20), (18, 17, 100), (16, 96, 20), (130, 100, 24), (130, 100, 30),
                                      (16, 250, 30), (34, 250, 35)])
def test_ddy(nx, ny, nz):
    p, bg, _, _ = t3.case(nx=nx, ny=ny, nz=nz, flow=False, dc=False)
    o, s = t3.pair(p, bg, None, None)
    f = np.random.default_rng(ny).standard_normal((1, nz, ny, nx))
    got = s.ddy(torch.as_tensor(f, device="cuda")).cpu().numpy()
    assert rel_l2(got, o.ddy(f)) < 1e-12
