"""Device memory of a 3D handle whose z passes run segmented: 34 fields of state, work
and background, one of sweep values and the layers', no room for four sweeps."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from sparc_flows_amd import background as B  # noqa: E402
from sparc_flows_amd.solver3d import Params3D, Sparc3D  # noqa: E402


def test_segmented_handle_holds_no_sweep_buffers():
    def create(n, nz):
        bg = B.polytrope(nz)
        return Sparc3D(Params3D(nx=n, ny=n, nz=nz, timestep=B.stable_timestep(bg), npmlbot=12, npmltop=12), bg)

    keep = create(32, 40)                       # loads the library's code
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    s = create(128, 150)
    torch.cuda.synchronize()
    fields = (free0 - torch.cuda.mem_get_info()[0]) / (8 * 128 * 128 * 150)
    assert 34 < fields < 37.5, fields           # az, bz, fz and four arrays of 24 of 150 rows: 1.1
    del s, keep
