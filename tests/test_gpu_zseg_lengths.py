"""The segment lengths of the 3D z passes (csrc/sparc_zseg.hip) that tests/test_gpu_zseg.py
leaves out: 5, 7 and 8, and 14, whose velocity pass keeps registers in scratch, as do 12
and 16 (nz = 121, 141, 241, 301 and eighteen more below 320); on blocks of 16 and of 32
columns, and on grids that give every compute unit more than one block.  Two steps against
the 3D oracle, with that file's tolerance."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import tests.test_gpu_zseg as zseg  # noqa: E402


@pytest.mark.parametrize("nx,ny,nz,npml", [
    (16, 17, 78, 6), (18, 17, 108, 11), (16, 16, 128, 12), (16, 17, 121, 12), (18, 17, 241, 13), (96, 90, 301, 12),
    (128, 128, 121, 12), (128, 130, 141, 12), (128, 66, 78, 6), (96, 90, 108, 11), (100, 96, 126, 12), (96, 90, 150, 13),
    (96, 90, 62, 6)])
def test_two_steps_match_oracle(nx, ny, nz, npml):
    zseg.test_two_steps_match_oracle(nx, ny, nz, npml)
