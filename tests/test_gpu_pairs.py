"""The row-pair fields and the two forms of the column pass (csrc/
sparc_colseg.hip) where their indexing can go wrong: an odd nz (a pad row), the
one-lane form that batches of 450 000 points and more take (16 sources at
256 x 111 and more), grids whose nx is not a power of two, a last segment of three
rows.  Against the oracle, tolerance as in the step tests (1e-11) and the trace
tests (1e-10), and batch against single source (which take different forms) at
the batch tests' 1e-13."""
import numpy as np
import pytest

from tests.cases import rel_l2, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import oracle  # noqa: E402
from sparc_flows_amd.solver import Sparc  # noqa: E402


@pytest.mark.parametrize("nx,nz,nsrc", [(64, 61, 2), (75, 33, 3), (256, 111, 16), (256, 123, 16), (300, 157, 10),
                                        (64, 299, 24)])
def test_run_snapshots_and_state_round_trip(nx, nz, nsrc):
    npml = 6 if nz > 40 else 4
    p, bg, c2d, psi = small_case(nx=nx, nz=nz, npml=npml, flow=True, dc=True)
    steps = p.steps
    maxtime = 2 * steps + 3
    xs = list(np.linspace(-12.0, 12.0, nsrc))
    s = Sparc(p, bg, nsrc=nsrc, c2d=c2d, psi=psi)
    norm2 = s.record_norms(maxtime + 1)
    vz, sn = s.forward(xs, maxtime, snapshots=True)
    state = s.state()
    for b in (0, nsrc - 1):
        o = oracle.Oracle(p, bg, c2d=c2d, psi=psi)
        o.set_forward_source(xs[b], maxtime)
        ovz, osn = o.run(maxtime, snapshots=True)
        assert np.abs(ovz).max() > 0
        assert rel_l2(vz[b].cpu().numpy(), ovz) < 1e-10
        assert rel_l2(sn[b].cpu().numpy(), osn) < 1e-10
        assert rel_l2(state[:, b].cpu().numpy(), o.state()) < 1e-10
        # the norm is a sum over the whole array: a pad row must hold nothing
        assert abs(float(norm2[b, maxtime]) / float((state[3, b] ** 2).sum()) - 1.0) < 1e-13
    s1 = Sparc(p, bg, nsrc=1, c2d=c2d, psi=psi)
    s1.forward([xs[0]], maxtime)
    assert rel_l2(state[:, 0].cpu().numpy(), s1.state()[:, 0].cpu().numpy()) < 1e-13
    # state and checkpoint through their plain layouts, bit for bit, then one more
    # step from each
    s.record_norms(None)
    ck = s.checkpoint_buffer()[0]
    s.set_forward_sources(xs, maxtime + 2)
    s.save_checkpoint(ck)
    assert torch.equal(ck[: state.numel()].reshape(state.shape), state)
    s.step(maxtime + 1)
    a = s.state()
    s.set_state(torch.zeros_like(state))
    s.load_checkpoint(ck)
    assert torch.equal(s.state(), state)
    s.step(maxtime + 1)
    assert torch.equal(s.state(), a)


@pytest.mark.parametrize("nz", [121, 482, 721, 722, 758, 841, 1024])
@pytest.mark.parametrize("nsrc", [1, 24])
def test_depths_that_only_long_segments_cut(nz, nsrc):
    """Depths whose last segment would hold fewer than three rows at every length up
    to 12 (at 721 and 722: at every length but 22), and the deepest: 6 steps of one
    source and of a batch against the oracle, 1e-11."""
    p, bg, c2d, psi = small_case(nx=32, nz=nz, npml=10, nph=4)
    xs = list(np.linspace(-12.0, 12.0, nsrc))
    s = Sparc(p, bg, nsrc=nsrc, c2d=c2d, psi=psi)
    s.set_forward_sources(xs, 30)
    s.reset()
    for t in range(6):
        s.step(t)
    state = s.state().cpu().numpy()
    for b in {0, nsrc - 1}:
        o = oracle.Oracle(p, bg, c2d=c2d, psi=psi)
        o.set_forward_source(xs[b], 30)
        for t in range(6):
            o.step(t)
        assert rel_l2(state[:, b], o.state()) < 1e-11, (s.query("colseg_ms"), s.query("colseg_tc"))
