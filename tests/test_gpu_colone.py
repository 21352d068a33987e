"""The column pass of large batches (csrc/sparc_colseg.hip: from 450 000 points on, at
segment lengths of 4, 6 and 8, k_colone or k_colsplit by the blocks that a compute unit
holds) at every launch shape that the autotuner can choose for a grid, each forced, so
that no timing outcome can select a shape that is not compared here.  Grids: both parities
of nz, a last segment of three rows, PML layers that end inside a segment, the deepest
grids of each length.

Against the oracle, 1e-11 on the state after 40 steps as in the step tests and 1e-10 on
traces and snapshots; every source of a shape against the first shape's, 1e-13 as in the
batch tests (segmentation changes rounding only).  The sources of all three kinds."""
import numpy as np
import pytest

from tests.cases import adjoint_source, rel_l2, small_case

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

import oracle  # noqa: E402
from sparc_flows_amd.solver import Sparc  # noqa: E402
from sparc_flows_amd.sources import gaussian_force  # noqa: E402

NX = 256
GRIDS = [(111, 16), (247, 8), (300, 8), (403, 8)]


def shapes(nz):
    """colsplit_fits (these grids' blocks all fit the LDS)."""
    for ms in (4, 6, 8):
        p = -(-nz // ms)
        if p <= 64 and nz - (p - 1) * ms >= 3:
            for tc in (1, 2, 4, 8, 16):
                if tc * p <= 512:
                    yield ms, tc


def force(monkeypatch, ms, tc):
    monkeypatch.setenv("SPARC_COLSEG_MS", str(ms))
    monkeypatch.setenv("SPARC_COLSEG_TC", str(tc))


def applied(s, ms, tc):
    """The forced shape is the one that ran; above 128 lanes in its one-lane form."""
    shape = s.query("colseg_ms"), s.query("colseg_tc")
    return shape == (ms, tc) and (s.query("colseg_one") == 1 or tc * s.query("colseg_p") <= 128)


@pytest.mark.parametrize("nz,nsrc", GRIDS)
def test_every_shape_matches_oracle(nz, nsrc, monkeypatch):
    p, bg, c2d, psi = small_case(nx=NX, nz=nz, npml=13, nph=9)
    maxtime = 40
    xs = list(np.linspace(-60.0, 55.0, nsrc))
    refs = {}
    for b in (0, nsrc - 1):
        o = oracle.Oracle(p, bg, c2d=c2d, psi=psi)
        o.set_forward_source(xs[b], maxtime)
        vz, sn = o.run(maxtime, snapshots=True)
        refs[b] = vz, sn, o.state()
        assert np.abs(vz).max() > 0
    base, bad, count = None, [], 0
    for ms, tc in shapes(nz):
        force(monkeypatch, ms, tc)
        s = Sparc(p, bg, nsrc=nsrc, c2d=c2d, psi=psi)
        print("nz", nz, "MS", ms, "TC", tc, flush=True)
        vz, sn = s.forward(xs, maxtime, snapshots=True)
        assert applied(s, ms, tc)
        st = s.state()
        base = st if base is None else base
        e_o = max(rel_l2(st[:, b].cpu().numpy(), refs[b][2]) for b in refs)
        e_t = max(max(rel_l2(vz[b].cpu().numpy(), refs[b][0]), rel_l2(sn[b].cpu().numpy(), refs[b][1])) for b in refs)
        e_b = float(((st - base).square().sum((0, 2, 3)) / base.square().sum((0, 2, 3))).sqrt().max())
        count += 1
        if not (e_o < 1e-11 and e_t < 1e-10 and e_b < 1e-13):
            bad.append((ms, tc, e_o, e_t, e_b))
    assert count and not bad, bad


@pytest.mark.parametrize("ms,tc", [(4, 8), (6, 8), (8, 16)])
@pytest.mark.parametrize("kind", ["adjoint", "profile"])
def test_other_sources_match_oracle(kind, ms, tc, monkeypatch):
    """The adjoint's interpolated receivers and the force with a vertical profile."""
    nz, nsrc = 111, 16
    p, bg, c2d, psi = small_case(nx=NX, nz=nz, npml=13, nph=9)
    adj = kind == "adjoint"
    maxtime = 2 * p.cadforcing_step + 5
    force(monkeypatch, ms, tc)
    s = Sparc(p, bg, nsrc=nsrc, adjoint=adj, c2d=c2d, psi=psi)
    o = {b: oracle.Oracle(p, bg, c2d=c2d, psi=psi, adjoint=adj) for b in (0, nsrc - 1)}
    if adj:
        nt = maxtime // p.cadforcing_step + 1
        vr = np.stack([adjoint_source(p, nt, NX, seed=b) for b in range(nsrc)])
        s.set_adjoint_sources(torch.as_tensor(vr, device="cuda"), maxtime)
        for b in o:
            o[b].set_adjoint_source(vr[b], maxtime)
    else:
        vr, zp, ser = gaussian_force(p, bg, np.linspace(-60.0, 55.0, nsrc), maxtime)
        s.set_forward_profile(vr, zp, ser, maxtime)
        for b in o:
            o[b].set_forward_profile(vr[b], zp, ser, maxtime)
    _, sn = s.run(snapshots=True)
    assert applied(s, ms, tc) and s.query("colseg_one") == 1
    for b in o:
        _, osn = o[b].run(maxtime, snapshots=True)
        assert np.abs(osn).max() > 0
        assert rel_l2(s.state()[:, b].cpu().numpy(), o[b].state()) < 1e-11
        assert rel_l2(sn[b].cpu().numpy(), osn) < 1e-10


@pytest.mark.parametrize("nx,nz,nsrc,ms,tc,one", [
    (100, 100, 64, 8, 4, 0), (100, 100, 64, 6, 4, 1), (250, 150, 16, 8, 2, 0), (255, 300, 8, 6, 1, 0),
    (256, 60, 100, 8, 8, 0), (300, 60, 30, 6, 4, 0), (17, 40, 1000, 6, 1, 1), (33, 32, 440, 8, 1, 1),
    (33, 44, 400, 4, 1, 0), (33, 44, 300, 4, 1, 0)])
def test_form_of_narrow_blocks(nx, nz, nsrc, ms, tc, one, monkeypatch):
    """Blocks that fit both forms take the faster one (the last case lies below 450 000
    points); 12 steps of the first and last source against the oracle."""
    npml = 12 if nz >= 60 else 6
    p, bg, c2d, psi = small_case(nx=nx, nz=nz, npml=npml, nph=4)
    force(monkeypatch, ms, tc)
    xs = list(np.linspace(-60.0, 55.0, nsrc))
    s = Sparc(p, bg, nsrc=nsrc, c2d=c2d, psi=psi)
    s.set_forward_sources(xs, 30)
    s.reset()
    s.run_range(0, 11)
    assert (s.query("colseg_ms"), s.query("colseg_tc"), s.query("colseg_one")) == (ms, tc, one)
    st = s.state()
    for b in (0, nsrc - 1):
        o = oracle.Oracle(p, bg, c2d=c2d, psi=psi)
        o.set_forward_source(xs[b], 30)
        for t in range(12):
            o.step(t)
        assert rel_l2(st[:, b].cpu().numpy(), o.state()) < 1e-11
