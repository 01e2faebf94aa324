"""GPU: the event/walk passes at queue lengths around their claim sizes (16 to 128 requests, 64 lanes), with one and
two slot groups and several emission batches, against the lane pipeline's same packet histories."""
import numpy as np
import pytest

from skirt7_amd import capi
from skirt7_amd import skirt as S
from skirt7_amd import workloads
from skirt7_amd.capi import SG_FP64, SG_MIXED

pytestmark = pytest.mark.gpu


def _run(w, count, precision):
    w["instr"].clear()
    c = w["sim"].run_packets(0, 3, count, 1000, precision)
    frames = np.concatenate([w["instr"].frame(i).ravel() for i in range(3)])
    return frames, {k: c[k] for k in ("packets", "own_crossings", "peel_crossings", "rewalk_crossings", "scatterings",
                                      "peeloffs", "walks")}


@pytest.fixture(scope="module")
def disc():
    return workloads.disc_cartesian(grid_n=14, pixels=24, packages=1000)


@pytest.mark.parametrize("precision", [SG_FP64, SG_MIXED])
@pytest.mark.parametrize("count,groups,batch", [(1, 2, 0), (2, 2, 0), (3, 1, 0), (4, 2, 0), (16, 1, 0), (17, 2, 0),
                                                (63, 1, 0), (129, 2, 64), (700, 2, 0), (701, 1, 100), (5001, 2, 1024),
                                                (130, 0, 64), (3000, 0, 0)])
def test_passes_equal_the_lane_pipeline(disc, count, groups, batch, precision):
    # the histories are the same, only the order of the tally additions differs: the sums of up to a few hundred
    # thousand positive FP64 terms agree to n eps < 1e-10
    try:
        S.set_pipeline(0)
        ref, cref = _run(disc, count, precision)
        S.set_pipeline(1)
        S.set_slot_groups(groups)
        S.set_emit_batch(batch)
        out, c = _run(disc, count, precision)
    finally:
        S.set_pipeline(1)
        S.set_slot_groups(0)
        S.set_emit_batch(0)
    assert c == cref
    np.testing.assert_allclose(out, ref, rtol=1e-10, atol=0)


@pytest.mark.parametrize("kind,chosen", [("cartesian", 1), ("voronoi", 2)])
def test_slot_groups_return_to_the_runs_choice(kind, chosen):
    """Set and set back to 0, a run takes the groups it chooses by itself: one on a Cartesian grid, two on a Voronoi
    grid, by its walk launches (every pass of every group; all packets start in the first pass, so that the number
    of passes is the packets' own)."""
    w = workloads.two_dust_disc(kind, grid_n=12, nsites=600, pixels=20, packages=4000)
    launches = {}
    try:
        for groups in (1, 2, 0):
            S.set_slot_groups(groups)
            launches[groups] = w["sim"].run_packets(0, 0, 2000, 2000, SG_FP64)["transport_launches"]
        for bad in (-1, 3):
            with pytest.raises(S.FatalError):
                S.set_slot_groups(bad)
    finally:
        S.set_slot_groups(0)
    assert launches[1] < launches[2] and launches[0] == launches[chosen]


@pytest.mark.parametrize("lists", ["as built", "shuffled", "superset"])
def test_voronoi_walks_of_several_lanes(lists):
    """The walk kernel's Voronoi walk (a group of lanes per walk) against the lane pipeline's (one lane): lists with
    their walls first, lists in any order, and lists longer than an entry's count holds (more than 127)."""
    rng = np.random.default_rng(3)
    ext = np.array([-20.0, -20.0, -20.0, 20.0, 20.0, 20.0])
    sites = ext[:3] + rng.random((400, 3)) * 40.0
    off, ids = S.voronoi_neighbors(ext, sites)
    per = [ids[off[i]:off[i + 1]] for i in range(len(sites))]
    if lists == "shuffled":
        per = [rng.permutation(p) for p in per]
    elif lists == "superset":
        # more sites than neighbours: planes beyond the cell's faces are never the nearest ahead
        extra = [np.setdiff1d(rng.choice(len(sites), 150, replace=False), np.append(p, i)) for i, p in enumerate(per)]
        per = [np.concatenate([p, e]).astype(np.int32) for p, e in zip(per, extra)]
        assert max(len(p) for p in per) > 127
    off = np.concatenate([[0], np.cumsum([len(p) for p in per])])
    grid = S.VoronoiDustGrid(ext, sites, off, np.concatenate(per))
    w = workloads.disc_cartesian(grid_n=4, pixels=20, packages=100)
    stars, mix = w["stars"], w["mix"]
    out = []
    for mode in (0, 1):
        dust = S.DustSystem(grid, np.full(len(sites), 0.05), mix, writeMeanIntensity=True)
        w["instr"].clear()
        sim = S.OligoMonteCarloSimulation(dust, stars, w["instr"], packages=3000, seed=11)
        try:
            S.set_pipeline(mode)
            c = sim.run_packets(0, 0, 3000, 3000, SG_FP64)
        finally:
            S.set_pipeline(1)
        out.append((np.concatenate([w["instr"].frame(i).ravel() for i in range(3)]), dust.Labs(), c["own_crossings"],
                    c["peel_crossings"], c["rewalk_crossings"], c["scatterings"]))
    assert out[0][2:] == out[1][2:]
    # sums of at most some ten thousand positive FP64 terms in another order
    np.testing.assert_allclose(out[1][0], out[0][0], rtol=1e-11, atol=0)
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=1e-11, atol=0)


@pytest.mark.parametrize("kind", ["cartesian", "octree", "voronoi"])
@pytest.mark.parametrize("precision", [SG_FP64, SG_MIXED])
@pytest.mark.parametrize("count,batch", [(1, 0), (511, 0), (513, 128), (3001, 0)])
def test_passes_of_several_dust_components(kind, precision, count, batch):
    """Two dust components in the passes against the lane pipeline, at packet counts around the event kernel's
    workgroup (512 slots): the same histories, absorption and counts."""
    w = workloads.two_dust_disc(kind, grid_n=12, maxlevel=4, nsites=600, pixels=20, packages=4000)
    out = []
    for mode in (0, 1):
        w["instr"].clear()
        w["dust"].clear()
        try:
            S.set_pipeline(mode)
            S.set_emit_batch(batch)
            c = w["sim"].run_packets(1, 5, count, count, precision)
        finally:
            S.set_pipeline(1)
            S.set_emit_batch(0)
        n = len(w["instr"].instruments)
        out.append((np.concatenate([w["instr"].frame(i).ravel() for i in range(n)]), w["dust"].Labs(),
                    {k: c[k] for k in ("packets", "own_crossings", "peel_crossings", "rewalk_crossings", "scatterings",
                                       "peeloffs", "walks")}))
    assert out[0][2] == out[1][2]
    # sums of at most some ten thousand positive FP64 terms in another order
    np.testing.assert_allclose(out[1][0], out[0][0], rtol=1e-11, atol=0)
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=1e-11, atol=0)


@pytest.mark.parametrize("precision", [SG_FP64, SG_MIXED])
@pytest.mark.parametrize("alone,batch", [(1, 0), (1, 1000), (900, 0)])
def test_batched_members_by_passes(alone, batch, precision):
    """More members than there are streams, each by passes of its own (from one packet up; with small emission batches
    the larger ones one at a time), or some of them in the shared launch, against their single runs."""
    counts = [700, 1, 3000, 64, 1500, 129, 2, 901]
    pop = workloads.fit_population(members=len(counts), packets=(1.0e3, 3.0e3), grid_n=(6, 14), pixels=(32, 16), nsamples=2)
    ms = pop["members"]
    single, walks = [], 0
    for m, n in zip(ms, counts):
        m["instr"].clear()
        walks += m["sim"].run_packets(0, 0, n, n, precision)["walks"]
        single.append(m["instr"].frame(0)[0].copy())
        m["instr"].clear()
    try:
        S.set_batch_alone(alone)
        S.set_emit_batch(batch)
        c = S.run_batch([m["sim"] for m in ms], counts, precision=precision)
    finally:
        S.set_batch_alone(3 << 16)
        S.set_emit_batch(0)
    assert c["packets"] == sum(counts) and c["walks"] == walks
    for m, f in zip(ms, single):
        # sums of at most some thousand positive FP64 terms in another order
        np.testing.assert_allclose(m["instr"].frame(0)[0], f, rtol=1e-11, atol=0)


@pytest.mark.parametrize("alone", [1, 100000])
def test_batched_run_reports_its_span(alone):
    """Members' passes overlap, beside each other and the shared launches: the transport's span lies within the whole
    call's."""
    pop = workloads.fit_population(members=8, packets=(1.0e3, 3.0e3), grid_n=(30, 50), pixels=(32, 16), nsamples=2)
    try:
        S.set_batch_alone(alone)
        for _ in range(2):   # the first call allocates the members' buffers
            c = S.run_batch([m["sim"] for m in pop["members"]], [60000] * 3 + [250000] * 5, precision=SG_MIXED)
    finally:
        S.set_batch_alone(3 << 16)
    assert 0 < c["transport_us"] <= c["kernel_us"]


@pytest.mark.parametrize("kind", ["cartesian", "octree"])
@pytest.mark.parametrize("count,batch", [(1, 0), (513, 0), (3001, 1024)])
def test_dust_emission_by_passes(kind, count, batch):
    """Dust emission in the passes against the lane pipeline: the same histories, with peel-offs and with absorption."""
    w = workloads.pan_disc(kind=kind, nlambda=12, grid_n=10, maxlevel=3, pixels=16, packages=500)
    pan = w["pan"]
    nc = w["grid"].numCells()
    Lv = np.ascontiguousarray(np.random.default_rng(4).random(nc))
    out = []
    for mode in (0, 1):
        pan.dust.ds.clear()
        w["instr"].clear()
        c = np.zeros(capi.SG_NCOUNTERS, np.uint64)
        try:
            S.set_pipeline(mode)
            S.set_emit_batch(batch)
            for peel in (1, 0):
                capi.check(capi.lib().sg_sim_run_dust(pan.sim._h, 9, 0, count, count, capi.dptr(Lv), 0.5, peel, 1 - peel, 5,
                                                      SG_MIXED, c.ctypes.data_as(capi._U64)))
        finally:
            S.set_pipeline(1)
            S.set_emit_batch(0)
        out.append((np.concatenate([w["instr"].frame(i).ravel() for i in range(len(w["instr"].instruments))]),
                    pan.dust.ds.Labs(), [int(c[k]) for k in (0, 1, 2, 3, 4, 7, 8)]))
    assert out[0][2] == out[1][2]
    np.testing.assert_allclose(out[1][0], out[0][0], rtol=1e-11, atol=0)
    np.testing.assert_allclose(out[1][1], out[0][1], rtol=1e-11, atol=0)
