"""The entry point that allocates nothing (p4g_treeLogLikeNoAlloc) against
the ordinary one (p4g_treeLogLike) through the C-ABI: two calls in a row,
the second on a smaller input, both equal to the ordinary entry point's
result bit for bit (the same kernels reduce in the same order); a tree
with no device state yet is refused."""
import numpy
import pytest

from p4gpu import Data, P4Error, Part, func, pf, synth

pytestmark = pytest.mark.gpu


def test_no_alloc_entry_point_matches_tree_log_like():
    assert pf.deviceAvailable()
    big, _ = synth.make_workload("het64", seed=21, nSites=6000, precision="fp32")
    small, _ = synth.make_workload("gtr16", seed=22, nSites=700, precision="fp64")
    for t in (big, small):
        t.calcLogLike(verbose=0)          # sets the tree up (allocates)
    for t in (big, small):
        want = pf.p4_treeLogLike(t.cTree, 0)
        got = pf.treeLogLikeNoAlloc(t.cTree)
        assert got == want, (got, want)
        # the scratch array keeps the last call's contents: a second call
        # after a parameter change still gives the ordinary result
        n = t.nodes[2]
        n.br.len *= 1.25
        pf.p4_setBrLen(n.cNode, n.br.len)
        pf.p4_setPrams(t.cTree, -1)
        got2 = pf.treeLogLikeNoAlloc(t.cTree)
        pf.p4_setPrams(t.cTree, -1)
        want2 = pf.p4_treeLogLike(t.cTree, 0)
        assert got2 == want2 and got2 != got, (got2, want2, got)
        assert numpy.isfinite(got2)


def test_no_alloc_entry_point_refuses_a_tree_without_device_state():
    t, _ = synth.make_workload("gtr16", seed=23, nSites=300, precision="fp64")
    t.calcLogLike(verbose=0)
    t.setPrecision("fp32")   # the FP32 partials do not exist yet
    with pytest.raises(P4Error, match="evaluate it once"):
        pf.treeLogLikeNoAlloc(t.cTree)
    v = t.calcLogLike(verbose=0)
    pf.p4_setPrams(t.cTree, -1)
    assert pf.treeLogLikeNoAlloc(t.cTree) == v


def test_no_alloc_limit_is_the_launchs_own_need():
    """A 20-state part of 44,000 tiles: its workgroups need 0.5 MB of scratch,
    which is there, whatever setAaTuning was told."""
    rng = numpy.random.default_rng(24)
    nPat, names = 44000 * 16 - 5, ["a", "b", "c", "d"]
    t = func.readNewick("((a:0.1,b:0.2):0.05,c:0.3,d:0.1);")
    t.taxNames = names
    codes = rng.integers(0, 20, (4, nPat))
    t.data = Data(parts=[Part.fromPatterns(codes, numpy.ones(nPat, int), "protein")], taxNames=names)
    t.newComp(free=1, spec="specified", val=list(rng.dirichlet(numpy.full(20, 5.0))))
    t.newRMatrix(free=1, spec="specified", val=list(rng.lognormal(0, 1, 190)))
    t.setNGammaCat(nGammaCat=1)
    t.setPInvar(free=0, val=0.0)
    t.setPrecision("fp32")
    want = t.calcLogLike(verbose=0)
    try:
        for on in (True, False):
            pf.setAaTuning(on, 0)
            pf.p4_setPrams(t.cTree, -1)
            assert pf.treeLogLikeNoAlloc(t.cTree) == want
    finally:
        pf.setAaTuning(True)
