"""Shared test helpers: golden fixtures and rebuilding trees from them."""
import os

import numpy

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")

LNL_CASES = ["gtr16_500", "het64_800", "prot128_150", "edge_dna_gaps_pinv",
             "multifurcation_root4", "leaf_root"]


def load(name):
    return dict(numpy.load(os.path.join(GOLDEN, name + ".npz"), allow_pickle=False))


def flat_from_fixture(fx):
    import oracle
    return oracle.Flat(parent=fx["parent"], leftChild=fx["leftChild"], sibling=fx["sibling"],
                       isLeaf=fx["isLeaf"], seqNum=fx["seqNum"], brLen=fx["brLen"],
                       postOrder=fx["postOrder"], root=int(fx["root"]), compNums=fx["compNums"],
                       rMatrixNums=fx["rMatrixNums"], gdasrvNums=fx["gdasrvNums"],
                       dim=int(fx["dim"]), nCat=int(fx["nCat"]), comps=fx["comps"],
                       bigR=fx["bigR"], rates=_rates(fx), alphas=fx["alphas"],
                       pInvar=float(fx["pInvar"]), relRate=float(fx["relRate"]),
                       patterns=fx["patterns"], counts=fx["counts"], equates=fx["equates"],
                       invarVec=numpy.zeros(1), invarArray=numpy.zeros(1))


def _rates(fx):
    import oracle
    K = int(fx["nCat"])
    if K == 1:
        return numpy.ones((1, 1))
    return numpy.array([oracle.discrete_gamma(float(a), K) for a in fx["alphas"]])


def oracle_flat(fx):
    """Flat description with invariant sites computed by the oracle."""
    import oracle
    f = flat_from_fixture(fx)
    iv, ia = oracle.invar_sites(f.patterns, f.dim, f.equates)
    kw = dict(f.kwargs)
    kw.update(invarVec=iv, invarArray=ia)
    return oracle.Flat(**kw)


def tree_from_fixture(fx, precision="fp64"):
    """A p4gpu Tree with the fixture's topology, model and patterns."""
    from p4gpu import Data, Part, Tree
    from p4gpu.node import Node
    N = len(fx["parent"])
    t = Tree()
    for i in range(N):
        n = Node()
        n.nodeNum = i
        n.isLeaf = int(fx["isLeaf"][i])
        n.seqNum = int(fx["seqNum"][i])
        if n.isLeaf:
            n.name = "t%d" % n.seqNum
        n.br.len = float(fx["brLen"][i]) if i != int(fx["root"]) else 0.1
        t.nodes.append(n)
    for i, n in enumerate(t.nodes):
        p, l, s = int(fx["parent"][i]), int(fx["leftChild"][i]), int(fx["sibling"][i])
        n.parent = t.nodes[p] if p >= 0 else None
        n.leftChild = t.nodes[l] if l >= 0 else None
        n.sibling = t.nodes[s] if s >= 0 else None
    t.root = t.nodes[int(fx["root"])]
    t.setPreAndPostOrder()
    dt = str(fx["dataType"])
    nTax = fx["patterns"].shape[0]
    part = Part.fromPatterns(fx["patterns"], fx["counts"], dt)
    t.data = Data(parts=[part], taxNames=["t%d" % i for i in range(nTax)])
    dim = int(fx["dim"])
    for c in fx["comps"]:
        t.newComp(free=1, spec="specified", val=list(c))
    iu = numpy.triu_indices(dim, 1)
    for R in fx["bigR"]:
        t.newRMatrix(free=1, spec="specified", val=list(R[iu]))
    K = int(fx["nCat"])
    t.setNGammaCat(nGammaCat=K)
    if K > 1:
        for a in fx["alphas"]:
            t.newGdasrv(free=1, val=float(a))
    t.setPInvar(free=1, val=float(fx["pInvar"]))
    if float(fx["relRate"]) != 1.0:
        t.setRelRate(val=float(fx["relRate"]))
    for i, n in enumerate(t.nodes):
        n.parts[0].compNum = int(fx["compNums"][i])
        if n is not t.root:
            n.br.parts[0].rMatrixNum = int(fx["rMatrixNums"][i])
            n.br.parts[0].gdasrvNum = int(fx["gdasrvNums"][i]) if K > 1 else -1
    t.precision = precision
    return t


def wide_partials(f):
    """{node: partials [nCat][dim][nPat]} of every internal node in 80-bit
    floats, whose exponents reach 2^-16382: site likelihoods far below a
    double's range stay exact.  P from exp(Q t), whose small entries are
    accurate however small t is (the eigensystem leaves 1e-17 of rounding in
    their place)."""
    import oracle
    import scipy.linalg
    K, S, nP = f.nCat, f.dim, f.patterns.shape[1]
    P = {}

    def pmat(n, k):
        t = f.brLen[n] * f.rates[f.gdasrvNums[n]][k] * f.relRate / (1.0 - f.pInvar)
        key = (int(f.rMatrixNums[n]), int(f.compNums[n]), t)
        if key not in P:
            P[key] = scipy.linalg.expm(oracle.bigq(f.bigR[key[0]], f.comps[key[1]]) * t).astype(numpy.longdouble)
        return P[key]

    # a tip code's states: one, all (gap, '?'), or the equate's
    tip = {c: numpy.eye(S)[c] for c in range(S)}
    tip.update({-1: numpy.ones(S), -2: numpy.ones(S)})
    tip.update({e - 64: numpy.asarray(row, float) for e, row in enumerate(f.equates)})
    kids = {}
    for n, p in enumerate(f.parent):
        if p >= 0:
            kids.setdefault(int(p), []).append(n)
    cl = {}
    for n in f.postOrder:
        n = int(n)
        if n not in kids:
            continue
        x = numpy.ones((K, S, nP), numpy.longdouble)
        for c in kids[n]:
            y = cl[c] if c in kids else [numpy.stack([tip[int(a)] for a in f.patterns[f.seqNum[c]]], axis=1)] * K
            x *= numpy.stack([pmat(c, k) @ y[k] for k in range(K)])
        cl[n] = x
        if n == int(f.root):
            return cl


def wide_root_cl(f):
    """The root's partials of wide_partials."""
    return wide_partials(f)[int(f.root)]


def wide_loglike(f):
    """The part's lnL from wide_root_cl (no invariant sites)."""
    assert f.pInvar == 0.0
    pi = numpy.asarray(f.comps)[int(f.compNums[f.root])]
    like = numpy.einsum("s,ksp->p", pi.astype(numpy.longdouble), wide_root_cl(f)) / f.nCat
    return float((f.counts * numpy.log(like)).sum())


def saturated_tree(dataType, nTax, nPat, nCat, alpha, precision):
    """A balanced tree whose sites, random states mixed into conserved ones by
    a share that grows from 0 to 1 over the patterns, are explained only by
    the fast categories: with a very small alpha the slowest category's rate
    is below 1e-40, so in FP32 its P is the identity and every site that
    varies has likelihood 0 in it."""
    from p4gpu import Data, Part, func
    rng = numpy.random.default_rng(nTax + nPat)
    L = ["t%d:1.0" % i for i in range(nTax)]
    while len(L) > 3:
        L = ["(%s,%s):0.5" % (L[i], L[i + 1]) if i + 1 < len(L) else L[i] for i in range(0, len(L), 2)]
    t = func.readNewick("(%s);" % ",".join(L))
    names = ["t%d" % i for i in range(nTax)]
    t.taxNames = names
    S = 4 if dataType == "dna" else 20
    share = numpy.linspace(0.0, 1.0, nPat)[None, :]
    codes = numpy.where(rng.random((nTax, nPat)) < share, rng.integers(0, S, (nTax, nPat)),
                        rng.integers(0, S, nPat)[None, :])
    t.data = Data(parts=[Part.fromPatterns(codes, rng.integers(1, 9, nPat), dataType)], taxNames=names)
    t.newComp(free=1, spec="specified", val=list(rng.dirichlet(numpy.full(S, 20.0))))
    t.newRMatrix(free=1, spec="specified", val=list(rng.lognormal(0, 0.3, S * (S - 1) // 2)))
    t.setNGammaCat(nGammaCat=nCat)
    t.newGdasrv(free=1, val=alpha)
    t.setPInvar(free=0, val=0.0)
    t.setPrecision(precision)
    return t
