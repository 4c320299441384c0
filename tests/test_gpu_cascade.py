"""Cascades of S-matrices as trees of star products: a work-space limit ("cascade.matrices") splits
them into several trees, chunks of products and batches of projections. The star product is
associative, so every split gives the unlimited result to rounding, and the oracle's slice by slice
(RCWAIntegrator::compute, src/core/RCWAIntegrator.cpp:20-87; RedhefferIntegrator::compute,
src/core/RedhefferIntegrator.cpp:174-314)."""
import numpy as np
import pytest

from oracle import rcwa_oracle as O
from tests import geometries as G
from varrcwa_amd import api
from varrcwa_amd._lib import from_dev_colmajor

pytestmark = pytest.mark.gpu

# Orderings differ by rounding in a chain of at most 13 well-conditioned star products of matrices
# of at most 18 rows: 13 * 18 * 8 products each of about 1e-16, with room for their conditions.
TOL = 1e-11


@pytest.fixture
def limit(ctx):
    def put(n):
        assert ctx.lib.vrc_tune_set(b"cascade.matrices", n) == 0
    yield put
    put(0)


def blocks(it):
    return [it.Tdd(), it.Tuu(), it.Rud(), it.Rdu()]


def dev(a, b):
    return max(np.abs(x - y).max() / np.abs(y).max() for x, y in zip(a, b))


def stack(seed, nlayers):
    rng = np.random.default_rng(seed)
    return dict(lam=0.8 + 0.03 * seed, layers=[G.random_rect_layer(rng, 0.6) for _ in range(nlayers)],
                thickness=[0.05 + 0.01 * j for j in range(nlayers)],
                bottom=([0.0, 0.6], [0.0, 0.6], np.array([[2.1 + 0j]])),
                top=([0.0, 0.6], [0.0, 0.6], np.array([[1.0 + 0j]])))


def oracle_transforms(inst, nx, ny):
    ze = np.concatenate([[0.0], np.cumsum(inst["thickness"])])
    s = O.StackLayerSampler(inst["lam"], nx, ny, inst["layers"], ze, inst["bottom"], inst["top"])
    return O.invariant_transforms(O.rcwa_integrate(s, ze[0], ze[-1], len(inst["layers"]), z_edges=ze))


def test_limit_is_checked(ctx):
    assert ctx.lib.vrc_tune_set(b"cascade.matrices", -1) == -1


@pytest.mark.parametrize("group", [64, 5])
def test_rcwa_trees(ctx, limit, group):
    """13 slices: one tree; trees of 1, 4 and 10 slices with products in chunks of 1 and 2; the same in
    launches of 5 slices (5, 5, 3)."""
    g = G.metasurface(1)
    s = G.gpu_sampler(g, ctx)
    it = api.RCWAIntegrator(g["z0"], g["z1"], s)
    assert ctx.lib.vrc_tune_set(b"rcwa.group", 64) == 0
    it.compute(13)
    ref = blocks(it)
    orc = O.invariant_transforms(O.rcwa_integrate(G.oracle_sampler(g), g["z0"], g["z1"], 13))
    try:
        ctx.lib.vrc_tune_set(b"rcwa.group", group)
        for n in (0, 1, 16, 40, 52):
            limit(n)
            it.compute(13)
            assert dev(blocks(it), ref) < TOL, n
            got = O.invariant_transforms(O.SResult(*blocks(it), it.W0(), it.V0(), it.gam0(), it.W1(), it.V1(),
                                                   it.gam1()))
            assert max(np.abs(got[k] - orc[k]).max() / np.abs(orc[k]).max() for k in got) < 1e-9, n
    finally:
        ctx.lib.vrc_tune_set(b"rcwa.group", 64)


@pytest.mark.parametrize("nlayers", [3, 7, 8])
def test_batch_trees(ctx, limit, nlayers):
    """Three stacks: one tree; trees of 3, 4 and 5 layers with an odd one carried past the products'
    chunks of 2, 3 and 3; layer by layer (limit 1). One stack alone takes a tree as well."""
    nx = ny = 3
    insts = [stack(k, nlayers) for k in range(3)]
    ref = from_dev_colmajor(api.batch_stack_rcwa(ctx, nx, ny, insts)["S"])
    for n in (1, 36, 48, 60):
        limit(n)
        S = from_dev_colmajor(api.batch_stack_rcwa(ctx, nx, ny, insts)["S"])
        assert dev(S, ref) < TOL, n
        one = from_dev_colmajor(api.batch_stack_rcwa(ctx, nx, ny, insts[1:2])["S"])
        assert dev(one, ref[1:2]) < TOL, n
    limit(0)
    out = api.batch_stack_rcwa(ctx, nx, ny, insts, want_bases=True)
    base = {k: from_dev_colmajor(out[k]) for k in ("W0", "V0", "W1", "V1")}
    gam = {k: out[k].cpu().numpy() for k in ("gam0", "gam1")}
    for i, inst in enumerate(insts):
        got = O.invariant_transforms(O.SResult(*ref[i], base["W0"][i], base["V0"][i], gam["gam0"][i], base["W1"][i],
                                               base["V1"][i], gam["gam1"][i]))
        orc = oracle_transforms(inst, nx, ny)
        assert max(np.abs(got[k] - orc[k]).max() / np.abs(orc[k]).max() for k in got) < 1e-9


def test_batch_trees_and_layer_by_layer(ctx):
    """127 stacks cascade as trees, 128 and more layer by layer: the same stacks give the same result."""
    nx = ny = 3
    insts = [stack(k % 5, 5) for k in range(129)]
    few = from_dev_colmajor(api.batch_stack_rcwa(ctx, nx, ny, insts[:5])["S"])
    for count in (127, 128, 129):
        S = from_dev_colmajor(api.batch_stack_rcwa(ctx, nx, ny, insts[:count])["S"])
        for k in range(count):
            assert dev(S[k:k + 1], few[k % 5:k % 5 + 1]) < TOL, (count, k)


@pytest.mark.parametrize("layer_block", [0, 3, 4])
def test_tape_trees(ctx, limit, layer_block):
    """A tape's checkpoints lie between the trees: S and the gradient from trees of 3 and 5 layers and
    layer by layer agree, with blocks of 3 and 4 layers and the whole stack (8) in one."""
    import torch
    nx = ny = 3
    insts = [stack(10 + k, 8) for k in range(2)]
    rng = np.random.default_rng(3)
    bar = torch.from_numpy(rng.standard_normal((2, 4, 18, 18)) + 1j * rng.standard_normal((2, 4, 18, 18))).cuda()
    ref = None
    for n in (1, 24, 40, 0):
        limit(n)
        out = api.batch_stack_rcwa(ctx, nx, ny, insts, tape=True, layer_block=layer_block)
        grad = out["tape"].vjp(bar).cpu().numpy()
        out["tape"].close()
        got = (from_dev_colmajor(out["S"]), grad)
        if ref is None:
            ref = got
        assert dev(got[0], ref[0]) < TOL, n
        assert np.abs(got[1] - ref[1]).max() < 1e-9 * np.abs(ref[1]).max(), n


def test_varrcwa_projection_batches(ctx, limit):
    """Accepted segments projected one, two and three at a time, each batch cascaded onto those before."""
    g = G.metasurface(1)
    s = G.gpu_sampler(g, ctx)
    it = api.RedhefferIntegrator(g["z0"], g["z1"], s)
    it.compute(0, 10, 2e-2)
    ref, tree = blocks(it), it.tree()
    assert len(tree) >= 7
    orc = O.redheffer_integrate(G.oracle_sampler(g), g["z0"], g["z1"], 2e-2)
    assert np.allclose(tree, orc.tree, rtol=0, atol=1e-14)
    want = O.invariant_transforms(orc)
    for n in (1, 48, 72):
        limit(n)
        it.compute(0, 10, 2e-2)
        assert it.tree() == tree
        assert dev(blocks(it), ref) < TOL, n
        got = O.invariant_transforms(O.SResult(*blocks(it), it.W0(), it.V0(), it.gam0(), it.W1(), it.V1(), it.gam1()))
        assert max(np.abs(got[k] - want[k]).max() / np.abs(want[k]).max() for k in got) < 1e-9, n
