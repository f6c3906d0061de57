"""The fluence bins that the layered and voxel kernels hold in LDS: packet-
keyed runs must give the oracle's integers for every launch shape and for
grids that fit the window, exceed it, are a single bin, lie beside the source
or outside the medium. Small runs over many lanes have small windows or none
(a window pays with four packets per bin); the production shapes (blocks of
1-4 waves per SIMD, two blocks of three each, thousands of bins added up by
every block) run with packets that are absorbed within a few steps."""
import numpy as np
import pytest

from pyxopto_amd import _native as N
from pyxopto_amd import workloads
from pyxopto_amd.mcml import mc
from pyxopto_amd.mcvox import mc as mcvox
from oracle import pyoracle as O

from helpers import XINIT

pytestmark = pytest.mark.gpu

F = mc.mcfluence
A = F.Axis
GRIDS = {
    'rz_fits': lambda: F.FluenceRz(A(0.0, 3e-3, 61), A(0.0, 1.5e-3, 31)),
    'rz_exceeds': lambda: F.FluenceRz(A(0.0, 3e-3, 211), A(0.0, 1.5e-3, 97)),
    'rz_off_axis': lambda: F.FluenceRz(A(0.0, 4e-3, 150), A(0.0, 1.5e-3, 90),
                                       center=(1.1e-3, -0.4e-3)),
    'xyz_odd': lambda: F.Fluence(A(-2e-3, 2e-3, 33), A(-1e-3, 1e-3, 7),
                                 A(0.0, 1.5e-3, 5)),
    'xyz_exceeds': lambda: F.Fluence(A(-2e-3, 2e-3, 41), A(-2e-3, 2e-3, 43),
                                     A(0.0, 1.5e-3, 37)),
    'xyz_beside': lambda: F.Fluence(A(1e-3, 3e-3, 50), A(1e-3, 3e-3, 50),
                                    A(2e-4, 1.5e-3, 30)),
    'xyz_one_bin': lambda: F.Fluence(A(-1e-3, 1e-3, 1), A(-1e-3, 1e-3, 1),
                                     A(0.0, 1e-3, 1)),
    'xyz_empty': lambda: F.Fluence(A(-1e-3, 1e-3, 20), A(-1e-3, 1e-3, 20),
                                   A(2e-3, 3e-3, 20)),
}
# waves per SIMD: a fraction of one, one, three, four, six and more
LANES = [64, 65536, 150000, 262144, 393216, 499999]


@pytest.mark.parametrize('grid', list(GRIDS))
def test_layered_window_matches_the_oracle(grid):
    print('case', grid, flush=True)
    L, D = mc.mclayer, mc.mcdetector
    pf = mc.mcpf.Hg(0.85)
    layers = L.Layers([
        L.Layer(d=np.inf, n=1.0, mua=0.0, mus=0.0, pf=pf),
        L.Layer(d=5e-4, n=1.37, mua=500.0, mus=1.5e4, pf=pf),
        L.Layer(d=1e-3, n=1.40, mua=50.0, mus=2e4, pf=pf),
        L.Layer(d=np.inf, n=1.45, mua=0.0, mus=0.0, pf=pf)])
    sim = mc.Mc(layers, mc.mcsource.Line(),
                D.Detectors(top=D.Radial(D.RadialAxis(0.0, 3e-3, 60))),
                fluence=GRIDS[grid](), rnginit=XINIT)
    cfg, lut, naccum = sim.pack()
    cfg.packet_seed, cfg.first_packet = 0xABCDEF12345, 0
    npk = 6000
    x, a = N.init_rng(1024, XINIT)
    ref, _, _ = O.mcml_run(cfg, lut, x, a, npk, naccum, O.MATH_KERNEL,
                           keyed=True)
    ctx = N.Context(0, 0, XINIT)
    for lanes in LANES + [0]:
        got, _ = ctx.run_mcml(cfg, lut, npk, naccum, lanes,
                              N.XO_FLAG_PACKET_KEYED)
        np.testing.assert_array_equal(got, ref, err_msg=str(lanes))
    fast = [ctx.run_mcml(cfg, lut, npk, naccum, lanes, N.XO_FLAG_PACKET_KEYED |
                         N.XO_FLAG_FAST_MATH)[0] for lanes in LANES + [0]]
    for got in fast[1:]:
        np.testing.assert_array_equal(got, fast[0])
    assert (ref[cfg.fluence.offset:].sum() > 0) == (grid != 'xyz_empty')
    ctx.close()


@pytest.mark.parametrize('n', [5, 24, 50])
def test_voxel_window_matches_the_oracle(n):
    print('case', n, flush=True)
    sim = workloads.skin_two_layer(n=n)
    cfg, lut, naccum = sim.pack()
    cfg.packet_seed, cfg.first_packet = 0xABCDEF12345, 0
    npk = 3000
    x, a = N.init_rng(1024, XINIT)
    ref = O.mcvox_run(cfg, sim.voxels.material, lut, x, a, npk, naccum,
                      O.MATH_KERNEL, keyed=True)[0]
    ctx = N.Context(0, 0, XINIT)
    for lanes in LANES + [0]:
        got, _ = ctx.run_mcvox(cfg, sim.voxels.material, lut, npk, naccum,
                               lanes, N.XO_FLAG_PACKET_KEYED)
        np.testing.assert_array_equal(got, ref, err_msg=str(lanes))
    ctx.close()


# threads per block of these lane counts on 256 CUs: one block per CU of one
# to four waves per SIMD, or two of three each where the registers of the
# build allow six waves
SHAPES = {65536: {256}, 131072: {512}, 196608: {768}, 262144: {1024},
          393216: {768, 1024}, 0: {1024, 768}}


def _production_shapes(ctx, run, ref, nbins, flags, two_blocks):
    """`run` at every shape against `ref`; the windows seen."""
    if ctx.compute_units != 256:
        pytest.skip('shapes of 256 CUs')
    windows, shapes = set(), set()
    for lanes, blocks in SHAPES.items():
        got = run(lanes, N.XO_FLAG_PACKET_KEYED | flags)
        block, nblocks, window = ctx.last_launch()
        print('case', lanes, block, nblocks, window, flush=True)
        np.testing.assert_array_equal(got, ref, err_msg=str(lanes))
        assert block in blocks and nblocks >= 200
        assert window >= min(nbins, 1500)
        windows.add(window)
        shapes.add((block, nblocks > 256))
    assert not two_blocks or (768, True) in shapes
    return windows


@pytest.mark.parametrize('fast', [0, N.XO_FLAG_FAST_MATH])
@pytest.mark.parametrize('grid', ['rz_fits', 'rz_exceeds', 'xyz_exceeds',
                                  'xyz_odd'])
def test_layered_production_shapes(grid, fast):
    print('case', grid, fast, flush=True)
    L, D = mc.mclayer, mc.mcdetector
    pf = mc.mcpf.Hg(0.5)
    layers = L.Layers([
        L.Layer(d=np.inf, n=1.0, mua=0.0, mus=0.0, pf=pf),
        L.Layer(d=3e-4, n=1.37, mua=4e3, mus=3e3, pf=pf),
        L.Layer(d=1e-3, n=1.40, mua=6e3, mus=2e3, pf=pf),
        L.Layer(d=np.inf, n=1.45, mua=0.0, mus=0.0, pf=pf)])
    sim = mc.Mc(layers, mc.mcsource.Line(),
                D.Detectors(top=D.Radial(D.RadialAxis(0.0, 3e-3, 60))),
                fluence=GRIDS[grid](), rnginit=XINIT)
    cfg, lut, naccum = sim.pack()
    cfg.packet_seed, cfg.first_packet = 0xABCDEF12345, 0
    npk = 1_050_000
    x, a = N.init_rng(1024, XINIT)
    ctx = N.Context(0, 0, XINIT)
    if fast:      # one block of one wave: the windows' shapes against it
        ref = ctx.run_mcml(cfg, lut, npk, naccum, 64,
                           N.XO_FLAG_PACKET_KEYED | fast)[0]
    else:
        ref = O.mcml_run(cfg, lut, x, a, npk, naccum, O.MATH_KERNEL,
                         keyed=True)[0]
    F_ = cfg.fluence
    nbins = F_.shape[0] * F_.shape[1] * F_.shape[2]
    windows = _production_shapes(
        ctx, lambda lanes, flags: ctx.run_mcml(cfg, lut, npk, naccum, lanes,
                                               flags)[0],
        ref, nbins, fast, two_blocks=True)
    if nbins <= 8000:
        assert windows == {nbins}
    else:
        assert max(windows) < nbins
    assert ref[F_.offset:].sum() > 0
    ctx.close()


@pytest.mark.parametrize('fast', [0, N.XO_FLAG_FAST_MATH])
@pytest.mark.parametrize('n', [16, 31])
def test_voxel_production_shapes(n, fast):
    print('case', n, fast, flush=True)
    M, G, D = mcvox.mcmaterial, mcvox.mcgeometry, mcvox.mcdetector
    pf = mcvox.mcpf.Hg(0.5)
    materials = M.Materials([
        M.Material(n=1.0, mua=0.0, mus=0.0, pf=pf),
        M.Material(n=1.34, mua=4e3, mus=3e3, pf=pf),
        M.Material(n=1.40, mua=6e3, mus=2e3, pf=pf)])
    ax = G.Axis(-1e-3, 1e-3, n)
    az = G.Axis(0.0, 2e-3, n)
    voxels = G.Voxels(ax, ax, az)
    sim = mcvox.Mc(voxels, materials, mcvox.mcsource.GaussianBeam(2e-4),
                   D.Detectors(top=D.Total()),
                   fluence=mcvox.mcfluence.Fluence(ax, ax, az),
                   rnginit=XINIT)
    voxels.material[:n // 4] = 1
    voxels.material[n // 4:] = 2
    voxels.update()
    cfg, lut, naccum = sim.pack()
    cfg.packet_seed, cfg.first_packet = 0xABCDEF12345, 0
    npk = 1_050_000
    ctx = N.Context(0, 0, XINIT)
    if fast:
        ref = ctx.run_mcvox(cfg, voxels.material, lut, npk, naccum, 64,
                            N.XO_FLAG_PACKET_KEYED | fast)[0]
    else:
        x, a = N.init_rng(1024, XINIT)
        ref = O.mcvox_run(cfg, voxels.material, lut, x, a, npk, naccum,
                          O.MATH_KERNEL, keyed=True)[0]
    windows = _production_shapes(
        ctx, lambda lanes, flags: ctx.run_mcvox(cfg, voxels.material, lut,
                                                npk, naccum, lanes, flags)[0],
        ref, n ** 3, fast, two_blocks=bool(fast))
    assert windows == {n ** 3} if n == 16 else max(windows) < n ** 3
    ctx.close()
