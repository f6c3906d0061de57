"""The fluence bins that the layered and voxel kernels hold in LDS: packet-
keyed runs must give the oracle's integers for every launch shape (one block
per CU of 1-4 waves per SIMD, two of three each, small blocks) and for grids
that fit the window, exceed it, are a single bin, lie beside the source or
outside the medium."""
import numpy as np
import pytest

from pyxopto_amd import _native as N
from pyxopto_amd import workloads
from pyxopto_amd.mcml import mc
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
