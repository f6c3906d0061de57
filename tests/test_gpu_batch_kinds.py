"""The batch kernel picks its transport rounds per wave by phase-function
kind and falls back to general ones: every instance of a batch that mixes
kinds, parameters at which the short divisions do not hold (g = 0 and tiny
g, index parameters c between 0 and 1), thin and degenerate layers and
finite radii must hold the oracle's integers, alone and mixed."""
import numpy as np
import pytest

from pyxopto_amd import _native as N
from pyxopto_amd.mcml import batch as mbatch
from pyxopto_amd.mcml import mc
from pyxopto_amd.mcbase import pf as hostpf

from helpers import XINIT
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

TABLE = hostpf.MHg(0.8, 0.7).mclut(300)
PFS = {
    'hg': lambda: mc.mcpf.Hg(0.85), 'hg_back': lambda: mc.mcpf.Hg(-0.4),
    'hg_zero': lambda: mc.mcpf.Hg(0.0), 'hg_tiny': lambda: mc.mcpf.Hg(1e-30),
    'hg_one': lambda: mc.mcpf.Hg(1.0), 'mhg': lambda: mc.mcpf.MHg(0.8, 0.7),
    'mhg_zero': lambda: mc.mcpf.MHg(0.0, 0.5),
    'lut': lambda: mc.mcpf.Lut(*TABLE),
    'lut_inside': lambda: mc.mcpf.Lut([0.375, -0.5, 0.25],
                                      np.linspace(-1.0, 1.0, 64)),
}


def _instance(name, k, rmax):
    L, D = mc.mclayer, mc.mcdetector
    pf = PFS[name]()
    layers = [L.Layer(d=np.inf, n=1.0, mua=0.0, mus=0.0, pf=pf),
              L.Layer(d=2e-4, n=1.38, mua=300.0, mus=1e4, pf=pf),
              L.Layer(d=1e-7, n=1.38, mua=300.0, mus=1e4, pf=pf),
              L.Layer(d=1e-3, n=1.45, mua=2000.0, mus=5e3, pf=pf),
              L.Layer(d=np.inf, n=1.0, mua=0.0, mus=0.0, pf=pf)]
    det = D.Detectors(top=D.Radial(D.RadialAxis(0.0, 2e-3, 30)),
                      bottom=D.Total(), specular=D.Total())
    return mbatch.Instance(layers, mc.mcsource.Line(), det,
                           nphotons=700 + 130 * k, seed=99 + k, rmax=rmax)


@pytest.mark.parametrize('method', [0, 1, 2])
@pytest.mark.parametrize('rmax', [float('inf'), 1.5e-3])
def test_kinds_match_the_oracle(method, rmax):
    print('case', method, rmax, flush=True)
    insts = [_instance(n, k, rmax if k % 3 else float('inf'))
             for k, n in enumerate(PFS)]
    opts = [mc.mcoptions.McMethod(method)]
    b = mbatch.Batch(insts, options=opts, rnginit=XINIT)
    packed = b.pack()
    arr, lut, naccum = packed
    ref = O.batch_run(arr, lut, naccum, method=method)[0]
    for chunk, block in ((64, 64), (4096, 256)):
        acc, _ = b.context.run_batch(arr, lut, b.opts(chunk=chunk,
                                                      block=block), naccum)
        for i, name in enumerate(PFS):
            lo, n = arr[i].accum_base, arr[i].accum_count
            np.testing.assert_array_equal(acc[lo:lo + n], ref[lo:lo + n],
                                          err_msg=name)


@pytest.mark.parametrize('name', list(PFS))
@pytest.mark.parametrize('method', [0, 1, 2])
def test_layered_kernel_matches_the_oracle(name, method):
    print('case', name, method, flush=True)
    inst = _instance(name, 0, 1.5e-3)
    sim = mc.Mc(inst.layers, inst.source, inst.detectors,
                options=[mc.mcoptions.McMethod(method)], rnginit=XINIT)
    sim.rmax = inst.rmax
    cfg, lut, naccum = sim.pack()
    cfg.packet_seed, cfg.first_packet = 0x1234567, 0
    x, a = N.init_rng(64, XINIT)
    ref = O.mcml_run(cfg, lut, x, a, 3000, naccum, O.MATH_KERNEL,
                     keyed=True)[0]
    for lanes in (64, 0):
        acc, _ = sim.context.run_mcml(cfg, lut, 3000, naccum, lanes,
                                      N.XO_FLAG_PACKET_KEYED)
        np.testing.assert_array_equal(acc, ref)
