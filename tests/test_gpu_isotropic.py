"""Layered runs that hold an isotropic medium (or other phase-function
parameters that the short sampling code does not cover) take a build of
their own: a stack that mixes such a layer with ordinary ones must hold the
oracle's integers in every form of that build, and the hardware arithmetic
the exact one's sums within the noise of the packets."""
import numpy as np
import pytest

from pyxopto_amd import _native as N
from pyxopto_amd.mcml import mc

from helpers import XINIT
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu

F = mc.mcfluence
NPK = 4000


def _packed(kind, method, fluence):
    L, D, P = mc.mclayer, mc.mcdetector, mc.mcpf
    pfs = {'hg': [P.Hg(0.8), P.Hg(0.0), P.Hg(0.9)],
           'mhg': [P.MHg(0.8, 0.9), P.MHg(0.0, 0.5), P.MHg(0.7, 1.0)]}[kind]
    out = lambda n: L.Layer(d=np.inf, n=n, mua=0.0, mus=0.0,  # noqa: E731
                            pf=pfs[1])
    layers = [out(1.0), L.Layer(d=2e-4, n=1.38, mua=300.0, mus=1e4,
                                pf=pfs[0]),
              L.Layer(d=4e-4, n=1.40, mua=200.0, mus=3e3, pf=pfs[1]),
              L.Layer(d=1e-3, n=1.36, mua=800.0, mus=5e3, pf=pfs[2]),
              out(1.45)]
    grid = F.FluenceRz(F.Axis(0.0, 1e-3, 20), F.Axis(0.0, 1e-3, 15)) \
        if fluence else None
    det = D.Detectors(top=D.Radial(D.RadialAxis(0.0, 2e-3, 30)),
                      bottom=D.Total(), specular=D.Total())
    sim = mc.Mc(L.Layers(layers), mc.mcsource.Line(), det, fluence=grid,
                options=[mc.mcoptions.McMethod(method)], rnginit=XINIT)
    cfg, lut, naccum = sim.pack()
    cfg.packet_seed, cfg.first_packet = 0xABCDEF, 0
    return sim, cfg, lut, naccum


@pytest.mark.parametrize('kind', ['hg', 'mhg'])
@pytest.mark.parametrize('method', [0, 1, 2])
@pytest.mark.parametrize('fluence', [False, True])
def test_mixed_stack_matches_the_oracle(kind, method, fluence):
    print('case', kind, method, fluence, flush=True)
    sim, cfg, lut, naccum = _packed(kind, method, fluence)
    x, a = N.init_rng(64, XINIT)
    ref, counts = O.mcml_run(cfg, lut, x, a, NPK, naccum, O.MATH_KERNEL,
                             keyed=True)[:2]
    ctx = sim.context
    for lanes in (64, 0):
        acc, rep = ctx.run_mcml(cfg, lut, NPK, naccum, lanes,
                                N.XO_FLAG_PACKET_KEYED)
        np.testing.assert_array_equal(acc, ref)
        assert int(rep.steps) == int(counts[0])
    t = N.XoTrace()
    t.max_events, t.options, t.plon = 20, N.XO_TRACE_ALL, 1
    got = ctx.run_mcml_trace(cfg, lut, NPK, naccum, t, 0,
                             N.XO_FLAG_PACKET_KEYED)
    x, a = N.init_rng(64, XINIT)
    racc, _, _, rdata, rn = O.mcml_run_trace(
        cfg, lut, x, a, NPK, naccum, t, O.MATH_KERNEL, keyed=True)
    np.testing.assert_array_equal(got[0], racc)
    np.testing.assert_array_equal(got[2], rdata)
    np.testing.assert_array_equal(got[3], rn)
    # hardware arithmetic: the escaped weight of NPK packets, each within
    # [0, 1], differs by no more than six standard errors of two such means
    fast, _ = ctx.run_mcml(cfg, lut, NPK, naccum, 0, N.XO_FLAG_PACKET_KEYED |
                           N.XO_FLAG_FAST_MATH)
    end = cfg.fluence.offset if fluence else naccum
    diff = float(fast[:end].sum()) - float(ref[:end].sum())
    assert abs(diff) / N.XO_ACCU_K / NPK < 6 * np.sqrt(2 * 0.25 / NPK)
