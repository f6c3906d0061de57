"""Work items of a batch are queued for all instances of a group in turn:
each packet of each instance must run once, whatever the budgets (none, one
packet, a few, many times the others') and the item size, in the batch, in a
captured plan and alone."""
import numpy as np
import pytest

from pyxopto_amd.mcml import batch as mbatch
from pyxopto_amd.mcml import mc

from helpers import XINIT

pytestmark = pytest.mark.gpu

BUDGETS = {'one': [1], 'none_among': [0, 5000, 0, 64, 65],
           'uneven': [1, 200001, 63, 4097, 128, 30000],
           'many': [100 + 7 * k for k in range(300)], 'large': [3000001] * 2}


def _instance(k, n):
    L, D = mc.mclayer, mc.mcdetector
    pf = mc.mcpf.Hg(0.5) if k % 3 else mc.mcpf.MHg(0.5, 0.5)
    layers = [L.Layer(d=np.inf, n=1.0, mua=0.0, mus=0.0, pf=pf),
              L.Layer(d=1e-4 * (1 + k % 5), n=1.3, mua=2e3, mus=3e3, pf=pf),
              L.Layer(d=np.inf, n=1.0, mua=0.0, mus=0.0, pf=pf)]
    det = D.Detectors(top=D.Radial(D.RadialAxis(0.0, 1e-3, 5)),
                      bottom=D.Total(), specular=D.Total())
    return mbatch.Instance(layers, mc.mcsource.Line(), det, nphotons=n,
                           seed=11 + k)


@pytest.mark.parametrize('name', list(BUDGETS))
def test_every_packet_runs_once(name):
    insts = [_instance(k, n) for k, n in enumerate(BUDGETS[name])]
    b = mbatch.Batch(insts, rnginit=XINIT)
    arr, lut, naccum = b.pack()
    total = sum(BUDGETS[name])
    # one instance after the other
    ref = np.zeros(naccum, np.uint64)
    for i in range(len(insts)):
        one = (type(arr[0]) * 1)(arr[i])
        ref += b.context.run_batch(one, lut, b.opts(chunk=4096), naccum)[0]
    for chunk in (1, 100, 2048, 1 << 20):
        if total // chunk > 1 << 20:
            continue
        print('case', name, chunk, flush=True)
        acc, rep = b.context.run_batch(arr, lut, b.opts(chunk=chunk), naccum)
        assert int(rep.packets) == total
        np.testing.assert_array_equal(acc, ref)
    acc, rep = b.context.batch_plan(arr, lut, b.opts(), naccum).run()
    assert int(rep.packets) == total
    np.testing.assert_array_equal(acc, ref)
    b.context.close()
