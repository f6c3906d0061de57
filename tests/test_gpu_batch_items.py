"""Work items of a batch are queued for all instances of a group in turn:
each packet of each instance must run once, whatever the budgets (none, one
packet, a few, many times the others') and the item size, in the batch, in a
captured plan and alone."""
import numpy as np
import pytest

from pyxopto_amd import _native as N
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


def test_item_size_follows_the_grid():
    """Items of at most the chunk, two for each wave of the grid that these
    options launch, at least 64 packets; the whole chunk if asked for; the
    results are those of any size."""
    insts = [_instance(k, 40000 + k) for k in range(30)]
    b = mbatch.Batch(insts, rnginit=XINIT)
    arr, lut, naccum = b.pack()
    ctx, total = b.context, sum(i.nphotons for i in insts)
    ref, rep = ctx.run_batch(arr, lut, b.opts(), naccum)
    for block, bpc in ((64, 0), (64, 1), (128, 3), (256, 0), (256, 1)):
        for chunk in (50, 2048, 1 << 20):
            print('case', block, bpc, chunk, flush=True)
            o = b.opts(chunk=chunk, block=block, blocks_per_cu=bpc)
            acc, rep = ctx.run_batch(arr, lut, o, naccum)
            np.testing.assert_array_equal(acc, ref)
            waves = int(rep.lanes) // 64
            if bpc:
                assert waves == bpc * block // 64 * ctx.compute_units
            assert ctx.batch_chunk(arr, o) == min(
                chunk, max(total // (2 * waves) // 64 * 64, 64))
            o.flags |= N.XO_FLAG_WHOLE_CHUNKS
            assert ctx.batch_chunk(arr, o) == chunk
            acc, _ = ctx.run_batch(arr, lut, o, naccum)
            np.testing.assert_array_equal(acc, ref)
    with pytest.raises(RuntimeError, match='block must be'):
        ctx.batch_chunk(arr, b.opts(block=96))
    ctx.close()
