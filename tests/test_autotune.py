"""The autotuner's sweep against a context that models a launch on the host:
both calibration runs of a candidate use the items that the whole batch is
run in, candidates that come to the same launch are run once, and the
prediction is that launch's time."""
import types

import pytest

from pyxopto_amd import _native as N
from pyxopto_amd.mcml import autotune


class _Context:
    """Rate and tail of a launch as functions of its real item size."""

    compute_units = 256

    def __init__(self, limit):
        self.limit, self.calls = limit, []

    def _chunk(self, arr, o):
        if o.flags & N.XO_FLAG_WHOLE_CHUNKS:
            return o.chunk
        total = sum(int(a.npackets) for a in arr)
        return min(o.chunk, max(total // self.limit // 64 * 64, 64))

    def batch_chunk(self, arr, o):
        return self._chunk(arr, o)

    def run_batch(self, arr, lut, o, naccum):
        chunk = self._chunk(arr, o)
        packets = sum(int(a.npackets) for a in arr)
        self.calls.append((packets, chunk, o.block))
        return None, types.SimpleNamespace(kernel_ms=self.time(packets, chunk,
                                                               o.block))

    @staticmethod
    def time(packets, chunk, block):
        return packets / (1e6 + 10.0 * chunk + block) + chunk / 1000.0


def _batch(n, packets):
    arr = (N.XoBatchInstance * n)()
    for i in range(n):
        arr[i].npackets = packets + i
    return arr


# packets that keep all of a candidate's chunk, some of it, the least
@pytest.mark.parametrize('n,packets', [(4096, 200_000), (1000, 100_000),
                                       (300, 20_000), (3, 40)])
def test_sweep_runs_the_items_of_the_whole_batch(n, packets):
    ctx, arr = _Context(14336), _batch(n, packets)
    base = N.XoBatchOpts()
    res = autotune.sweep(ctx, arr, None, 1, base)
    shapes = [r[1:4] for r in res]
    assert len(set(shapes)) == len(shapes)
    plain = N.XoBatchOpts()
    want = set()
    for chunk, block, bpc in autotune.CANDIDATES:
        plain.chunk, plain.block = chunk, block
        want.add((ctx._chunk(arr, plain), block, bpc))
    assert set(shapes) == want
    assert len(ctx.calls) == 2 * len(want)
    assert {c[1:] for c in ctx.calls} == {s[:2] for s in shapes}
    total = sum(int(a.npackets) for a in arr)
    for r in res:
        if total > autotune.CALIBRATION_PACKETS:
            assert r[0] == pytest.approx(ctx.time(total, r[1], r[2]),
                                         rel=1e-9)
