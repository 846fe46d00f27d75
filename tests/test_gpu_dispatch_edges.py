"""Both sides of the lines at which a dispatch changes kernels, at sizes around the kernels' own tiles."""
import numpy as np
import pytest

import layered_common as lc
from layered_common import oracle

pytestmark = pytest.mark.gpu

# f32 sums over at most a few hundred terms, errors of the logits relative to their r.m.s.: the bar of the other f32 tests
F32_TOL = 2e-4


@pytest.fixture
def tune():
    from fandhe_ai_amd.capi import lib
    keys = []

    def set_(key, value):
        keys.append(key)
        assert lib.fa_set_tuning(key, value) == 0

    yield set_
    for key in keys:
        lib.fa_set_tuning(key, 0)


_OPS = []


def ops():
    import fandhe_ai_amd as fa
    if not _OPS:
        _OPS.append(fa.tape_for(fa.Device.Rocm(0)))
    return _OPS[0]


RECURRENCES = {
    "delta": lambda dim, vdim: lc.config([lc.delta(heads=3, kv_heads=1, dim=dim, vdim=vdim)]),
    "channel": lambda dim, vdim: lc.bubetar([lc.parallel_2(right=lc.channel_right(heads=2, kv_heads=1, dim=dim, vdim=vdim))]),
    "lightning": lambda dim, vdim: lc.bubetar([lc.parallel(right=lc.lightning_right(heads=3, dim=dim, vdim=vdim))]),
}


@pytest.mark.parametrize("form", [2, 3], ids=["split", "one wavefront per tile"])
@pytest.mark.parametrize("dim,vdim", [(9, 7), (24, 20), (40, 72), (128, 128), (130, 36)])
@pytest.mark.parametrize("kind", sorted(RECURRENCES))
def test_scan_forms(kind, dim, vdim, form, tune):
    """Sequences around the chunk's 32 tokens in one pass, then more of them behind the states that pass left."""
    tune(31, form)
    cfg = RECURRENCES[kind](dim, vdim)
    w = lc.weights(cfg, 5)
    lens, more = [65, 33, 12, 31, 96], 14
    toks = [lc.tokens(cfg, n + more, 40 + n) for n in lens]
    dec = lc.make_decoder(ops(), cfg, w, max_tokens=1024, max_batch=len(lens))
    table = np.full((len(lens), dec.cfg.max_blocks_per_seq), 0xFFFFFFFF, dtype=np.uint32)
    table[:, :8] = np.arange(8 * len(lens)).reshape(8, len(lens)).T
    dec.set_sequences(table, [0] * len(lens))
    first = dec.forward([t[:n] for t, n in zip(toks, lens)], [list(range(n)) for n in lens])
    second = dec.forward([t[n:] for t, n in zip(toks, lens)], [list(range(more))] * len(lens))
    at = 0
    for b, n in enumerate(lens):
        want = oracle.forward(cfg, w, toks[b])
        got = np.concatenate([first[at:at + n], second[b * more:(b + 1) * more]])
        assert lc.error(got, want) < F32_TOL, (b, n)
        at += n
    dec.close()
