"""fp32-cache decode attention over its work-item shapes: query heads per
workgroup, head sizes, tile and chunk edges, contexts split (merged in the
launch and by a second one) or whole, against the oracle.

Bar: |out - ref| <= 2e-5 sum_t p_t |v_t| per element, the attention tests'.
Positions at or past a length are NaN, so reading one fails.
"""
import numpy as np
import pytest
import torch

import jinf_amd
import oracle
import testutil as tu
from gpu_util import dev as to_dev
from gpu_util import host, say

pytestmark = pytest.mark.gpu


def run(hd, nh, nk, lens, max_ctx, ws, seed):
    r = tu.rng(seed)
    n = len(lens)
    q = tu.normal(r, (n, nh * hd), 0.0, 1.0, np.float32)
    k = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32)
    v = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32)
    for s, ln in enumerate(lens):
        k[s, ln:] = np.nan
        v[s, ln:] = np.nan
    w = jinf_amd.attention_workspace(n, nh, hd, max_ctx) if ws else None
    L = to_dev(np.asarray(lens, np.int32))
    args = (to_dev(q), to_dev(k), to_dev(v), L, nh, nk)
    got = host(jinf_amd.attention_decode(*args, workspace=w))
    again = host(jinf_amd.attention_decode(*args, workspace=w))
    assert tu.bits_equal(got, again)  # the merge counters are back at zero
    for s, ln in enumerate(lens):
        for h in range(nh):
            o = got[s, h * hd:(h + 1) * hd]
            if ln == 0:
                assert np.all(o == 0.0)
                continue
            j = h // (nh // nk)
            kk = k[s, :ln, j * hd:(j + 1) * hd].astype(np.float64)
            vv = v[s, :ln, j * hd:(j + 1) * hd].astype(np.float64)
            z = kk @ q[s, h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
            p = np.exp(z - z.max())
            p /= p.sum()
            err = np.abs(o - p @ vv)
            assert np.all(err <= 2e-5 * (p @ np.abs(vv))), (s, h, ln, float(err.max()))


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("nh,nk", [(2, 2), (4, 2), (8, 2), (16, 2), (12, 2), (10, 2)])
def test_tile_and_chunk_edges(hd, nh, nk):
    say(f"fp32 attention hd={hd} heads={nh}/{nk}")
    lens = [0, 1, 15, 16, 17, 127, 128, 129, 255, 256, 257, 300, 512, 513, 700]
    run(hd, nh, nk, lens, 700, True, 3)
    run(hd, nh, nk, lens, 700, False, 4)


@pytest.mark.parametrize("hd,n,nh,nk", [(64, 70, 16, 2), (128, 40, 8, 4), (128, 1, 32, 8)])
def test_many_sequences(hd, n, nh, nk):
    """Enough (sequence, head group) pairs for the merge launch, and one."""
    say(f"fp32 attention n={n} hd={hd} heads={nh}/{nk}")
    lens = [int(x) for x in np.random.default_rng(n).integers(0, 1101, size=n)]
    lens[0] = 1100
    run(hd, nh, nk, lens, 1100, True, n)
