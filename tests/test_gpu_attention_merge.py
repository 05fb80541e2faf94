"""Decode attention whose contexts are split over workgroups: one workspace
shared by calls of different row counts, through the entry point and through
prompts continued past a split context, against fp64 and the oracle's loop.
"""
import numpy as np
import pytest

import jinf_amd
import model_util as mu
import oracle
import testutil as tu
from gpu_util import dev as to_dev
from gpu_util import host, say
from oracle import engine as oeng

pytestmark = pytest.mark.gpu

KV = {"f32": (np.float32, oracle.F32), "f16": (np.float16, oracle.F16)}


def reference(q, k, v, ln, nh, nk, hd):
    """One sequence in fp64: the outputs and sum_t p_t |v_t| ([nh, hd] each)."""
    out, mag = np.empty((nh, hd)), np.empty((nh, hd))
    for h in range(nh):
        j = h // (nh // nk)
        kk = k[:ln, j * hd:(j + 1) * hd].astype(np.float64)
        vv = v[:ln, j * hd:(j + 1) * hd].astype(np.float64)
        z = kk @ q[h * hd:(h + 1) * hd].astype(np.float64) / np.sqrt(hd)
        p = np.exp(z - z.max())
        p /= p.sum()
        out[h], mag[h] = p @ vv, p @ np.abs(vv)
    return out, mag


@pytest.mark.parametrize("kv", list(KV))
@pytest.mark.parametrize("nh,nk,hd,rows", [(32, 8, 128, (10, 14, 3, 15)), (8, 8, 64, (2, 11, 5, 15)),
                                           (16, 2, 128, (40, 63, 1, 20))])
def test_row_counts_share_a_workspace(dev, kv, nh, nk, hd, rows):
    """Calls of growing and shrinking row counts through one workspace, each
    with contexts past a 256-position chunk and few enough pairs to merge in
    the launch (bar of the attention tests: 2e-5 sum_t p_t |v_t|)."""
    r = tu.rng(nh + nk)
    max_ctx = 600
    ws = jinf_amd.attention_workspace(max(rows), nh, hd, max_ctx)
    for n in rows:
        say(f"attention {kv} heads {nh}/{nk} x {hd}: {n} rows in a shared workspace")
        q = tu.normal(r, (n, nh * hd), 0.0, 1.0, np.float32)
        k = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32).astype(KV[kv][0])
        v = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32).astype(KV[kv][0])
        lens = np.random.default_rng(n).integers(257, max_ctx + 1, size=n).astype(np.int32)
        got = host(jinf_amd.attention_decode(to_dev(q), to_dev(k), to_dev(v), to_dev(lens), nh, nk,
                                             workspace=ws))
        for s in range(n):
            ref, mag = reference(q[s], k[s], v[s], lens[s], nh, nk, hd)
            assert np.all(np.abs(got[s].reshape(nh, hd) - ref) <= 2e-5 * mag), (n, s)


@pytest.mark.parametrize("kv", list(KV))
@pytest.mark.parametrize("heads,kv_heads", [(4, 1), (4, 2)])
def test_prompts_continued_past_a_split_context(dev, kv, heads, kv_heads):
    """A 300-token prompt, then prompts of 10, 64 (merged by a launch of its
    own when 64 rows x head groups reach 128), 3 and 40 tokens at its end,
    each a batched step whose contexts are split, through the engine and the
    batch decoder."""
    parts = (300, 10, 64, 3, 40)
    kt = KV[kv][1]
    tol = 1e-4 if kv == "f32" else 4e-4
    hp, W = mu.tiny_model(seed=31 + heads, n_embd=256, n_heads=heads, n_heads_kv=kv_heads,
                          n_vocab=301)
    toks = [int(t) for t in np.random.default_rng(heads).integers(3, 301, size=sum(parts))]
    ref = oeng.Decoder(hp, W, max_context=512, kv_type=kt)
    want = [ref.step(t) for t in toks]
    with jinf_amd.Engine(hp, mu.to_device(W), 512, kt) as e, \
            jinf_amd.Batch(e, 64, 512, kt) as b:
        at = 0
        for n in parts:
            say(f"{n} prompt tokens at {at}, kv {kv}, heads {heads}/{kv_heads}")
            e.prefill(toks[at:at + n])
            b.prefill(3, toks[at:at + n])
            at += n
            w = want[at - 1]
            bar = tol * float(np.max(np.abs(w)))
            assert float(np.max(np.abs(e.logits() - w))) <= bar, n
            assert float(np.max(np.abs(b.logits()[(n - 1) % 64] - w))) <= bar, n
