"""Decode attention whose contexts are split over workgroups: one workspace
shared by calls of different row counts, through the entry point and through
prompts continued past a split context, and non-finite scores inside a
context, whole or split, against fp64 and the oracle's loop.
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


# ---- non-finite values inside a context ----

def check_rows(got, want, mag, what):
    """NaN where the fp64 result is NaN, the usual bar elsewhere."""
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan), what
    assert np.all(np.abs(got - want)[~nan] <= 2e-5 * mag[~nan]), what


def reference_nonfinite(q, k, v, ln, nh, nk, hd):
    """reference() where scores may be NaN or infinite: one NaN or +inf score
    makes the whole row's softmax NaN, -inf ones weigh nothing unless all are."""
    with np.errstate(invalid="ignore"):
        return reference(q, k, v, ln, nh, nk, hd)


@pytest.mark.parametrize("split", [False, True], ids=["whole", "split"])
@pytest.mark.parametrize("many", [False, True], ids=["few", "many"])
@pytest.mark.parametrize("kv", list(KV))
def test_nan_scores_give_nan(dev, kv, many, split):
    """A NaN in one key (in the first, a middle and the last chunk), in every
    key of one chunk, and in q: NaN for the heads that read it, whether the
    context is whole, merged in the launch or merged by a launch of its own;
    the other rows and heads keep their values."""
    nh, nk, hd, max_ctx = 8, 2, 64, 700
    n = 70 if many else 6
    r = tu.rng(77)
    q = tu.normal(r, (n, nh * hd), 0.0, 1.0, np.float32)
    k = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32).astype(KV[kv][0])
    v = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32).astype(KV[kv][0])
    lens = np.full(n, max_ctx, np.int32)
    lens[5] = 0
    k[0, 3, 5] = np.nan            # kv head 0, first chunk
    k[1, 300, hd + 5] = np.nan     # kv head 1, second chunk
    k[2, 699, 5] = np.nan          # last position
    k[3, 256:512, hd:] = np.nan    # every key of a chunk
    q[4, 2 * hd + 1] = np.nan      # query head 2
    say(f"attention {kv}, NaN scores, {n} sequences, split {split}")
    ws = jinf_amd.attention_workspace(n, nh, hd, max_ctx) if split else None
    args = (to_dev(q), to_dev(k), to_dev(v), to_dev(lens), nh, nk)
    for _ in range(2):
        got = host(jinf_amd.attention_decode(*args, workspace=ws)).reshape(n, nh, hd)
        assert np.all(got[5] == 0.0)
        for s in [0, 1, 2, 3, 4] + ([n - 1] if many else []):
            want, mag = reference_nonfinite(q[s], k[s], v[s], lens[s], nh, nk, hd)
            check_rows(got[s], want, mag, s)


@pytest.mark.parametrize("split", [False, True], ids=["whole", "split"])
def test_infinite_scores_fp32(dev, split):
    """Infinite keys in an fp32 cache: a +inf score gives NaN, -inf scores
    weigh nothing, also when they fill whole tiles, a whole chunk or all but
    one position; all of them -inf give NaN."""
    nh, nk, hd, max_ctx, n = 4, 1, 64, 700, 6
    r = tu.rng(78)
    q = np.abs(tu.normal(r, (n, nh * hd), 0.0, 1.0, np.float32)) + 0.01
    k = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32)
    v = tu.normal(r, (n, max_ctx, nk * hd), 0.0, 1.0, np.float32)
    lens = np.full(n, max_ctx, np.int32)
    k[0, 40, 7] = np.inf
    k[1, 32:64, 7] = -np.inf
    k[2, 0:512, 7] = -np.inf
    k[3, :, 7] = -np.inf
    k[3, 650, 7] = 1.0
    k[4, :, 7] = -np.inf
    say(f"attention f32, infinite scores, split {split}")
    ws = jinf_amd.attention_workspace(n, nh, hd, max_ctx) if split else None
    got = host(jinf_amd.attention_decode(to_dev(q), to_dev(k), to_dev(v), to_dev(lens), nh, nk,
                                         workspace=ws)).reshape(n, nh, hd)
    for s in range(n):
        want, mag = reference_nonfinite(q[s], k[s], v[s], lens[s], nh, nk, hd)
        check_rows(got[s], want, mag, s)
