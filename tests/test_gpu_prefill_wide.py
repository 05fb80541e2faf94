"""Prompts longer than a batched step (the wide path: matrix products over
128-token tiles, attention over tiles of rows) against the oracle's
token-by-token loop.

Bars as for the engine's other paths, relative to the logit scale: 1e-4 with
an fp32 cache (fp32 sums), 4e-4 with an fp16 cache (a cached value may round
to its other fp16 neighbour).
"""
import threading

import numpy as np
import pytest
import torch

import jinf_amd
import model_util as mu
import oracle
from oracle import engine as oeng

pytestmark = pytest.mark.gpu

F32, F16 = oracle.F32, oracle.F16
Q4_0, Q8_0, Q4_K, Q6_K = oracle.Q4_0, oracle.Q8_0, oracle.Q4_K, oracle.Q6_K
MATS = ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")


def tokens(n, vocab, seed):
    return [int(x) for x in np.random.default_rng(seed).integers(3, vocab, size=n)]


def check(got, want, kv, what):
    err = float(np.max(np.abs(got.astype(np.float64) - want)))
    bar = (4e-4 if kv == F16 else 1e-4) * float(np.max(np.abs(want)))
    assert err <= bar, f"{what}: {err:.3e} > {bar:.3e}"


def decode(ref, toks):
    for t in toks:
        out = ref.step(t)
    return out


# One token past a batched step, the edges of a 128-token tile and of its
# 32-token parts; every weight format alone and mixed within a layer; each
# head size the attention kernel takes and one it does not.
@pytest.mark.parametrize("n,types,heads,kv", [
    (65, Q4_0, (8, 2), F16),
    (127, Q8_0, (4, 4), F16),
    (128, Q4_K, (8, 1), F32),
    (129, Q6_K, (8, 4), F16),
    (161, mu.MIXED, (4, 2), F16),
    (300, mu.MIXED, (16, 2), F32),
])
def test_engine_prefill(n, types, heads, kv):
    t = types if isinstance(types, dict) else {m: types for m in MATS}
    hp, W = mu.tiny_model(seed=n, n_embd=512, n_heads=heads[0], n_heads_kv=heads[1], n_ff=768,
                          n_vocab=301, types=t)
    toks = tokens(n + 3, 301, n)
    ref = oeng.Decoder(hp, W, max_context=n + 8, kv_type=kv)
    with jinf_amd.Engine(hp, mu.to_device(W), n + 8, kv) as e:
        e.prefill(toks[:n])
        check(e.logits(), decode(ref, toks[:n]), kv, f"prompt of {n}")
        assert e.n_past == n
        # the cache rows and the position: decoding goes on from there
        e.forward(toks[n:])
        check(e.logits(), decode(ref, toks[n:]), kv, "after the prompt")


# The x preparation holds a row in 1, 2, 4, 8 or 16 groups of 8 columns a
# thread (2048 columns each): both sides of every step, with a norm (n_embd)
# and without (n_ff), the last one the widest row taken.
@pytest.mark.parametrize("n_embd,heads,n_ff", [
    (256, (4, 2), 2048), (256, (4, 2), 2304), (256, (4, 2), 4352), (256, (4, 2), 8448),
    (256, (4, 2), 16640), (256, (4, 2), 32768), (2304, (18, 2), 512), (4352, (34, 2), 512),
])
def test_row_widths(n_embd, heads, n_ff):
    hp, W = mu.tiny_model(seed=n_ff + n_embd, n_layers=1, n_embd=n_embd, n_heads=heads[0],
                          n_heads_kv=heads[1], n_ff=n_ff, n_vocab=301,
                          types=dict.fromkeys(MATS, Q4_K))
    toks = tokens(67, 301, n_ff)
    ref = oeng.Decoder(hp, W, max_context=80, kv_type=F32)
    with jinf_amd.Engine(hp, mu.to_device(W), 80, F32) as e:
        e.prefill(toks)
        check(e.logits(), decode(ref, toks), F32, f"{n_embd} / {n_ff}")


def test_whole_rounds_and_a_split_tail():
    """A gate / up product of 300 tiles: one round of 256 and 44 split in two."""
    hp, W = mu.tiny_model(seed=15, n_layers=1, n_embd=512, n_heads=8, n_heads_kv=2, n_ff=12800,
                          n_vocab=301, types=dict.fromkeys(MATS, Q4_0))
    toks = tokens(260, 301, 15)
    ref = oeng.Decoder(hp, W, max_context=272, kv_type=F16)
    with jinf_amd.Engine(hp, mu.to_device(W), 272, F16) as e:
        e.prefill(toks)
        check(e.logits(), decode(ref, toks), F16, "260 tokens")


def test_wide_rows_against_batched_steps():
    """Residual adds of 264 tiles (one round, 8 split) and Q / K / V of 280 (24
    split), 8448 columns: the logits of a 1000-token prompt against the same
    prompt in batched steps of 50."""
    hp, W = mu.tiny_model(seed=16, n_layers=1, n_embd=256, n_heads=2, n_heads_kv=2, n_ff=512,
                          n_vocab=301)
    n, kvd, ff = 8448, 256, 512
    hp.update(n_embd=n, n_heads=66, n_heads_kv=2)
    r = np.random.default_rng(16)

    def q4_0(rows, cols, rms):
        b = r.integers(0, 256, size=(rows, cols // 32, 18), dtype=np.uint8)
        d = (r.uniform(0.5, 1.5, size=(rows, cols // 32)) * rms / 4.6).astype(np.float16)
        b[:, :, :2] = d[..., None].view(np.uint8)
        return b.reshape(rows, -1), Q4_0

    W = {"token_embd.weight": q4_0(301, n, 1.0), "output.weight": q4_0(301, n, n ** -0.5),
         "output_norm.weight": (mu.norm_weight(1, n, F32), F32)}
    for name, rows, cols in (("attn_q", n, n), ("attn_k", kvd, n), ("attn_v", kvd, n),
                             ("attn_output", n, n), ("ffn_gate", ff, n), ("ffn_up", ff, n),
                             ("ffn_down", n, ff)):
        W[f"blk.0.{name}.weight"] = q4_0(rows, cols, cols ** -0.5)
    for name in ("attn_norm", "ffn_norm"):
        W[f"blk.0.{name}.weight"] = (mu.norm_weight(2, n, F32), F32)
    toks = tokens(1000, 301, 16)
    with jinf_amd.Engine(hp, mu.to_device(W), 8, F16) as e, jinf_amd.Batch(e, 50, 1000, F16) as b:
        b.prefill(0, toks)
        got = b.logits()
        for c in range(0, 1000, 50):
            b.prefill(1, toks[c:c + 50])
        check(got, b.logits().astype(np.float64), F16, "rows 950 .. 999")


def test_two_chunks_and_a_later_prompt():
    """A prompt of two wide chunks, then another at a position inside the
    context (an attention tile starting past its first row)."""
    hp, W = mu.tiny_model(seed=5, n_layers=1, n_vocab=301)
    toks = tokens(1250, 301, 5)
    ref = oeng.Decoder(hp, W, max_context=1300, kv_type=F16)
    with jinf_amd.Engine(hp, mu.to_device(W), 1300, F16) as e:
        e.prefill(toks[:1100])
        check(e.logits(), decode(ref, toks[:1100]), F16, "1100 tokens")
        e.prefill(toks[1100:])
        check(e.logits(), decode(ref, toks[1100:]), F16, "150 more")


@pytest.mark.parametrize("kv", [F16, F32], ids=["f16", "f32"])
@pytest.mark.parametrize("n_embd,heads", [(256, (4, 2)), (256, (2, 1)), (768, (6, 2))])
def test_prompts_deep_in_a_context(n_embd, heads, kv):
    """Prompts whose contexts the attention splits: 600 tokens (short rows
    written directly, long ones merged), then 65, 130 and 200 at its end, and
    2 tokens in a batch of one sequence; one, two and three query heads per
    kv head, head sizes 64 and 128."""
    hp, W = mu.tiny_model(seed=n_embd + heads[1], n_layers=1, n_embd=n_embd, n_heads=heads[0],
                          n_heads_kv=heads[1], n_vocab=301)
    parts = (600, 65, 130, 200, 2)
    toks = tokens(sum(parts), 301, heads[0])
    ref = oeng.Decoder(hp, W, max_context=1024, kv_type=kv)
    want = [ref.step(t) for t in toks]
    with jinf_amd.Engine(hp, mu.to_device(W), 1024, kv) as e, jinf_amd.Batch(e, 1, 1024, kv) as b:
        at = 0
        for n in parts:
            e.prefill(toks[at:at + n])
            b.prefill(0, toks[at:at + n])
            at += n
            check(e.logits(), want[at - 1], kv, f"engine, {n} tokens")
            check(b.logits()[0], want[at - 1], kv, f"batch, {n} tokens")


@pytest.mark.parametrize("n_seq,n", [(1, 40), (3, 131), (50, 120)])
def test_batch_prefill_logits_rows(n_seq, n):
    """The batch's rows after a wide prompt: the last chunk of n_seq tokens'
    logits at rows 0 .. (n - 1) % n_seq, and no other sequence touched."""
    hp, W = mu.tiny_model(seed=9, n_vocab=301)
    toks = tokens(n, 301, n)
    ref = oeng.Decoder(hp, W, max_context=160, kv_type=F16)
    want = [ref.step(t) for t in toks]
    with jinf_amd.Engine(hp, mu.to_device(W), 8, F16) as e, \
            jinf_amd.Batch(e, n_seq, 160, F16) as b:
        other = (n_seq - 1) if n_seq > 1 else None
        if other is not None:
            b.prefill(other, toks[:2])
        b.prefill(0, toks)
        rows = (n - 1) % n_seq + 1
        got = b.logits()
        for i in range(rows):
            check(got[i], want[n - rows + i], F16, f"row {i}")
        assert b.n_past(0) == n
        if other is not None:
            assert b.n_past(other) == 2
            r2 = oeng.Decoder(hp, W, max_context=160, kv_type=F16)
            for t in toks[:2]:
                r2.step(t)
            step = [-1] * n_seq
            step[other] = toks[2]
            b.forward(step)
            check(b.logits()[other], r2.step(toks[2]), F16, "the other sequence")


def test_nonfinite_token_leaves_earlier_rows_alone():
    """A token whose K and V rows are not finite changes no earlier token's
    logits (their attention does not reach it); its own are NaN."""
    hp, W = mu.tiny_model(seed=11, n_vocab=301, embd_type=F32)
    n, n_seq, at = 40, 16, 37
    toks = tokens(n, 300, 11)
    toks[at] = 300
    for value in (np.nan, np.inf):
        W["token_embd.weight"][0][300] = 0.0
        W["token_embd.weight"][0][300, 5] = value
        ref = oeng.Decoder(hp, W, max_context=64, kv_type=F16)
        want = [ref.step(t) for t in toks[:at]]
        with jinf_amd.Engine(hp, mu.to_device(W), 8, F16) as e, \
                jinf_amd.Batch(e, n_seq, 64, F16) as b:
            b.prefill(0, toks)
            got = b.logits()
            first = n - 8  # rows 0 .. 7 are tokens 32 .. 39
            for i in range(8):
                if first + i < at:
                    check(got[i], want[first + i], F16, f"row {i}")
                elif first + i == at:
                    assert np.all(np.isnan(got[i])), f"row {i}"


def test_nonfinite_keys_with_finite_values():
    """NaN weights in one kv head's K projection (V finite): every query head
    of that group reads NaN scores, so every logit is NaN, as in a batched
    step and in the oracle's loop."""
    hp, W = mu.tiny_model(seed=12, n_vocab=301, types=dict.fromkeys(MATS, Q8_0))
    hd = hp["n_embd"] // hp["n_heads"]
    wk = W["blk.0.attn_k.weight"][0]
    wk[hd + 3, 0:2] = np.frombuffer(np.float16(np.nan).tobytes(), np.uint8)
    toks = tokens(40, 301, 12)
    ref = oeng.Decoder(hp, W, max_context=64, kv_type=F16)
    assert np.all(np.isnan(decode(ref, toks)))
    for n_seq in (16, 40):  # wide; one batched step
        with jinf_amd.Engine(hp, mu.to_device(W), 8, F16) as e, \
                jinf_amd.Batch(e, n_seq, 64, F16) as b:
            b.prefill(0, toks)
            rows = (len(toks) - 1) % n_seq + 1
            assert np.all(np.isnan(b.logits()[:rows])), n_seq


@pytest.mark.parametrize("qt", [Q4_0, Q8_0], ids=["q4_0", "q8_0"])
def test_small_columns_beside_large_ones(qt):
    """One 256-column slab of the down projection's input 2^26 times the rest,
    against zero weights: the other columns keep their 22 bits (each slab is
    split under a scale of its own).  Bar 2^-18 of the logit scale, four bits
    for the sums; under one scale per row the columns keep 14 bits."""
    hp, W = mu.tiny_model(seed=14, n_layers=1, n_embd=256, n_ff=2048, n_vocab=301,
                          types=dict.fromkeys(MATS, qt))
    bs = {Q4_0: 18, Q8_0: 34}[qt]
    up = W["blk.0.ffn_up.weight"][0].reshape(2048, 256 // 32, bs)
    d = np.ascontiguousarray(up[:256, :, :2]).view(np.float16).astype(np.float32)
    up[:256, :, :2] = (d * 2.0 ** 26 / 2.0 ** 10).astype(np.float16).view(np.uint8)
    gate = W["blk.0.ffn_gate.weight"][0].reshape(2048, 256 // 32, bs)
    d = np.ascontiguousarray(gate[:256, :, :2]).view(np.float16).astype(np.float32)
    gate[:256, :, :2] = (d * 2.0 ** 10).astype(np.float16).view(np.uint8)
    W["blk.0.ffn_down.weight"][0].reshape(256, 2048 // 32, bs)[:, :8, :2] = 0
    toks = tokens(72, 301, 14)
    ref = oeng.Decoder(hp, W, max_context=80, kv_type=F32)
    want = decode(ref, toks)
    with jinf_amd.Engine(hp, mu.to_device(W), 80, F32) as e:
        e.prefill(toks)
        err = float(np.max(np.abs(e.logits().astype(np.float64) - want)))
    print(f"error / scale {err / np.max(np.abs(want)):.2e}", flush=True)
    assert err <= 2.0 ** -18 * float(np.max(np.abs(want)))


@pytest.mark.parametrize("mode", ["thread_local", "relaxed"])
def test_first_wide_prompt_beside_a_capture(mode):
    """The first wide prompt (which allocates) in one thread while another
    captures a graph: both succeed, and the graph replays.  (Beside a capture
    of the global mode no prompt succeeds: the call waits for its stream.)"""
    hp, W = mu.tiny_model(seed=13, n_vocab=301)
    toks = np.asarray(tokens(100, 301, 13), np.int32)
    ref = oeng.Decoder(hp, W, max_context=128, kv_type=F16)
    want = decode(ref, [int(t) for t in toks])
    with jinf_amd.Engine(hp, mu.to_device(W), 8, F16) as e, \
            jinf_amd.Batch(e, 8, 128, F16) as b:
        x = torch.arange(64, device="cuda", dtype=torch.float32)
        y = torch.zeros_like(x)
        torch.cuda.synchronize()
        rc = []
        prompt = threading.Thread(target=lambda: rc.append(
            jinf_amd.lib().jinf_hip_batch_prefill(b._h, 0, toks.ctypes.data, toks.size, None)))
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, capture_error_mode=mode):
            y.add_(x)
            prompt.start()
            prompt.join()
            y.add_(1.0)
        assert rc == [0]
        for k in range(3):
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, (k + 1) * (x + 1.0))
        check(b.logits()[(toks.size - 1) % 8], want, F16, "prompt beside a capture")
