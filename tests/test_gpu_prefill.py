"""Prompt passes (many positions at once) against the same prompt taken one
position a step: the logits of the position after the prompt, from a cache
that the passes filled and from one that the steps filled."""
import threading

import numpy as np
import pytest
import torch

import lutmac_amd as L
import oracle
from conftest import rel_max_err
from lutmac_amd import decode as D

pytestmark = pytest.mark.gpu

# Both forms are fp32 sums of the same terms in other orders; the bound is the
# decoder tests' own against the oracle.
DECODE_TOL = 1e-5


def both(model, batch, prompt):
    """Logits [batch, vocab] after the prompt: passes, then steps."""
    n = prompt.shape[1]
    dec = D.Decoder(model, batch=batch)
    p = prompt if batch > 1 else prompt[0]
    out, _, _ = dec.generate(p, 2)
    vocab = model.cfg.vocab
    a, b = (torch.empty(batch * vocab, device="cuda") for _ in range(2))
    dec.step(a)
    toks = np.asarray(out).reshape(batch, n + 2)
    dec.reset(toks if batch > 1 else toks[0])
    for _ in range(n + 2):
        dec.step(b)
    torch.cuda.synchronize()
    dec.close()
    return a.cpu().numpy().reshape(batch, vocab), b.cpu().numpy().reshape(batch, vocab)


# Prompt lengths: the shortest that takes a pass, one and more 16-row query
# tiles (16 / group positions each), past a 64-position cache chunk, and, with
# 512 rows a pass, several passes; heads with 1, 4 and 6 queries per key head;
# ffn 264 (no whole row tiles per half) leaves SiLU(gate)*up to a kernel of its
# own, there with every family of formats among the linears.
@pytest.mark.parametrize("batch,n", [(1, 5), (1, 17), (1, 130), (3, 65), (16, 70), (1, 700)])
@pytest.mark.parametrize("heads,kv,hd,ffn", [(8, 2, 64, 512), (6, 1, 128, 264), (4, 4, 64, 512)])
def test_prompt_passes(cuda, batch, n, heads, kv, hd, ffn):
    cfg = D.small_config(n_heads=heads, n_kv_heads=kv, head_dim=hd, ffn=ffn, max_seq=n + 4, vocab=515,
                         qkv_bias=kv == 4)
    model = quantized(cfg) if ffn == 264 else D.SyntheticModel(cfg, seed=n + heads, group=128, random_norms=True)
    prompt = np.random.default_rng(n).integers(0, cfg.vocab, (batch, n)).astype(np.int32)
    passes, steps = both(model, batch, prompt)
    for b in range(batch):
        assert rel_max_err(passes[b], steps[b]) < DECODE_TOL, b


def quantized(cfg):
    return D.QuantizedModel(cfg, {"q": (L.FMT_TERNARY, 128, 0), "k": (L.FMT_TERNARY, 128, 0),
                                  "v": (L.FMT_TERNARY, 128, 0), "o": (L.FMT_RRQ2, 128, L.QUANT_RESIDUAL),
                                  "gate": (L.FMT_INT8, 256, 0), "up": (L.FMT_INT8, 256, 0),
                                  "down": (L.FMT_BINARY, 128, 0), "embed": (L.FMT_INT4, 128, 0)}, seed=4)


# Passes without the memory for their rows (for none of them, not for all, not for
# the last) leave the prompt to steps, and nothing behind them: the tokens and the
# logits after it are those of the passes, once there is memory.
@pytest.mark.parametrize("batch,limit", [(1, 0), (1, 150000), (1, 900000), (6, 0), (6, 1000000), (6, 2850000)])
def test_prompt_without_memory_for_passes(cuda, monkeypatch, batch, limit):
    cfg = D.small_config(max_seq=40, vocab=515)
    model = D.SyntheticModel(cfg, seed=2, group=128, random_norms=True)
    prompt = np.random.default_rng(batch).integers(0, cfg.vocab, (batch, 30)).astype(np.int32)
    p = prompt if batch > 1 else prompt[0]
    dec = D.Decoder(model, batch=batch)
    logits = {}
    for name in ("steps", "steps again", "passes"):
        if name == "passes":
            monkeypatch.delenv("LMX_PROMPT_BYTES")
        else:
            monkeypatch.setenv("LMX_PROMPT_BYTES", str(limit))
        out, _, _ = dec.generate(p, 6)
        lg = torch.empty(batch * cfg.vocab, device="cuda")
        dec.step(lg)
        torch.cuda.synchronize()
        logits[name] = out, lg.cpu().numpy().reshape(batch, cfg.vocab)
    dec.close()
    want_out, want = logits["passes"]
    for name in ("steps", "steps again"):
        out, got = logits[name]
        assert np.array_equal(out, want_out)
        for b in range(batch):
            assert rel_max_err(got[b], want[b]) < DECODE_TOL, (name, b)


# Two decoders that share their weights, each in a thread of its own: the passes
# share no scratch or ticket (down, K 4096, is summed over k-slices).
def test_prompt_passes_side_by_side(cuda):
    cfg = D.small_config(max_seq=72, ffn=4096, vocab=515)
    model = D.SyntheticModel(cfg, seed=3, group=128, random_norms=True)
    a, b = D.Decoder(model), D.Decoder(model)
    for i, layer in enumerate(model.layers):
        L.check(L.lib().lmx_decoder_set_layer(b._h, i, *[w.handle for w in a.weights[4 * i:4 * i + 4]],
                                              L._np_ptr(layer["in_norm"]), L._np_ptr(layer["post_norm"]), None))
    rng = np.random.default_rng(4)
    prompts = [rng.integers(0, cfg.vocab, 60).astype(np.int32) for _ in range(2)]

    def logits(dec, prompt, out):
        for _ in range(8):
            tokens, _, _ = dec.generate(prompt, 2)
            lg = torch.empty(cfg.vocab, device="cuda")
            dec.step(lg)
            torch.cuda.synchronize()
            out.append((tokens, lg.cpu().numpy()))

    alone = [[], []]
    for dec, prompt, out in zip((a, b), prompts, alone):
        logits(dec, prompt, out)
    together = [[], []]
    threads = [threading.Thread(target=logits, args=t) for t in zip((a, b), prompts, together)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for want, got in zip(alone, together):
        assert len(got) == 8
        for (wt, wl), (gt, gl) in zip(want, got):
            assert np.array_equal(wt, gt) and np.array_equal(wl.view(np.uint32), gl.view(np.uint32))
    b.close()
    a.close()


# Norm weights that put one channel far above the rest, where the linears have
# code 8 (weight 0): the chunk is multiplied in fp32 by the kernels that norm as
# they split, one launch (1 and 3 sequences, the SiLU pair too), split vectors (6)
# and a pass in the tile form (300 positions of gate|up's 1024 rows).
def far_model(max_seq):
    cfg = D.small_config(n_layers=3, max_seq=max_seq, vocab=515)
    model = D.SyntheticModel(cfg, seed=8, group=128, random_norms=True)

    def zero(entry, k):
        planes = entry[0]
        bit = 1 << (7 - k % 8)
        planes[:3, :, k // 8] &= 255 - bit
        planes[3, :, k // 8] |= bit

    for layer in model.layers:
        for norm, w, k in (("in_norm", "qkv", 5), ("post_norm", "gate_up", 200)):
            layer[norm][k] = 1e6
            zero(layer[w], k)
    model.final_norm[77] = 1e6
    zero(model.head, 77)
    return model


@pytest.mark.parametrize("batch", [1, 3, 6])
def test_far_norm_channel_steps(cuda, batch):
    model = far_model(16)
    vocab = model.cfg.vocab
    toks = np.random.default_rng(batch).integers(0, vocab, (batch, 8)).astype(np.int32)
    dec = D.Decoder(model, batch=batch)
    dec.reset(toks if batch > 1 else toks[0])
    refs = [oracle.OracleDecoder(model) for _ in range(batch)]
    lg = torch.empty(batch * vocab, device="cuda")
    for pos in range(8):
        dec.step(lg)
        got = lg.cpu().numpy().reshape(batch, vocab)
        for b in range(batch):
            assert rel_max_err(got[b], refs[b].step(toks[b, pos], pos)) < DECODE_TOL, (pos, b)
    dec.close()


def test_far_norm_channel_pass(cuda):
    model = far_model(304)
    prompt = np.random.default_rng(5).integers(0, model.cfg.vocab, (1, 300)).astype(np.int32)
    passes, steps = both(model, 1, prompt)
    assert rel_max_err(passes[0], steps[0]) < DECODE_TOL
