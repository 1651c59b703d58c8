"""The GEMM of a few dozen rows (9 to 64 tokens of one forward, 9 and more rows of a decode call) against the oracle
and against the routes it replaces (CIH_GEMM_ROWS=0), at the edges of its 16-row groups, of the row ranges in which it
runs, and of the 16-, 32- and 64-column workgroups, for every weight format and splits of the residual projections."""
import numpy as np
import pytest

import codon_hip as ch
import cpu_ref as cr
from test_gpu_forward import check_argmax, quantized, rand_tokens

pytestmark = pytest.mark.gpu


# K of 96 to 2560 (short last k-chunks), N down to 96 columns (no whole 64-column workgroup: 96, 480, 1440)
@pytest.mark.parametrize("d,F,H", [(96, 160, 4), (480, 1920, 20), (640, 2560, 20)])
@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("tokens", [9, 16, 17, 32, 33, 48, 49, 64, 65])
def test_forward_of_a_few_dozen_tokens(d, F, H, dtype, tokens, monkeypatch):
    """Logits and hidden states of one sequence or three against the oracle (1e-3, the forward's tolerance, which
    random models of this size meet a hundred times over) and against the other GEMMs: the same products in FP32
    sums of another order, 1e-5 of the largest value (a few thousand additions of 2^-24 each, as random walks)."""
    cfg = ch.EsmConfig(d, F, 2, H)
    w = quantized(ch.EsmWeights.random(cfg, seed=d + dtype, std=0.03, bias_std=0.02), dtype)
    rng = np.random.default_rng(tokens)
    lens = [tokens] if tokens % 2 else [tokens - 5, 3, 2]
    seqs = [rand_tokens(rng, n - 2) for n in lens]
    flags = ch.OUT_LOGITS | ch.OUT_HIDDEN
    got = []
    for env in (None, "0"):
        if env:
            monkeypatch.setenv("CIH_GEMM_ROWS", env)
        m = ch.GpuModel(cfg, w, max_batch=len(seqs), max_len=max(lens), outputs=flags)
        got.append(m.forward(seqs, flags))
        m.close()
    for b, toks in enumerate(seqs):
        ref = cr.forward(cfg, w, toks, 4)
        for k in ("logits", "hidden"):
            a, o = got[0][k][b, :len(toks)], got[1][k][b, :len(toks)]
            r = ref[k].reshape(a.shape)
            assert np.abs(a - r).max() <= 1e-3
            assert np.abs(a - o).max() <= 1e-5 * max(1.0, np.abs(o).max())
        check_argmax(got[0]["logits"][b, :len(toks)], ref["logits"], f"T={tokens}")


@pytest.mark.parametrize("rows", [9, 16, 31, 50])
@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_decode_rows_on_limbs(rows, dtype):
    """A prompt prefilled in one call of `rows` rows, then one step of `rows` streams at once, against the oracle's
    one-token forwards (1e-3)."""
    cfg = ch.EsmConfig(480, 1920, 2, 20, max_seq_len=64)
    w = quantized(ch.EsmWeights.random(cfg, seed=rows, std=0.03, bias_std=0.02), dtype)
    toks = rand_tokens(np.random.default_rng(rows), rows - 1)[:rows]
    m = ch.GpuModel(cfg, w, max_batch=1, max_len=16)
    dec = ch.GpuDecoder(m, n_slots=rows, max_len=64, max_rows=rows)
    got = dec.decode(np.zeros(rows), toks, np.arange(rows))
    rs = cr.RunState(cfg, w, max_len=64, num_threads=4)
    for p in range(rows):
        assert np.abs(got[p] - rs.step(int(toks[p]), p)).max() <= 1e-3, p
    dec.reset()
    first = dec.decode(np.arange(rows), toks, np.zeros(rows))
    for s in range(0, rows, 5):
        alone = cr.RunState(cfg, w, max_len=64, num_threads=4)
        assert np.abs(first[s] - alone.step(int(toks[s]), 0)).max() <= 1e-3, s
    dec.close()
    m.close()
