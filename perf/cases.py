"""The work whose speed counts: whole calls of the public entry points
(GpuModel.forward_device, GpuModel.dms, GpuDecoder.decode) on the ESM-2
presets, from one peptide and one decode step to a full batch, a long protein
and a mutational scan.

A case is a dict: "kind" (forward, dms, decode, prefill), "model" (an ESM-2
preset), "dtype" (fp32, q8, q4) and its sizes.  Weights are N(0, 0.02) with
unit LayerNorms and biases N(0, 0.02), tokens uniform over the 20 amino acids
between BOS and EOS; weights, tokens and quantized blocks are made here from
the seed, with torch on the GPU.  The activations between the layers travel as
about 22 bits and are summed in FP32, so whole forwards keep a tolerance of
32-bit sums and no single layer needs a case of its own.
"""
import json
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "codon-infer_amd"))
import codon_hip as ch  # noqa: E402

#          dim, hidden, layers, heads
PRESETS = {"8M": (320, 1280, 6, 20), "35M": (480, 1920, 12, 20), "150M": (640, 2560, 30, 20),
           "650M": (1280, 5120, 33, 20), "3B": (2560, 10240, 36, 40)}
VOCAB, MASK = 33, 32
BLOCK_BYTES = {"fp32": 4.0, "q8": 1.125, "q4": 0.625}  # bytes a weight
CANONICAL = [5, 23, 13, 9, 18, 6, 21, 12, 15, 4, 20, 17, 14, 16, 10, 8, 11, 7, 22, 19]  # A C D E ... W Y
FLAGS = {"logits": ch.OUT_LOGITS, "hidden": ch.OUT_HIDDEN, "final_att": ch.OUT_FINAL_ATT,
         "contacts": ch.OUT_CONTACTS, "attn": ch.OUT_ATTN}


def listed():
    return [
        # the peptide of the reference's own latency table: one 41-token sequence, as its forward fills the
        # run state (logits, hidden state, last attention map)
        dict(name="peptide_650m_q8_l41", kind="forward", model="650M", dtype="q8", lens="41", s_max=41,
             outputs="logits,hidden,final_att"),
        # the shortest sequences: eight tokens, where every weight is read for next to no arithmetic
        dict(name="short_650m_q8_l8", kind="forward", model="650M", dtype="q8", lens="8", s_max=8, outputs="logits"),
        # the smallest model in FP32 on one protein, every attention map exported
        dict(name="maps_8m_fp32_l256", kind="forward", model="8M", dtype="fp32", lens="256", s_max=256,
             outputs="logits,attn"),
        # one ordinary protein with contacts, the reference's default call
        dict(name="contacts_650m_q8_l257", kind="forward", model="650M", dtype="q8", lens="257", s_max=257,
             outputs="logits,final_att,contacts"),
        # a small ragged batch of proteins on a mid-sized model
        dict(name="ragged_35m_q8_b8", kind="forward", model="35M", dtype="q8",
             lens="512,131,387,254,449,173,318,505", s_max=512, outputs="logits"),
        # unquantized weights, a few ragged sequences, hidden states as embeddings
        dict(name="embed_150m_fp32_b3", kind="forward", model="150M", dtype="fp32", lens="347,61,190", s_max=347,
             outputs="logits,hidden"),
        # long proteins with contacts
        dict(name="contacts_150m_q4_b4_l1024", kind="forward", model="150M", dtype="q4", lens="1024,1024,1024,1024",
             s_max=1024, outputs="logits,contacts"),
        # one very long protein on the largest model
        dict(name="long_3b_q4_l2048", kind="forward", model="3B", dtype="q4", lens="2048", s_max=2048,
             outputs="logits"),
        # a full batch: the throughput workload
        dict(name="batch_650m_q8_b16_l512", kind="forward", model="650M", dtype="q8", lens=",".join(["512"] * 16),
             s_max=512, outputs="logits,final_att"),
        # the deep mutational scan of a 200-residue protein, masked copies in chunks of 32
        dict(name="dms_650m_q8_n200", kind="dms", model="650M", dtype="q8", n=200, chunk=32),
        # generation: one step of one stream, and of eight streams further on
        dict(name="decode_650m_q4_1", kind="decode", model="650M", dtype="q4", streams=1, pos=280),
        dict(name="decode_650m_q8_8", kind="decode", model="650M", dtype="q8", streams=8, pos=700),
    ]


def draw(rng):
    """One more case: forwards and scans over all models, formats and outputs, decode steps and prompt prefills."""
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["forward"] * 6 + ["dms", "decode", "decode", "prefill"])
    model = rng.choice(["8M", "35M", "150M", "650M", "650M"] + (["3B"] if kind != "dms" else []))
    dtype = rng.choice(["q8", "q8", "q4", "q4", "fp32"] if model != "3B" else ["q8", "q4"])
    if kind == "forward":
        d = PRESETS[model][0]
        most = min(16384, 8192 * 1280 * 33 * 1280 // (d * d * PRESETS[model][2]))  # tokens: the full batch's work
        top = log_int(3, 2048 if model == "3B" else 1024)
        b = min(log_int(1, 24), max(1, most // top))
        lens = [max(3, rng.randint(top // 4, top)) for _ in range(b)] if rng.random() < 0.6 else [max(3, top)] * b
        lens[0] = max(3, top)
        outputs = rng.choice(["logits", "logits,final_att", "logits,hidden", "logits,hidden,final_att",
                              "logits,final_att,contacts"])
        if top - 2 > 1024:
            outputs = outputs.replace(",contacts", "")
        if model == "8M" and b * top * top <= 4 * 256 * 256 and rng.random() < 0.3:
            outputs = "logits,attn"
        return dict(kind=kind, model=model, dtype=dtype, lens=",".join(map(str, lens)), s_max=max(lens),
                    outputs=outputs)
    if kind == "dms":
        return dict(kind=kind, model=model, dtype=dtype, n=log_int(12, 200), chunk=rng.choice([8, 16, 32]))
    if kind == "decode":
        return dict(kind=kind, model=model, dtype=dtype, streams=log_int(1, 32), pos=log_int(2, 900))
    return dict(kind=kind, model=model, dtype=dtype, rows=log_int(2, 600))


def _lens(case):
    return [int(n) for n in case["lens"].split(",")]


# ---- weights and inputs -------------------------------------------------------


def _generator(seed, stream):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1000003 + stream) % (1 << 62))


def _quantize(w, dtype):
    """[n] float32 -> packed blocks of 32 (Q8_0: f32 scale + 32 int8; Q4_0: f32 scale + 16 nibble pairs)."""
    x = w.view(-1, 32)
    if dtype == "q8":
        scale = x.abs().amax(1, keepdim=True) / 127.0
        q = torch.round(x / scale).clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        top = x.gather(1, x.abs().argmax(1, keepdim=True))
        scale = top / -8.0
        n = (torch.round(x / scale) + 8).clamp_(0, 15).to(torch.uint8)
        q = n[:, :16] | (n[:, 16:] << 4)
    return torch.cat([scale.contiguous().view(torch.uint8), q], 1).reshape(-1)


def _dequantize(blocks, dtype):
    """Packed blocks -> float64 values: the quants times their scale, rounded to FP32 as the model defines it."""
    if dtype == "q8":
        b = blocks.view(-1, 36)
        q = b[:, 4:].contiguous().view(torch.int8).to(torch.float32)
    else:
        b = blocks.view(-1, 20)
        q = torch.cat([b[:, 4:] & 15, b[:, 4:] >> 4], 1).to(torch.float32) - 8.0
    return (q * b[:, :4].contiguous().view(torch.float32)).double().reshape(-1)


MATRICES = ("wq", "wk", "wv", "wo", "fc1_weight", "fc2_weight")


def _tensors(case, seed):
    """Every tensor of the model on the GPU, by field name: float32, or packed blocks for the quantized ones."""
    d, f, layers, _ = PRESETS[case["model"]]
    gen = _generator(seed, 1)

    def normal(n):
        return torch.randn(n, generator=gen, device="cuda") * 0.02

    one, zero = (lambda n: torch.ones(n, device="cuda")), (lambda n: torch.zeros(n, device="cuda"))
    sizes = {"wq": d * d, "wk": d * d, "wv": d * d, "wo": d * d, "fc1_weight": f * d, "fc2_weight": d * f}
    t = {"token_embedding_table": normal(VOCAB * d)}
    for name, n in sizes.items():
        parts = [normal(n) if case["dtype"] == "fp32" else _quantize(normal(n), case["dtype"]) for _ in range(layers)]
        t[name] = torch.cat(parts)
    for name, n in (("bq", d), ("bk", d), ("bv", d), ("bo", d), ("fc1_bias", f), ("fc2_bias", d)):
        t[name] = normal(layers * n)
    for name in ("ln_1", "ln_2"):
        t[name + "_weight"], t[name + "_bias"] = one(layers * d), zero(layers * d)
    t["ln_f_weight"], t["ln_f_bias"] = one(d), zero(d)
    t["classifier_weights"] = torch.cat([one(d), zero(d), normal(d * d), normal(d), normal(VOCAB * d), normal(VOCAB)])
    if case["dtype"] == "q8":
        t["token_embedding_table"] = _quantize(t["token_embedding_table"], "q8")
    return t


def _residues(seed, stream, n):
    return (4 + torch.randint(0, 20, (n,), generator=_generator(seed, stream), device="cuda")).cpu().numpy().astype(
        np.int32)


def _sequences(case, seed):
    """The case's token arrays (forward: one a sequence; dms: the protein's residues; decode and prefill: one a stream)."""
    if case["kind"] == "dms":
        return [_residues(seed, 2, case["n"])]
    if case["kind"] == "forward":
        return [np.concatenate([[0], _residues(seed, 2 + i, n - 2), [2]]).astype(np.int32)
                for i, n in enumerate(_lens(case))]
    streams, n = (case["streams"], case["pos"] + 1) if case["kind"] == "decode" else (1, case["rows"])
    return [np.concatenate([[0], _residues(seed, 2 + i, n)])[:n].astype(np.int32) for i in range(streams)]


def _model(case, seed, **reserve):
    classes = {"fp32": ch.EsmWeights, "q8": ch.EsmWeightsQ8, "q4": ch.EsmWeightsQ4}
    config = ch.EsmConfig.by_name(case["model"])
    weights = classes[case["dtype"]](**{k: v.cpu().numpy() for k, v in _tensors(case, seed).items()})
    head = config.contact_head_weights() if "contacts" in case.get("outputs", "") else None
    return ch.GpuModel(config, weights, contact_head=head, **reserve)


def _output_shapes(case):
    d, _, layers, heads = PRESETS[case["model"]]
    b, s = len(_lens(case)), case["s_max"]
    shapes = {"logits": (b, s, VOCAB), "hidden": (b, s, d), "final_att": (b, s, s), "contacts": (b, s - 2, s - 2),
              "attn": (b, layers, heads, s, s)}
    return {name: shapes[name] for name in case["outputs"].split(",")}


def prepare(case, seed):
    """A loaded model with its workspace, and the call's inputs: device tokens and output buffers for a forward, the
    residues for a scan, a decoder whose caches hold each stream's earlier positions for a decode step."""
    seqs = _sequences(case, seed)
    state = {"kind": case["kind"]}
    if case["kind"] == "forward":
        shapes = _output_shapes(case)
        flags = sum(FLAGS[name] for name in shapes)
        state["model"] = _model(case, seed, max_batch=len(seqs), max_len=case["s_max"], outputs=flags | ch.IO_DEVICE)
        tokens = np.zeros((len(seqs), case["s_max"]), np.int32)
        for i, s in enumerate(seqs):
            tokens[i, :len(s)] = s
        state["tokens"] = torch.from_numpy(tokens).cuda()
        state["lens"] = np.array(_lens(case), np.int32)
        state["s_max"], state["flags"] = case["s_max"], flags
        state["out"] = {name: torch.zeros(shape, device="cuda") for name, shape in shapes.items()}
    elif case["kind"] == "dms":
        state["model"] = _model(case, seed, max_batch=case["chunk"], max_len=case["n"] + 2, outputs=ch.OUT_LOGITS)
        state["residues"], state["chunk"] = seqs[0], case["chunk"]
    else:
        state["model"] = _model(case, seed, max_batch=1, max_len=16, outputs=ch.OUT_LOGITS)
        rows = len(seqs[0])
        if case["kind"] == "prefill":
            state["decoder"] = ch.GpuDecoder(state["model"], n_slots=1, max_len=1024, max_rows=rows)
            state["call"] = (np.zeros(rows, np.int32), seqs[0], np.arange(rows, dtype=np.int32))
        else:
            n = len(seqs)
            state["decoder"] = ch.GpuDecoder(state["model"], n_slots=n, max_len=1024, max_rows=max(256, n))
            for slot, s in enumerate(seqs):
                for at in range(0, rows - 1, 256):
                    part = s[at:min(at + 256, rows - 1)]
                    state["decoder"].decode(np.full(len(part), slot), part, at + np.arange(len(part)))
            state["call"] = (np.arange(n, dtype=np.int32), np.array([s[-1] for s in seqs], np.int32),
                             np.full(n, rows - 1, np.int32))
    torch.cuda.synchronize()
    return state


def run(state):
    """One call: a batched forward, a whole scan, a decode step or a prompt's prefill."""
    if state["kind"] == "forward":
        state["model"].forward_device(state["tokens"].data_ptr(), state["lens"], state["s_max"], state["flags"],
                                      {name: t.data_ptr() for name, t in state["out"].items()})
        return state["out"]
    if state["kind"] == "dms":
        deltas, entropy = state["model"].dms(state["residues"], chunk=state["chunk"])
        return {"deltas": deltas, "entropy": entropy}
    return {"logits": state["decoder"].decode(*state["call"])}


def work(case):
    """Weights read once, tokens in and requested outputs out; for a decode step the cached keys and values too."""
    d, f, layers, heads = PRESETS[case["model"]]
    layer, head = 4 * d * d + 2 * d * f, d * d + VOCAB * d
    weights = layers * layer * BLOCK_BYTES[case["dtype"]] + 4.0 * head
    if case["kind"] == "forward":
        lens, outputs = _lens(case), 0.0
        for name, shape in _output_shapes(case).items():
            inner = {"logits": lambda n: n * VOCAB, "hidden": lambda n: n * d, "final_att": lambda n: n * n,
                     "contacts": lambda n: (n - 2) ** 2, "attn": lambda n: layers * heads * n * n}[name]
            outputs += 4.0 * sum(inner(n) for n in lens)
        pairs = sum(n * n for n in lens)
        rows = logit_rows = sum(lens)
        more = outputs + 4.0 * rows
    elif case["kind"] == "dms":
        rows, logit_rows, pairs = case["n"] * (case["n"] + 2), case["n"], case["n"] * (case["n"] + 2) ** 2
        more = 4.0 * case["n"] * 22
    elif case["kind"] == "decode":
        rows = logit_rows = case["streams"]
        pairs = rows * (case["pos"] + 1)
        more = 8.0 * layers * d * pairs + 4.0 * rows * VOCAB
    else:
        rows = logit_rows = case["rows"]
        pairs = rows * (rows + 1) // 2
        more = 8.0 * layers * d * rows + 4.0 * rows * VOCAB
    flops = 2.0 * rows * layers * layer + 4.0 * pairs * d * layers + 2.0 * logit_rows * head
    return {"bytes": weights + more, "flops": flops}


def tolerance(case):
    """FP32 sums of values that carry about 22 bits, through every layer of the model: 1e-7 to 1.3e-6 against
    exact() over the listed and some drawn cases, about four times the largest is stated."""
    return {"rel": 5e-6, "max": 1e-4}


# ---- the same in 64 bits ------------------------------------------------------


def _erf(x):
    # Abramowitz & Stegun 7.1.26, the polynomial that the model's GELU is defined with
    t = 1.0 / (1.0 + 0.3275911 * x.abs())
    poly = ((((1.061405429 * t - 1.453152027) * t + 1.421413741) * t - 0.284496736) * t + 0.254829592) * t
    return torch.sign(x) * (1.0 - poly * torch.exp(-x * x))


def _gelu(x):
    return 0.5 * x * (1.0 + _erf(x / math.sqrt(2.0)))


def _norm(x, w, b):
    mu = x.mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + 1e-5) * w + b


def _rope_tables(n, hd):
    # the angles are FP32 products of the position and an FP32 frequency
    j = np.arange(hd // 2, dtype=np.float32) * np.float32(2) / np.float32(hd)
    freq = np.float32(1) / np.power(np.float32(10000), j)
    angle = (np.arange(n, dtype=np.float32)[:, None] * freq[None, :]).astype(np.float64)
    return torch.from_numpy(np.cos(angle)).cuda(), torch.from_numpy(np.sin(angle)).cuda()


def _rope(x, c, s):  # [B, H, S, hd]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


class _Exact:
    """The encoder in float64 on padded [B, S] token batches, one layer's weights unpacked at a time."""

    def __init__(self, case, seed):
        self.case, self.t = case, _tensors(case, seed)
        self.d, self.f, self.layers, self.heads = PRESETS[case["model"]]

    def matrix(self, name, layer, out_dim, in_dim):
        t = self.t[name].view(self.layers, -1)[layer]
        w = t.double() if self.case["dtype"] == "fp32" else _dequantize(t, self.case["dtype"])
        return w.view(out_dim, in_dim).t().contiguous()

    def vector(self, name, layer, n):
        return self.t[name].view(self.layers, n)[layer].double()

    def embed(self, tokens, lens, causal):
        table = self.t["token_embedding_table"]
        table = (_dequantize(table, "q8") if self.case["dtype"] == "q8" else table.double()).view(VOCAB, self.d).clone()
        table[MASK] = 0.0
        keep = np.float32(1.0) - np.float32(0.12)
        scale = [keep] * len(lens) if causal else [
            keep / (np.float32(1) - np.float32((t[:n] == MASK).sum()) / np.float32(n)) for t, n in zip(tokens, lens)]
        scale = torch.tensor([float(x) for x in scale], dtype=torch.float64, device="cuda")
        return table[torch.from_numpy(tokens).cuda().long()] * scale[:, None, None]

    def __call__(self, tokens, lens, causal=False, on_map=None):
        """[B, S] tokens -> (logits, hidden) float64; on_map(layer, batch, P [H, S, S]) for every attention map."""
        b, s = tokens.shape
        d, f, heads = self.d, self.f, self.heads
        hd = d // heads
        x = self.embed(tokens, lens, causal)
        c, sn = _rope_tables(s, hd)
        at = torch.arange(s, device="cuda")
        for layer in range(self.layers):
            h = _norm(x, self.vector("ln_1_weight", layer, d), self.vector("ln_1_bias", layer, d))
            q, k, v = ((h.view(-1, d) @ self.matrix(w, layer, d, d) + self.vector(bias, layer, d))
                       .view(b, s, heads, hd).transpose(1, 2) for w, bias in (("wq", "bq"), ("wk", "bk"), ("wv", "bv")))
            q, k = _rope(q, c, sn), _rope(k, c, sn)
            o = torch.zeros(b, s, heads, hd, dtype=torch.float64, device="cuda")
            for i, n in enumerate(lens):
                score = q[i].contiguous() @ k[i].transpose(1, 2).contiguous() / math.sqrt(hd)
                hide = (at[None, :] > at[:, None]) if causal else (at >= n)[None, :].expand(s, s)
                p = torch.softmax(score.masked_fill_(hide, float("-inf")), -1)
                if on_map:
                    on_map(layer, i, p)
                o[i] = (p @ v[i].contiguous()).transpose(0, 1)
            x = x + (o.view(-1, d) @ self.matrix("wo", layer, d, d) + self.vector("bo", layer, d)).view(b, s, d)
            h = _norm(x, self.vector("ln_2_weight", layer, d), self.vector("ln_2_bias", layer, d))
            h = _gelu(h.view(-1, d) @ self.matrix("fc1_weight", layer, f, d) + self.vector("fc1_bias", layer, f))
            x = x + (h @ self.matrix("fc2_weight", layer, d, f) + self.vector("fc2_bias", layer, d)).view(b, s, d)
        hidden = _norm(x, self.t["ln_f_weight"].double(), self.t["ln_f_bias"].double())
        w = self.t["classifier_weights"].double()
        ln_w, ln_b, dense, dense_b, dec, dec_b = torch.split(w, [d, d, d * d, d, VOCAB * d, VOCAB])
        h = _gelu(hidden.view(-1, d) @ dense.view(d, d).t().contiguous() + dense_b)
        logits = _norm(h, ln_w, ln_b) @ dec.view(VOCAB, d).t().contiguous() + dec_b
        return logits.view(b, s, VOCAB), hidden


def _contact_head(model):
    with open(os.path.join(os.getcwd(), "codon-infer_amd", "codon_hip", "data", "contact_heads.json")) as f:
        head = json.load(f)[model]
    _, _, layers, heads = PRESETS[model]
    return np.asarray(head["weight"], np.float32).reshape(layers, heads), float(np.float32(head["bias"]))


def exact(case, seed):
    """What run() returns, in float64."""
    net, seqs = _Exact(case, seed), _sequences(case, seed)
    if case["kind"] == "dms":
        return _exact_dms(net, seqs[0])
    if case["kind"] != "forward":
        tokens = np.stack(seqs)
        logits, _ = net(tokens, [tokens.shape[1]] * len(seqs), causal=True)
        return {"logits": logits[0] if case["kind"] == "prefill" else logits[:, -1]}
    lens, layers, heads = _lens(case), net.layers, net.heads
    out = {name: torch.zeros(shape, dtype=torch.float64, device="cuda")
           for name, shape in _output_shapes(case).items()}
    weights, bias = _contact_head(case["model"]) if "contacts" in out else (None, None)
    tokens = np.zeros((len(seqs), case["s_max"]), np.int32)
    for i, t in enumerate(seqs):
        tokens[i, :len(t)] = t

    def on_map(layer, i, p):
        n = lens[i]
        if "attn" in out:
            out["attn"][i, layer, :, :n, :n] = p[:, :n, :n]
        if "final_att" in out and layer == layers - 1:
            out["final_att"][i, :n, :n] = p[:, :n, :n].mean(0)
        if weights is not None:
            for h in range(heads):
                if weights[layer, h] != 0.0 and n > 2:
                    a = p[h, 1:n - 1, 1:n - 1]
                    a = a + a.t()
                    r = a.sum(1)
                    out["contacts"][i, :n - 2, :n - 2] += float(weights[layer, h]) * (a - torch.outer(r, r) / r.sum())

    logits, hidden = net(tokens, lens, on_map=on_map if len(out) > ("hidden" in out) + 1 else None)
    for i, n in enumerate(lens):
        out["logits"][i, :n] = logits[i, :n]
        if "hidden" in out:
            out["hidden"][i, :n] = hidden[i, :n]
        if weights is not None and n > 2:
            z = out["contacts"][i, :n - 2, :n - 2]
            out["contacts"][i, :n - 2, :n - 2] = torch.sigmoid(z + bias)
    return out


def _exact_dms(net, residues):
    n = len(residues)
    wild = np.concatenate([[0], residues, [2]]).astype(np.int32)
    rows = []
    for at in range(0, n, 16):
        here = range(at, min(at + 16, n))
        tokens = np.stack([wild] * len(here))
        for i, p in enumerate(here):
            tokens[i, p + 1] = MASK
        logits, _ = net(tokens, [n + 2] * len(here))
        rows += [logits[i, p + 1, 4:24] for i, p in enumerate(here)]
    lp = torch.log_softmax(torch.stack(rows), -1)
    wt = torch.from_numpy(residues).cuda().long() - 4
    deltas = lp[:, torch.tensor(CANONICAL, device="cuda") - 4] - lp.gather(1, wt[:, None])
    return {"deltas": deltas, "entropy": -(lp.exp() * lp).sum(1)}
