"""Performance cases of the library: the calls that a decoding program makes, one dict a case.

Tensors come from torch.  torch is imported before the library, so that both use the HIP runtime that is loaded first
(they ask for it under one soname) and torch's device memory is the library's.
"""

import math
import os
import shutil
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "faie2-flashnext_amd"))
import fn  # noqa: E402
import model_synth  # noqa: E402

HD = 256           # head dimension of the attention layers
DK = 128           # head dimension of the DeltaNet layers
IXD = 128          # indexer dimension; 4 indexer heads, blocks of 4 keys
NROT, THETA, EPS = 64, 1e7, 1e-6
DEV = "cuda"

# weight formats by GGUF id: values and bytes per block, byte offsets of the fp16 scales in a block, and the root mean
# square of a value whose scales are 1 and whose other bytes are random
Q8_0, Q4_K, Q5_K, Q6_K, IQ4_NL, IQ3_S, IQ4_XS, BF16 = 8, 12, 13, 14, 20, 21, 23, 30
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q5_K: (256, 176), Q6_K: (256, 210), IQ4_NL: (32, 18), IQ3_S: (256, 110),
         IQ4_XS: (256, 136), BF16: (1, 2)}
SCALES = {Q8_0: [0], Q4_K: [0, 2], Q5_K: [0, 2], Q6_K: [208], IQ4_NL: [0], IQ3_S: [0], IQ4_XS: [0]}
RMS = {Q8_0: 73.9, IQ4_NL: 67.4, IQ4_XS: 67.4 * 18.5, IQ3_S: 18.5 * 7.6, Q6_K: 73.9 * 18.5, Q4_K: 36.5 * 8.8,
       Q5_K: 36.5 * 18.0}
IQ4_LEVELS = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]

# the projections that read one activation row, as the reference model's layers have them: (format, rows)
GROUPS = {
    "deltanet": [(IQ4_XS, 10240), (Q6_K, 6144), (BF16, 96)],
    "deltanet0": [(IQ4_XS, 10240), (IQ3_S, 6144), (BF16, 96)],
    "attention": [(IQ4_XS, 12288), (IQ4_XS, 512), (Q6_K, 512), (BF16, 640)],
    "ffn": [(BF16, 513), (IQ4_XS, 640), (IQ3_S, 640)],
}

# A model of the reference's widths and formats with one period of its layers (three DeltaNet, one attention) and
# small n-gram tables, so that its file is about 2 GB.
MODEL_DIMS = dict(model_synth.REFERENCE_DIMS, NL=4,
                  ple_sizes=[2003, 2011, 2017, 2027, 2029, 2039, 2053, 2063, 2069, 2081, 2083, 2087, 2089, 2099, 2111, 2113])
MODEL_CTX = 512

_fn = None
_loaded = {}


def lib():
    global _fn
    if _fn is None:
        torch.cuda.init()
        _fn = fn.FN()
    return _fn


def listed():
    return [
        # a DeltaNet layer of one sequence with its projections, one token: the decode latency of a single user,
        # replayed from a graph as an engine does
        dict(name="deltanet_layer_b1", kind="layer", nt=1, hidden=2560, nkh=16, nvh=48),
        # the fused DeltaNet block of a full batch, one token a sequence: the headline decode step
        dict(name="gdn_b64", kind="gdn", B=64, nt=1, nkh=16, nvh=32, head_map=0, gate_act=0),
        # a speculative verify step of a full batch: 4 drafted tokens, up to 4 accepted ones committed
        dict(name="gdn_verify_b64_nt4", kind="verify", B=64, nt=4, rnt=4, nkh=16, nvh=32, head_map=0, gate_act=0),
        # dense attention decode, one user and a short context: the smallest attention call
        dict(name="attn_b1_4k", kind="attn", B=1, ctx=4096, nt=1, nq=16, nkv=2, ragged=0.0),
        # dense attention decode, a batch of long contexts of different lengths
        dict(name="attn_b16_32k", kind="attn", B=16, ctx=32768, nt=1, nq=16, nkv=2, ragged=0.5),
        # the attention layers of a verify step (or a chunk of a prompt) over a long-context batch
        dict(name="attn_b16_32k_nt8", kind="attn", B=16, ctx=32768, nt=8, nq=16, nkv=2, ragged=0.0),
        # sparse attention of one user at 32K keys with the reference model's heads
        dict(name="qsa_b1_32k", kind="qsa", B=1, ctx=32767, nt=1, nq=24, nkv=2, ragged=0.0),
        # sparse attention, several tokens of a few users: a verify step or a prompt chunk
        dict(name="qsa_b4_16k_nt4", kind="qsa", B=4, ctx=16384, nt=4, nq=24, nkv=2, ragged=0.3),
        # the attention layer's projections for a verify step or a prompt chunk of 8 tokens
        dict(name="proj_attention_nt8", kind="group", group="attention", cols=2560, nt=8),
        # the output projection of a DeltaNet layer, a few drafted tokens
        dict(name="out_q8_0_nt3", kind="gemv", type=Q8_0, rows=2560, cols=6144, nt=3),
        # the LM head of the reference model, one token: the largest single weight of a decode step
        dict(name="lm_head_q5_k", kind="gemv", type=Q5_K, rows=248320, cols=2560, nt=1),
        # a short completion with the whole forward: a prompt in calls of at most 8 tokens, then one-token calls
        dict(name="model_21_plus_4", kind="model", prompt=21, decode=4),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "gdn", "verify", "attn", "attn", "qsa", "gemv", "gemv", "group", "model"])
    if kind == "layer":
        return dict(kind=kind, nt=rng.randint(1, 8), hidden=256 * rng.randint(4, 12), nkh=16, nvh=rng.choice([32, 48]))
    if kind in ("gdn", "verify"):
        c = dict(kind=kind, B=_log(rng, 1, 80), nt=rng.choice([1, 1, 2, 3, 4, 5, 8]), nkh=16, nvh=rng.choice([16, 32, 48]),
                 head_map=rng.randint(0, 1), gate_act=rng.randint(0, 1))
        return dict(c, rnt=rng.randint(1, 5)) if kind == "verify" else c
    if kind in ("attn", "qsa"):
        B = _log(rng, 1, 64)
        ctx = _log(rng, 130, min(131072, 500000 // B))
        return dict(kind=kind, B=B, ctx=ctx, nt=rng.choice([1, 1, 2, 3, 4, 6, 8]) if kind == "attn" else
                    rng.choice([1, 1, 1, 2, 4]), nq=rng.choice([16, 24, 8]), nkv=2, ragged=rng.choice([0.0, 0.3, 0.6]))
    if kind == "gemv":
        ty = rng.choice([Q8_0, Q4_K, Q5_K, Q6_K, IQ4_NL, IQ4_XS, BF16])
        return dict(kind=kind, type=ty, rows=_log(rng, 90, 60000), cols=256 * _log(rng, 2, 32), nt=rng.randint(1, 8))
    if kind == "group":
        return dict(kind=kind, group=rng.choice(sorted(GROUPS)), cols=256 * rng.randint(4, 12), nt=rng.randint(1, 8))
    return dict(kind="model", prompt=rng.randint(1, 30), decode=rng.randint(1, 5))


# ---- inputs ----

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _n(g, *shape, mean=0.0, std=1.0):
    t = torch.randn(shape, generator=g, device=DEV)
    return t if mean == 0.0 and std == 1.0 else t * std + mean


def _raw(g, ty, rows, cols):
    """GGUF bytes of a rows x cols weight: random codes, values of spread about 1 / sqrt(cols)."""
    if ty == BF16:
        return _n(g, rows, cols, std=cols ** -0.5).to(torch.bfloat16).view(torch.uint8).reshape(rows, cols * 2)
    qk, bb = BLOCK[ty]
    blk = torch.randint(0, 256, (rows * (cols // qk), bb), generator=g, device=DEV, dtype=torch.uint8)
    for o in SCALES[ty]:
        s = (torch.rand(blk.shape[0], 1, generator=g, device=DEV) + 0.5) * (cols ** -0.5 / RMS[ty])
        blk[:, o:o + 2] = s.to(torch.float16).view(torch.uint8)
    return blk.reshape(rows, cols // qk * bb)


def _pack(ty, raw, rows, cols):
    L = lib()
    p = torch.empty(L.gemv_packed_bytes(ty, rows, cols), dtype=torch.uint8, device=DEV)
    L.gemv_pack_dev(ty, raw.data_ptr(), rows, cols, p.data_ptr())
    torch.cuda.synchronize()
    return p


def _positions(c):
    """Tokens already in each sequence's cache: the last new token of the longest sits at ctx - 1."""
    return [max(0, c["ctx"] - c["nt"] - int(c["ragged"] * c["ctx"] * b / max(1, c["B"]))) for b in range(c["B"])]


def _i32(v):
    return torch.tensor(v, dtype=torch.int32, device=DEV)


def _gdn_inputs(c, seed):
    g = _gen(seed)
    B, nt, nkh, nvh = c["B"], c["nt"], c["nkh"], c["nvh"]
    C = 2 * nkh * DK + nvh * DK
    rnt = c.get("rnt", 0)
    ring = 4
    while ring < max(nt, rnt) + 3:
        ring *= 2
    s = dict(ring=ring, conv_w=_n(g, C, 4, std=0.3), ssm_a=-torch.exp(_n(g, nvh, std=0.5)), dt_bias=_n(g, nvh, std=0.5),
             norm_w=_n(g, DK, mean=1.0, std=0.1), S=_n(g, B, nvh, DK, DK, std=0.05), conv=_n(g, B, ring, C),
             qkv=_n(g, B, nt, C), ab=_n(g, B, nt, 2 * nvh), z=_n(g, B, nt, nvh * DK),
             pos=torch.randint(16, 4000, (B,), generator=g, device=DEV, dtype=torch.int32),
             out=torch.empty(B, nt, nvh * DK, device=DEV))
    if rnt:
        s.update(rqkv=_n(g, B, rnt, C), rab=_n(g, B, rnt, 2 * nvh),
                 kr=torch.randint(0, rnt + 1, (B,), generator=g, device=DEV, dtype=torch.int32))
    return s


def _attn_inputs(c, seed):
    g = _gen(seed)
    B, nt, nq, nkv = c["B"], c["nt"], c["nq"], c["nkv"]
    step = 256 if c["kind"] == "qsa" else 64
    T = (max(_positions(c)) + nt + step - 1) // step * step
    s = dict(T=T, pos=_i32(_positions(c)), qg=_n(g, B, nt, nq, 2, HD), k=_n(g, B, nt, nkv, HD), v=_n(g, B, nt, nkv, HD),
             wq=_n(g, HD, mean=1.0, std=0.1), wk=_n(g, HD, mean=1.0, std=0.1),
             Kc=_n(g, B, nkv, T // 64, HD // 4, 64, 4), Vc=_n(g, B, nkv, T, HD), og=torch.empty(B, nt, nq, HD, device=DEV))
    if c["kind"] == "qsa":
        s.update(iqk=_n(g, B, nt, 5 * IXD), wqn=_n(g, IXD, mean=1.0, std=0.1), wkn=_n(g, IXD, mean=1.0, std=0.1),
                 IKc=_n(g, B, T, IXD), BKc=torch.zeros(B, T // 256, IXD // 4, 64, 4, device=DEV))
    return s


def _parts(c):
    if c["kind"] == "group":
        return GROUPS[c["group"]]
    if c["kind"] == "layer":
        C = 2 * c["nkh"] * DK + c["nvh"] * DK
        return [(IQ4_XS, C), (Q6_K, c["nvh"] * DK), (BF16, 2 * c["nvh"])]
    return [(c["type"], c["rows"])]


def _weights(c, seed):
    """Raw GGUF weights and the activation rows x [nt][cols]."""
    g = _gen(seed)
    cols = c["hidden"] if c["kind"] == "layer" else c["cols"]
    w = [(ty, rows, cols, _raw(g, ty, rows, cols)) for ty, rows in _parts(c)]
    if c["kind"] == "layer":
        w.append((Q8_0, cols, c["nvh"] * DK, _raw(g, Q8_0, cols, c["nvh"] * DK)))
    return w, _n(g, c["nt"], cols)


def _model():
    """The one model that a program keeps loaded."""
    if "model" not in _loaded:
        base = "/dev/shm" if os.path.isdir("/dev/shm") and shutil.disk_usage("/dev/shm").free > 8 << 30 else None
        d = tempfile.mkdtemp(prefix="fn_model_", dir=base)
        try:
            path = os.path.join(d, "model.gguf")
            model_synth.write_model(path, MODEL_DIMS, seed=7, fast=True)
            lib().load(path, "", max_ctx=MODEL_CTX)
        finally:
            shutil.rmtree(d, ignore_errors=True)
        _loaded["model"] = True


def prepare(case, seed):
    c, L, kind = case, lib(), case["kind"]
    s = dict(case=c)
    if kind in ("gdn", "verify"):
        s.update(_gdn_inputs(c, seed))
    elif kind in ("attn", "qsa"):
        s.update(_attn_inputs(c, seed))
        B, nt, nq, nkv = c["B"], c["nt"], c["nq"], c["nkv"]
        if kind == "attn":
            s["nsplit"] = L.attn_nsplit(B, nkv, nt, c["ctx"])
            wb = L.attn_work_bytes(B, nq, nt, s["nsplit"])
        else:
            s["nsplit"] = L.attn_nsplit(B, nkv, nt, 4 * 512 + 4)
            wb = L.attn_qsa_work_bytes(B, nq, nt, s["nsplit"], s["T"], 512)
            done = min(_positions(c)) // 4
            for j0, j1, b0, b1 in [(0, done, 0, B)] + [(done, p // 4, b, b + 1) for b, p in enumerate(_positions(c))]:
                if j1 > j0:
                    L.ix_blocks_dev(b1 - b0, s["T"], j0, j1, s["IKc"][b0].data_ptr(), s["wkn"].data_ptr(),
                                    s["BKc"][b0].data_ptr())
        s["work"], s["wb"] = torch.empty(max(wb, 16), dtype=torch.uint8, device=DEV), wb
    elif kind == "model":
        _model()
        r = np.random.default_rng(seed)
        s["tokens"] = r.integers(0, MODEL_DIMS["VOCAB"], size=c["prompt"] + c["decode"]).astype(np.int32)
    else:
        w, x = _weights(c, seed)
        s["x"], s["w"] = x, [(ty, rows, cols, _pack(ty, raw, rows, cols)) for ty, rows, cols, raw in w]
        s["y"] = [torch.empty(c["nt"], rows, device=DEV) for _, rows, _, _ in w]
        wbs = [L.gemv_work_bytes(ty, rows, cols, c["nt"]) for ty, rows, cols, _ in w]
        s["work"] = torch.empty(max(wbs + [16]), dtype=torch.uint8, device=DEV)
        if kind == "layer":
            s["block"] = _gdn_inputs(dict(c, B=1), seed + 1)
            s["graph"] = torch.cuda.CUDAGraph()
            _layer(s, 0, dry=True)
            torch.cuda.synchronize()
            with torch.cuda.graph(s["graph"]):
                _layer(s, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return s


def _p(*tensors):
    return [t.data_ptr() for t in tensors]


def _layer(s, stream, dry=False):
    """The projections, the block and the output projection of one layer on `stream` (dry: the projections only, which
    change no state)."""
    c, L, b, w, y = s["case"], lib(), s["block"], s["w"], s["y"]
    ty, rows, cols, pk = zip(*w)
    L.gemv_group_dev(ty[:3], rows[:3], cols[0], _p(*pk[:3]), s["x"].data_ptr(), c["nt"], _p(*y[:3]), stream)
    if not dry:
        L.gdn_block_dev(1, c["nkh"], c["nvh"], c["nt"], b["ring"], *_p(b["pos"], y[0], b["conv_w"], b["conv"], y[2],
                        b["dt_bias"], b["ssm_a"], b["S"], y[1], b["norm_w"], b["out"]), stream=stream)
    L.gemv_dev(ty[3], pk[3].data_ptr(), rows[3], cols[3], b["out"].data_ptr(), c["nt"], y[3].data_ptr(),
               s["work"].data_ptr(), s["work"].numel(), stream)


def run(s):
    c, L = s["case"], lib()
    kind = c["kind"]
    if kind == "gdn":
        L.gdn_block_dev(c["B"], c["nkh"], c["nvh"], c["nt"], s["ring"], *_p(s["pos"], s["qkv"], s["conv_w"], s["conv"],
                        s["ab"], s["dt_bias"], s["ssm_a"], s["S"], s["z"], s["norm_w"], s["out"]),
                        head_map=c["head_map"], gate_act=c["gate_act"])
        return [s["out"], s["S"], s["conv"]]
    if kind == "verify":
        L.gdn_verify_dev(c["B"], c["nkh"], c["nvh"], c["nt"], s["ring"], *_p(s["pos"], s["kr"]), c["rnt"],
                         *_p(s["rqkv"], s["rab"], s["qkv"], s["conv_w"], s["conv"], s["ab"], s["dt_bias"], s["ssm_a"],
                             s["S"], s["z"], s["norm_w"], s["out"]), head_map=c["head_map"], gate_act=c["gate_act"])
        return [s["out"], s["S"], s["conv"]]
    if kind == "attn":
        L.attn_dev(c["B"], c["nq"], c["nkv"], c["nt"], s["T"], *_p(s["pos"], s["qg"], s["k"], s["v"], s["wq"], s["wk"],
                   s["Kc"], s["Vc"]), s["nsplit"], s["work"].data_ptr(), s["wb"], s["og"].data_ptr())
        return [s["og"], s["Kc"], s["Vc"]]
    if kind == "qsa":
        L.attn_qsa_dev(c["B"], c["nq"], c["nkv"], c["nt"], s["T"], *_p(s["pos"], s["qg"], s["k"], s["v"], s["wq"],
                       s["wk"], s["Kc"], s["Vc"], s["iqk"], s["wqn"], s["wkn"], s["IKc"], s["BKc"]), 512, s["nsplit"],
                       s["work"].data_ptr(), s["wb"], s["og"].data_ptr())
        return [s["og"], s["Kc"], s["Vc"], s["IKc"], s["BKc"]]
    if kind == "gemv":
        ty, rows, cols, pk = s["w"][0]
        L.gemv_dev(ty, pk.data_ptr(), rows, cols, s["x"].data_ptr(), c["nt"], s["y"][0].data_ptr(),
                   s["work"].data_ptr(), s["work"].numel())
        return s["y"]
    if kind == "group":
        ty, rows, cols, pk = zip(*s["w"])
        L.gemv_group_dev(ty, rows, cols[0], _p(*pk), s["x"].data_ptr(), c["nt"], _p(*s["y"]))
        return s["y"]
    if kind == "layer":
        s["graph"].replay()
        return [s["y"][3], s["block"]["S"], s["block"]["conv"]]
    # the whole model: the prompt, then one token a call; logits at the end of the prompt and of the last call
    t, n, out = s["tokens"], c["prompt"], []
    L.reset()
    for i in range(0, n - 1, 8):
        out.append(L.forward(t[i:min(i + 8, n - 1)]))
    am, first = L.forward(t[n - 1:n], logits=True)
    out.append(am)
    for i in range(n, n + c["decode"] - 1):
        out.append(L.forward(t[i:i + 1]))
    am, last = L.forward(t[n + c["decode"] - 1:], logits=True)
    return [np.concatenate(out + [am]), first, last]


# ---- the work a pass cannot do without ----

def _row_bytes(ty, cols):
    qk, bb = BLOCK[ty]
    return cols // qk * bb


def work(case):
    c, kind = case, case["kind"]
    nt = c.get("nt", 1)
    if kind in ("gdn", "verify", "layer"):
        B, nkh, nvh, rnt = c.get("B", 1), c["nkh"], c["nvh"], c.get("rnt", 0)
        C = 2 * nkh * DK + nvh * DK
        kr = rnt / 2
        b = B * 4 * (2 * nvh * DK * DK + 3 * C + min(3, kr if rnt else nt) * C + (nt + kr) * (C + 2 * nvh) +
                     2 * nt * nvh * DK) + 4 * (4 * C + DK + 2 * nvh)
        f = B * (nt + kr) * nvh * DK * DK * 8
        if kind != "layer":
            return dict(bytes=b, flops=f)
        w = _parts(c) + [(Q8_0, c["hidden"])]
        cols = [c["hidden"]] * 3 + [nvh * DK]
        b += sum(r * _row_bytes(ty, n) for (ty, r), n in zip(w, cols)) + 4 * nt * 2 * c["hidden"]
        return dict(bytes=b, flops=f + sum(2 * nt * r * n for (_, r), n in zip(w, cols)))
    if kind in ("attn", "qsa"):
        nq, nkv, B = c["nq"], c["nkv"], c["B"]
        b = B * nt * 4 * HD * (3 * nq + 4 * nkv)
        f = 0
        for p in _positions(c):
            # keys a query attends: all of them, or the best 512 blocks of 4 and the incomplete block.  Several
            # queries of a sequence may attend different blocks; those of one query are counted for the bytes.
            def keys(n):
                return 2048 + n % 4 if kind == "qsa" and n // 4 > 512 else n
            b += 4 * 2 * nkv * HD * keys(p + nt)
            f += sum(4 * nq * HD * keys(p + t + 1) for t in range(nt))
            if kind == "qsa":
                b += 4 * IXD * ((p + nt) // 4 + 7 * nt) if (p + nt) // 4 > 512 else 4 * IXD * 7 * nt
                f += sum(8 * IXD * ((p + t + 1) // 4) for t in range(nt))
        return dict(bytes=b, flops=f)
    if kind in ("gemv", "group"):
        p, cols = _parts(c), c["cols"]
        return dict(bytes=sum(r * _row_bytes(ty, cols) for ty, r in p) + 4 * nt * (cols + sum(r for _, r in p)),
                    flops=sum(2 * nt * r * cols for _, r in p))
    # the model: the weights of every call once (of the routed experts those that its tokens pick), by format
    m, by = MODEL_DIMS, lambda ty, r, n: r * model_synth.BLOCK[ty][1] * n // model_synth.BLOCK[ty][0]  # noqa: E731
    T, D, HCD = model_synth.TYPES, m["D"], m["HC"] * m["D"]
    n0 = c["prompt"] - 1
    calls = [min(8, n0 - i) for i in range(0, n0, 8)] + [1] * (1 + c["decode"])
    b = f = 0
    for n in calls:
        picked = m["NE"] * (1 - (1 - m["NEU"] / m["NE"]) ** n)
        per = by(T["output"], m["VOCAB"], D) + 2 * by(BF16, m["HCR"], HCD) + by(T["ple"], HCD + D, D)
        vals = m["VOCAB"] * D + 2 * m["HCR"] * HCD + (HCD + D) * D
        for il in range(m["NL"]):
            per += 4 * by(BF16, m["HCR"], HCD) + by(BF16, m["NE"] + 1, D)
            vals += 4 * m["HCR"] * HCD + (m["NE"] + 1) * D
            mix = ([(T["attn_q"], m["NH"] * 2 * HD, D), (T["attn_k"], m["NKV"] * HD, D), (T["attn_v"], m["NKV"] * HD, D),
                    (T["attn_output"], D, m["NH"] * HD), (BF16, 5 * IXD, D)] if (il + 1) % 4 == 0 else
                   [(T["attn_qkv"], 2 * m["NKH"] * DK + m["NVH"] * DK, D),
                    (model_synth.pick(T["attn_gate"], il), m["NVH"] * DK, D), (BF16, 2 * m["NVH"], D),
                    (T["ssm_out"], D, m["NVH"] * DK)])
            mix += [(T["shexp_gate"], m["FFS"], D), (T["shexp_up"], m["FFS"], D), (T["shexp_down"], D, m["FFS"])]
            per += sum(by(*w) for w in mix) + (0 if (il + 1) % 4 == 0 else 2 * 4 * m["NVH"] * DK * DK)
            vals += sum(r * k for _, r, k in mix)
            exps = [(model_synth.pick(T["exps_gate"], il), m["FFE"], D), (model_synth.pick(T["exps_up"], il), m["FFE"], D),
                    (model_synth.pick(T["exps_down"], il), D, m["FFE"])]
            per += int(picked * sum(by(*w) for w in exps))
            vals += m["NEU"] * sum(r * k for _, r, k in exps)
        b += per
        f += 2 * n * vals
    return dict(bytes=b, flops=f)


# About four times what the path shows against the same step in 64 bits (see exact): sums in 32 bits.  The model has no
# such value; its layers' differences add up over four layers and the LM head.
TOLERANCE = {"layer": 1e-6, "gdn": 1e-6, "verify": 1e-6, "attn": 4e-6, "qsa": 1.5e-6, "gemv": 1e-6, "group": 1e-6,
             "model": 1e-5}


def tolerance(case):
    rel = TOLERANCE[case["kind"]]
    return dict(rel=rel, max=20 * rel)


# ---- the same step in 64 bits ----

def _silu(x):
    return x * torch.sigmoid(x)


def _gdn_exact(c, s, qkv, ab, z):
    """One block over the case's tokens: (out, S, conv) as the call leaves them."""
    B, nt, nkh, nvh, ring = c.get("B", 1), c["nt"], c["nkh"], c["nvh"], s["ring"]
    w, S, conv = s["conv_w"].double(), s["S"].double(), s["conv"].double()
    heads = torch.arange(nvh, device=DEV)
    heads = heads // (nvh // nkh) if c.get("head_map", 0) else heads % nkh
    pos, rnt = s["pos"].long(), c.get("rnt", 0)
    at = torch.arange(B, device=DEV)
    kr = s["kr"].long() if rnt else torch.zeros(B, dtype=torch.long, device=DEV)
    hist = [conv[at, (pos - kr - d) % ring] for d in (3, 2, 1)]  # the raw inputs before the first token, oldest first

    def token(S, hist, x, a, on):
        """The state after raw input x with logits a, where `on`; and the token's readout."""
        y = _silu(sum(h * w[:, j] for j, h in enumerate(hist + [x])))
        q = y[:, :nkh * DK].reshape(B, nkh, DK)
        k = y[:, nkh * DK:2 * nkh * DK].reshape(B, nkh, DK)
        v = y[:, 2 * nkh * DK:].reshape(B, nvh, DK)
        q, k = (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6) for t in (q, k))
        q, k = q[:, heads], k[:, heads]
        g = torch.exp(torch.nn.functional.softplus(a[:, :nvh] + s["dt_bias"].double()) * s["ssm_a"].double())[..., None]
        beta = torch.sigmoid(a[:, nvh:])[..., None]
        delta = (v - g * (S * k[..., None]).sum(2)) * beta
        S2 = S * g[..., None] + k[..., None] * delta[:, :, None, :]
        o = (S2 * q[..., None]).sum(2) / math.sqrt(DK)
        m = on.reshape(B, 1, 1, 1)
        keep = on.reshape(B, 1)
        return torch.where(m, S2, S), [torch.where(keep, n, h) for n, h in zip(hist[1:] + [x], hist)], o

    for i in range(rnt):  # the accepted tokens of the call before are the first kr of its rnt
        x = s["rqkv"][:, i].double()
        on = i < kr
        S, hist, _ = token(S, hist, x, s["rab"][:, i].double(), on)
        for b in range(B):
            n = int(kr[b])
            if i < n and i >= n - 3:
                conv[b, int(pos[b] - n + i) % ring] = x[b]
    kept, outs = S, []
    for t in range(nt):
        x = qkv[:, t].double()
        S, hist, o = token(S, hist, x, ab[:, t].double(), torch.ones(B, dtype=torch.bool, device=DEV))
        if not rnt:
            kept = S
            if t >= nt - 3:
                conv[at, (pos + t) % ring] = x
        r = torch.rsqrt((o * o).mean(-1, keepdim=True) + EPS)
        zz = z[:, t].double().reshape(B, nvh, DK)
        gate = _silu(zz) if c.get("gate_act", 0) else torch.sigmoid(zz)
        outs.append((o * r * s["norm_w"].double() * gate).reshape(B, nvh * DK))
    return [torch.stack(outs, 1), kept, conv]


def _norm_rope(x, w, pos):
    """RMSNorm and the rotation of the first NROT dimensions; the angle is the product of 32-bit numbers."""
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()
    i = torch.arange(NROT // 2, device=DEV, dtype=torch.float64)
    inv = (1.0 / THETA ** (2.0 * i / NROT)).float()
    ang = (pos.float()[..., None] * inv).double()
    a, b = y[..., :NROT // 2].clone(), y[..., NROT // 2:NROT].clone()
    y[..., :NROT // 2] = a * torch.cos(ang) - b * torch.sin(ang)
    y[..., NROT // 2:NROT] = b * torch.cos(ang) + a * torch.sin(ang)
    return y


def _attn_exact(c, s):
    B, nt, nq, nkv = c["B"], c["nt"], c["nq"], c["nkv"]
    grp, T = nq // nkv, s["T"]
    Kc, Vc = s["Kc"].double(), s["Vc"].double()
    og = torch.empty(B, nt, nq, HD, dtype=torch.float64, device=DEV)
    sparse = c["kind"] == "qsa"
    IK = s["IKc"].double() if sparse else None
    BK = s["BKc"].double() if sparse else None
    for b, p in enumerate(_positions(c)):
        tp = torch.arange(p, p + nt, device=DEV)
        q = _norm_rope(s["qg"][b, :, :, 0].double(), s["wq"], tp[:, None].expand(nt, nq))
        kn = _norm_rope(s["k"][b].double(), s["wk"], tp[:, None].expand(nt, nkv))
        for t in range(nt):
            Kc[b, :, (p + t) // 64, :, (p + t) % 64, :] = kn[t].reshape(nkv, HD // 4, 4)
            Vc[b, :, p + t] = s["v"][b, t].double()
        if sparse:
            IK[b, p:p + nt] = s["iqk"][b, :, 4 * IXD:].double()
            j = torch.arange(0, (p + nt) // 4, device=DEV)
            bk = _norm_rope(IK[b, :4 * len(j)].reshape(-1, 4, IXD).mean(1), s["wkn"], 4 * j)
            full = torch.zeros(T // 4, IXD, dtype=torch.float64, device=DEV)
            full[:len(j)] = bk
            BK[b] = full.reshape(T // 256, 64, IXD // 4, 4).permute(0, 2, 1, 3)
            iq = _norm_rope(s["iqk"][b, :, :4 * IXD].double().reshape(nt, 4, IXD), s["wqn"], tp[:, None].expand(nt, 4))
        for t in range(nt):
            n = p + t + 1
            at = torch.arange(n, device=DEV)
            if sparse and n // 4 > 512:
                score = torch.relu(iq[t] @ bk[:n // 4].t().contiguous()).sum(0)
                top = torch.sort(torch.sort(score, descending=True, stable=True).indices[:512]).values
                at = torch.cat([(top[:, None] * 4 + torch.arange(4, device=DEV)).reshape(-1), at[n // 4 * 4:]])
            for h in range(nkv):
                K = Kc[b, h].permute(0, 2, 1, 3).reshape(T, HD)[at]
                sc = (q[t, h * grp:(h + 1) * grp] @ K.t().contiguous()) / math.sqrt(HD)
                o = torch.softmax(sc, -1) @ Vc[b, h][at]
                og[b, t, h * grp:(h + 1) * grp] = o * torch.sigmoid(s["qg"][b, t, h * grp:(h + 1) * grp, 1].double())
    return [og, Kc, Vc] + ([IK, BK] if sparse else [])


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _values(ty, raw, rows, cols):
    """GGUF rows as float64, None for a format whose values come from a codebook file."""
    if ty == BF16:
        return raw.contiguous().view(torch.bfloat16).double().reshape(rows, cols)
    qk, bb = BLOCK[ty]
    blk = raw.reshape(-1, bb)
    n = blk.shape[0]
    lev = torch.tensor(IQ4_LEVELS, dtype=torch.float64, device=DEV)
    if ty == Q8_0:
        y = _f16(blk[:, :2]) * blk[:, 2:].contiguous().view(torch.int8).double()
    elif ty == IQ4_NL:
        y = _f16(blk[:, :2]) * lev[torch.cat([blk[:, 2:] & 15, blk[:, 2:] >> 4], 1).long()]
    elif ty == IQ4_XS:
        sh = blk[:, 2:4].contiguous().view(torch.int16).int() & 0xFFFF
        ib = torch.arange(8, device=DEV)
        ls = ((blk[:, 4:8].int()[:, ib // 2] >> (4 * (ib % 2))) & 15) | (((sh >> (2 * ib)) & 3) << 4)
        q = blk[:, 8:].reshape(n, 8, 16)
        y = (_f16(blk[:, :2]) * (ls - 32))[:, :, None] * lev[torch.cat([q & 15, q >> 4], 2).long()]
    elif ty in (Q4_K, Q5_K):
        sc = blk[:, 4:16].int()
        d = torch.cat([sc[:, 0:4] & 63, (sc[:, 8:12] & 15) | ((sc[:, 0:4] >> 6) << 4)], 1)
        m = torch.cat([sc[:, 4:8] & 63, (sc[:, 8:12] >> 4) | ((sc[:, 4:8] >> 6) << 4)], 1)
        qs = blk[:, bb - 128:].reshape(n, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(n, 8, 32).int()
        if ty == Q5_K:
            q |= ((blk[:, 16:48].int()[:, None, :] >> torch.arange(8, device=DEV)[:, None]) & 1) << 4
        y = (_f16(blk[:, 0:2]) * d)[:, :, None] * q - (_f16(blk[:, 2:4]) * m)[:, :, None]
    elif ty == Q6_K:
        ql, qh = blk[:, 0:128].reshape(n, 2, 2, 32).int(), blk[:, 128:192].reshape(n, 2, 1, 32).int()
        high = (qh >> (2 * torch.arange(4, device=DEV)).reshape(1, 1, 4, 1)) & 3
        q = (torch.cat([ql & 15, ql >> 4], 2) | (high << 4)) - 32
        sc = _f16(blk[:, 208:210])[:, :, None] * blk[:, 192:208].contiguous().view(torch.int8).double().reshape(n, 8, 2)
        y = sc.reshape(n, 2, 4, 2).repeat_interleave(16, 3) * q
    else:
        return None
    return y.reshape(rows, cols)


def _gemv_exact(ty, rows, cols, raw, x):
    step = max(1, (1 << 27) // cols)
    out = []
    for i in range(0, rows, step):
        W = _values(ty, raw[i:i + step], min(step, rows - i), cols)
        if W is None:
            return None
        out.append(x.double() @ W.t().contiguous())
    return torch.cat(out, 1)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "model":
        return None
    if kind in ("gdn", "verify"):
        s = _gdn_inputs(c, seed)
        return _gdn_exact(c, s, s["qkv"], s["ab"], s["z"])
    if kind in ("attn", "qsa"):
        return _attn_exact(c, _attn_inputs(c, seed))
    w, x = _weights(c, seed)
    if kind != "layer":
        return [_gemv_exact(*p, x) for p in w]
    qkv, z, ab = (_gemv_exact(*p, x)[None] for p in w[:3])
    out, S, conv = _gdn_exact(c, _gdn_inputs(dict(c, B=1), seed + 1), qkv, ab, z)
    return [_gemv_exact(*w[3], out[0]), S, conv]
