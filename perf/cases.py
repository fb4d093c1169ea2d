"""Performance cases of the framework: requests as a user's program makes them, through the public plans.

Two families.  "gguf": block-quantised models behind HipMasterPlan (bit-exact by contract); "layers": the layer-list designs behind
HybridPlan.  A pass is one request against a loaded model: `prompt` tokens go through the batched prefill, then `steps` tokens are
decoded one by one with their logits copied to the host.  `fill` positions are in the cache before the pass (an ongoing conversation;
only models whose whole state is a key / value cache, so that a pass can be repeated).  `sequences` > 1 is the static-batched decode.

Layer sizes are those of the models that the benchmark and the tests use; a case takes `layers` of them, and a vocabulary cut in
about the same proportion, so that a model is made in a second and the share of each part of a step stays that of the whole model.
"""
import importlib
import json
import math
import os
import shutil
import struct
import tempfile

import numpy as np
import torch

DEVICE = "cuda"
PORTION = 512                # batched-prefill portion of every plan, as in the benchmark (-b 512)

# width, feed-forward, heads, kv heads, head size, vocabulary, tied head, rope base, norm eps
GGUF_MODELS = {
    "llama-3.2-1b": dict(arch=0, dim=2048, hidden=8192, heads=32, kv=8, hs=64, vocab=32064, tied=True, theta=500000.0, eps=1e-5),
    "llama-3-8b": dict(arch=0, dim=4096, hidden=14336, heads=32, kv=8, hs=128, vocab=16032, tied=False, theta=500000.0, eps=1e-5),
    "qwen3-4b": dict(arch=1, dim=2560, hidden=9728, heads=32, kv=8, hs=128, vocab=16896, tied=True, theta=1000000.0, eps=1e-6),
}
GGML_TYPES = {"f32": 0, "f16": 1, "q4_0": 2, "q8_0": 8}
BYTES_PER_WEIGHT = {"f16": 2.0, "q4_0": 18 / 32, "q8_0": 34 / 32, "bf16": 2.0, "f32": 4.0}

# layer sizes of the layer-list designs as the benchmark has them
LAYER_SIZES = {"1b": dict(width=2048, ff=8192, heads=32, kv=8, dim=64, q_rank=768, kv_rank=224, experts=32, top=4, expert_ff=1024, shared_ff=4096, m_dim=128, m_vdim=256, l_dim=64, l_vdim=128),
               "8b": dict(width=4096, ff=14336, heads=32, kv=8, dim=128, q_rank=1536, kv_rank=448, experts=32, top=4, expert_ff=1792, shared_ff=7168, m_dim=256, m_vdim=512, l_dim=128, l_vdim=256)}
LAYER_VOCAB = 12000


def gguf_case(name, model, weights, layers, fill, prompt, steps, sequences=1):
    case = {"family": "gguf", "model": model, "weights": weights, "layers": layers, "fill": fill, "prompt": prompt, "steps": steps, "sequences": sequences}
    return dict(case, name=name) if name else case


def layers_case(name, design, size, dtype, layers, prompt, steps):
    case = {"family": "layers", "design": design, "size": size, "dtype": dtype, "layers": layers, "prompt": prompt, "steps": steps}
    return dict(case, name=name) if name else case


def listed():
    return [
        # the first answer token of a small model behind a short question: the smallest call, launches and latency
        gguf_case("llama1b-q8-first-token", "llama-3.2-1b", "q8_0", 4, 9, 0, 1),
        # steady generation of the benchmark's model in the middle of a conversation
        gguf_case("llama8b-q8-generate", "llama-3-8b", "q8_0", 4, 389, 0, 8),
        # generation behind a long document
        gguf_case("llama8b-q8-generate-long", "llama-3-8b", "q8_0", 4, 8000, 0, 4),
        # time to the first token of the benchmark's prompt
        gguf_case("llama8b-q8-prompt", "llama-3-8b", "q8_0", 4, 0, 512, 1),
        # 4-bit weights, the other common download of the same model
        gguf_case("llama8b-q4-generate", "llama-3-8b", "q4_0", 4, 200, 0, 8),
        # many users at once: static-batched decode
        gguf_case("qwen4b-q8-batch32", "qwen3-4b", "q8_0", 4, 117, 0, 4, 32),
        # layer-list design (attention, state-space, latent attention): short answer of a small model
        layers_case("noditar1b-bf16-generate", "noditar", "1b", "bf16", 3, 7, 16),
        # its ordinary prompt at the large layer size
        layers_case("noditar8b-bf16-prompt", "noditar", "8b", "bf16", 3, 512, 0),
        # a long, ragged prompt in portions and the first words of the answer
        layers_case("noditar8b-bf16-document", "noditar", "8b", "bf16", 2, 2041, 4),
        # the design with windows and pooled blocks beside retention, and matrix memories: prompt
        layers_case("kosusun8b-bf16-prompt", "kosusun", "8b", "bf16", 2, 600, 0),
        # ... and generation, at the small layer size
        layers_case("kosusun1b-bf16-generate", "kosusun", "1b", "bf16", 3, 5, 24),
        # mixture of experts in float32 (reference precision): a question and its answer
        layers_case("kugadra1b-f32-chat", "kugadra", "1b", "f32", 2, 181, 4),
    ]


def log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    if rng.random() < 0.5:
        model = rng.choice(sorted(GGUF_MODELS))
        mode = rng.choice(["generate", "generate", "prompt", "batch"])
        layers = rng.randint(2, 4)
        if mode == "batch":
            return gguf_case(None, model, "q8_0", layers, log_int(rng, 8, 300), 0, rng.randint(1, 4), rng.randint(2, 32))
        if mode == "prompt":
            weights = rng.choice(["q8_0", "q8_0", "q8_0", "f16"])
            prompt = log_int(rng, 2, 512 if weights == "q8_0" else 128)
            return gguf_case(None, model, weights, layers, rng.choice([0, log_int(rng, 1, 2000)]), prompt, 1)
        return gguf_case(None, model, rng.choice(["q8_0", "q8_0", "q8_0", "q4_0", "f16"]), layers, log_int(rng, 1, 8000), 0, rng.randint(1, 8))
    design = rng.choice(["noditar", "noditar", "kosusun", "kosusun", "kugadra"])
    size = "1b" if design == "kugadra" else rng.choice(["1b", "1b", "8b"])
    return layers_case(None, design, size, "f32" if design == "kugadra" else "bf16", rng.randint(2, 3), log_int(rng, 4, 1500 if design != "kugadra" else 500), log_int(rng, 1, 16))


# ---- models ---------------------------------------------------------------------------------------------------------------------------
def product():
    ge = importlib.import_module("__graft_entry__")
    pkg = ge.load_package()
    return pkg, importlib.import_module(ge.PKG_NAME + ".plan"), importlib.import_module(ge.PKG_NAME + ".hybrid")


def generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def tokens_of(case, seed, vocab):
    """One row of token ids per sequence: everything it reads, in order."""
    n = case.get("fill", 0) + case["prompt"] + case["steps"]
    return np.random.RandomState(int(seed) & 0x7FFFFFFF).randint(0, vocab, (case.get("sequences", 1), n)).astype(np.int32)


def gguf_shapes(case):
    """(name, rows, columns, kind) of every tensor in file order."""
    m = GGUF_MODELS[case["model"]]
    q, kv = m["heads"] * m["hs"], m["kv"] * m["hs"]
    out = [("token_embd.weight", m["vocab"], m["dim"], "mat")]
    for i in range(case["layers"]):
        p = "blk.%d." % i
        out += [(p + "attn_norm.weight", 1, m["dim"], "norm"), (p + "attn_q.weight", q, m["dim"], "mat"), (p + "attn_k.weight", kv, m["dim"], "mat"),
                (p + "attn_v.weight", kv, m["dim"], "mat"), (p + "attn_output.weight", m["dim"], q, "mat")]
        if m["arch"] == 1:
            out += [(p + "attn_q_norm.weight", 1, m["hs"], "norm"), (p + "attn_k_norm.weight", 1, m["hs"], "norm")]
        out += [(p + "ffn_norm.weight", 1, m["dim"], "norm"), (p + "ffn_gate.weight", m["hidden"], m["dim"], "mat"),
                (p + "ffn_down.weight", m["dim"], m["hidden"], "mat"), (p + "ffn_up.weight", m["hidden"], m["dim"], "mat")]
    out.append(("output_norm.weight", 1, m["dim"], "norm"))
    if not m["tied"]:
        out.append(("output.weight", m["vocab"], m["dim"], "mat"))
    return out


def gguf_tensors(case, seed):
    """name -> (raw bytes on the GPU, type, rows, columns): N(0, 0.02^2) matrices in the file format's blocks of 32."""
    g = generator(seed)
    for name, rows, cols, kind in gguf_shapes(case):
        w = torch.randn((rows, cols), generator=g, device=DEVICE) * 0.02
        if kind == "norm":
            yield name, (w + 1.0).view(torch.uint8).reshape(-1), "f32", rows, cols
        elif case["weights"] == "f16":
            yield name, w.half().view(torch.uint8).reshape(-1), "f16", rows, cols
        elif case["weights"] == "q8_0":
            w = w.view(-1, 32)
            d = w.abs().amax(1, keepdim=True) / 127.0
            q = torch.round(w / d).to(torch.int8)
            yield name, torch.cat([d.half().view(torch.uint8), q.view(torch.uint8)], 1).reshape(-1), "q8_0", rows, cols
        else:
            w = w.view(-1, 32)
            d = w.gather(1, w.abs().argmax(1, keepdim=True)) / -8.0
            q = torch.clamp(torch.floor(w / d + 8.5), 0, 15).to(torch.uint8)
            yield name, torch.cat([d.half().view(torch.uint8), q[:, :16] | (q[:, 16:] << 4)], 1).reshape(-1), "q4_0", rows, cols


def layer_config(case):
    z, n = LAYER_SIZES[case["size"]], case["layers"]
    W, H, G, D = z["width"], z["heads"], z["kv"], z["dim"]
    cfg = {"vocab": LAYER_VOCAB, "width": W}
    if case["design"] == "noditar":
        mlp = {"kind": "dense", "ff": z["ff"], "limit": 7.0}
        kinds = [{"type": "attention", "mixer": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5}, "mlp": mlp},
                 {"type": "mamba2", "mixer": {"heads": 2 * W // 64, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4}, "mlp": None},
                 {"type": "latent_attention", "mixer": {"heads": H, "dim": D, "vdim": D, "kv_rank": 512, "scale": D ** -0.5}, "mlp": mlp}]
        return dict(cfg, architecture="Noditar", streams=2, norm={"eps": 1e-5}, layers=kinds[:n])
    if case["design"] == "kosusun":
        mlp = {"kind": "dense", "ff": z["ff"]}
        decay = [1.0 - 2.0 ** (-5.0 - 3.0 * i / 15) for i in range(16)]
        par = {"type": "parallel", "mlp": mlp, "mixer": {
            "left": {"heads": H, "kv_heads": G, "dim": D, "vdim": D, "scale": D ** -0.5, "mask": {"size": 1024, "pool": 16}, "rot": {"base": 500000.0, "dims": D, "scaling": {"factor": 2.0}}},
            "right": {"heads": 16, "dim": z["l_dim"], "vdim": z["l_vdim"], "rot": {"base": 10000.0, "dims": z["l_dim"]}, "decay": decay}, "left_scale": 0.7, "right_scale": 0.7}}
        mls = {"type": "mlstm", "mlp": mlp, "mixer": {"heads": 8, "dim": z["m_dim"], "vdim": z["m_vdim"], "gate_cap": 15.0}}
        return dict(cfg, architecture="Kosusun", embedding={"scale": float(W) ** 0.5}, norm={"eps": 1e-6}, residual_mult=0.5, logit_scale=0.5, layers=[par, mls, par][:n])
    moe = {"kind": "moe", "expert": {"ff": z["expert_ff"]}, "router": {"experts": z["experts"], "top": z["top"], "scale": 2.5}, "shared": {"ff": z["shared_ff"]}}
    lig = {"type": "lightning", "mixer": {"heads": 16, "dim": z["l_dim"], "vdim": z["l_vdim"], "decay": [1.0 - 2.0 ** (-5.0 - 3.0 * i / 15) for i in range(16)]}}
    lat = {"type": "latent_attention", "mixer": {"heads": H, "dim": D, "rot_dim": D // 2, "vdim": D, "kv_rank": z["kv_rank"], "q_rank": z["q_rank"], "scale": float(D + D // 2) ** -0.5,
           "rot": {"base": 500000.0, "dims": D // 2, "scaling": {"factor": 8.0, "original": 4096, "fast": 16.0, "slow": 2.0}}}}
    second = dict(lat, mlp=moe)
    third = {"type": "latent_attention", "mixer": dict(lat["mixer"], kv_from=1), "mlp": moe}
    return dict(cfg, architecture="Kugadra", embedding={"scale": float(W) ** 0.5}, norm={"eps": 1e-6}, logit_softcap=50.0,
                layers=[dict(lig, mlp={"kind": "dense", "ff": z["ff"]}), second, third][:n])


def layer_shapes(cfg):
    """name -> shape of every tensor of a configuration, in file order."""
    W, V, design, S = cfg["width"], cfg["vocab"], cfg["architecture"], cfg.get("streams", 1)
    out = {"embed": (V, W)}
    for i, layer in enumerate(cfg["layers"]):
        p, m, ff, kind = "l%d." % i, layer["mixer"], layer.get("mlp"), layer["type"]
        out[p + "norm1"] = (W,)
        if design == "Kugadra":
            out[p + "norm1b"] = (W,)
        x = p + "mix."
        if kind == "parallel":
            a, r = m["left"], m["right"]
            nq, nk, nv, rk, rv = a["heads"] * a["dim"], a["kv_heads"] * a["dim"], a["kv_heads"] * a["vdim"], r["heads"] * r["dim"], r["heads"] * r["vdim"]
            left = {"q": (nq, W), "q.b": (nq,), "k": (nk, W), "k.b": (nk,), "v": (nv, W), "v.b": (nv,), "q.norm": (nq,), "k.norm": (nk,), "sink": (a["heads"],), "o": (W, a["heads"] * a["vdim"])}
            out.update({x + "left." + k: v for k, v in left.items()})
            out.update({x + "right." + k: v for k, v in {"q": (rk, W), "k": (rk, W), "v": (rv, W), "g": (rv, W), "o": (W, rv)}.items()})
        else:
            od, H = m["heads"] * m["vdim"], m["heads"]
            if kind == "attention":
                t = {"q": (H * m["dim"], W), "k": (m["kv_heads"] * m["dim"], W), "v": (m["kv_heads"] * m["vdim"], W), "g": (od, W)}
            elif kind == "mamba2":
                ch = od + 2 * m["groups"] * m["state"]
                t = {"in": (od + ch + H, W), "conv": (ch, m["conv"]), "conv.b": (ch,), "dt_bias": (H,), "A_log": (H,), "D": (H,), "norm": (od,)}
            elif kind == "mlstm":
                t = {"q": (H * m["dim"], W), "k": (H * m["dim"], W), "v": (od, W), "g": (od, W), "norm": (od,), "i": (H, W), "i.b": (H,), "f": (H, W), "f.b": (H,)}
            elif kind == "lightning":
                t = {"q": (H * m["dim"], W), "k": (H * m["dim"], W), "v": (od, W), "g": (od, W), "norm": (od,)}
            elif design == "Kugadra":
                P = m["rot_dim"]
                t = {"dq": (m["q_rank"], W), "dq.norm": (m["q_rank"],), "uq": (H * (m["dim"] + P), m["q_rank"]), "uk": (H * m["dim"], m["kv_rank"]), "uv": (od, m["kv_rank"]), "g": (H, W)}
                if m.get("kv_from") is None:
                    t.update({"dkv": (m["kv_rank"] + P, W), "dkv.norm": (m["kv_rank"],)})
            else:
                t = {"q": (H * m["dim"], W), "dkv": (m["kv_rank"], W), "dkv.norm": (m["kv_rank"],), "uk": (H * m["dim"], m["kv_rank"]), "uv": (od, m["kv_rank"]), "g": (od, W)}
            out.update({x + k: v for k, v in t.items()})
            out[x + "o"] = (W, od)
        if ff:
            if design != "Kosusun":
                out[p + "norm2"] = (W,)
            if design == "Kugadra":
                out[p + "norm2b"] = (W,)
            x = p + "mlp."
            if ff["kind"] == "moe":
                f, E = ff["expert"]["ff"], ff["router"]["experts"]
                for e in range(E):
                    out.update({x + "e%d.gate" % e: (f, W), x + "e%d.up" % e: (f, W), x + "e%d.down" % e: (W, f)})
                f = ff["shared"]["ff"]
                out.update({x + "router": (E, W), x + "correction": (E,), x + "shared.gate": (f, W), x + "shared.up": (f, W), x + "shared.down": (W, f)})
            elif design == "Kugadra":
                out.update({x + "up": (ff["ff"], W), x + "down": (W, ff["ff"])})
            else:
                out.update({x + "gate": (ff["ff"], W), x + "up": (ff["ff"], W), x + "down": (W, ff["ff"])})
        if design == "Noditar":
            for q in ((1, 2) if ff else (1,)):
                out.update({p + "hc%d.in" % q: (S,), p + "hc%d.out" % q: (S,), p + "hc%d.mix" % q: (S, S)})
    out["final.norm"] = (W,)
    if design != "Kugadra":
        out["head"] = (V, W)
    return out


def layer_tensors(cfg, seed):
    """name -> bfloat16 tensor on the GPU, scaled so that activations stay of order one and gates, routers and decays move."""
    g = generator(seed)
    emb = (cfg.get("embedding") or {}).get("scale", 1.0)
    out = {}
    for name, shp in layer_shapes(cfg).items():
        leaf = name.split(".", 1)[1] if name[0] == "l" else name
        last = leaf.rsplit(".", 1)[-1]
        a = torch.randn(shp, generator=g, device=DEVICE)
        if leaf.startswith("hc"):
            S = shp[0]
            a = torch.eye(S, device=DEVICE) + 0.1 * a if last == "mix" else 1.0 / S + 0.1 * a if last == "in" else 1.0 + 0.2 * a
        elif last in ("norm", "norm1", "norm2", "norm1b", "norm2b"):
            a = 1.0 + 0.1 * a
        elif name == "embed":
            a = a / emb
        elif last == "A_log":
            a = -0.5 + 0.5 * torch.tanh(a)
        elif last == "dt_bias":
            a = -0.75 + torch.tanh(a)
        elif last == "D":
            a = 1.0 + 0.2 * a
        elif leaf == "mix.conv":
            a = 0.4 * a
        elif leaf == "mix.f.b":
            a = 2.0 + a
        elif leaf == "mlp.correction":
            a = 0.3 * a / shp[0]
        elif leaf == "mlp.router":
            a = 3.0 * a / math.sqrt(shp[-1])
        elif len(shp) == 1:
            a = 0.3 * a
        else:
            a = a / math.sqrt(shp[-1])
        out[name] = a.bfloat16()
    return out


def write_folder(cfg, tensors, path):
    """config.json and model.safetensors, as a user has them on disk."""
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump(cfg, f)
    head, at = {}, 0
    for name, t in tensors.items():
        head[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + 2 * t.numel()]}
        at += 2 * t.numel()
    text = json.dumps(head).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for t in tensors.values():
            f.write(t.contiguous().view(torch.int16).cpu().numpy().data)


# ---- the request ------------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    pkg, plans, hybrid = product()
    if case["family"] == "gguf":
        m = GGUF_MODELS[case["model"]]
        n, B = case["fill"] + case["prompt"] + case["steps"], case["sequences"]
        synth = pkg.synth
        cfg = synth.ModelConfig(case["model"], m["arch"], m["dim"], m["hidden"], case["layers"], m["heads"], m["kv"], m["hs"], m["vocab"], n + 8, m["eps"], m["theta"], m["tied"])
        model = synth.StreamModel(cfg, GGML_TYPES[case["weights"]], ((name, raw.cpu().numpy(), GGML_TYPES[kind], r, c) for name, raw, kind, r, c in gguf_tensors(case, seed)))
        plan = plans.HipMasterPlan.initializeTornadoVMPlan(model, prefill_batch_size=PORTION, n_seqs=B)
        tok = tokens_of(case, seed, m["vocab"])
        for b in range(B):
            if case["fill"]:
                plan.prefill_seq(b, tok[b, :case["fill"]], 0)
        return {"case": case, "plan": plan, "tokens": tok}
    cfg = layer_config(case)
    path = tempfile.mkdtemp(prefix="cases_", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
    try:
        write_folder(cfg, layer_tensors(cfg, seed), path)
        plan = hybrid.HybridPlan.from_dir(path, dtype="float32" if case["dtype"] == "f32" else "bfloat16", ctx=case["prompt"] + case["steps"] + 8, max_batch=PORTION)
    finally:
        shutil.rmtree(path, ignore_errors=True)
    return {"case": case, "plan": plan, "seq": plan.acquire(), "tokens": tokens_of(case, seed, cfg["vocab"])}


def run(state):
    """The logits of the request: one row (per sequence) for the prompt's end (layer-list plans) and one for every decoded token."""
    case, plan, tok = state["case"], state["plan"], state["tokens"]
    p, s = case["prompt"], case["steps"]
    out = []
    if case["family"] == "gguf":
        f, B = case["fill"], case["sequences"]
        if B > 1:
            for i in range(s):
                logits, ids = plan.forward_decode_batch(tok[:, f + i], np.arange(B), np.full(B, f + i))
                out.append({"logits": logits, "ids": ids})
            return out
        if p:
            plan.prefill(tok[0, f:f + p], f)
        for i in range(s):
            out.append(plan.forward_decode(int(tok[0, f + p + i]), f + p + i))
        return out
    out.append(plan.step(state["seq"], tok[0, :p], 0, want=[p - 1]))
    for i in range(s):
        out.append(plan.step(state["seq"], tok[0, p + i:p + i + 1], p + i, want=[0]))
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------------------
def work(case):
    """Weights once per call (a prompt portion or a decoded token; of the experts, those that can be chosen), cached rows once per call,
    logits once; two operations per weight and token and per cached element and query."""
    p, s = case["prompt"], case["steps"]
    calls = [(min(PORTION, p - a), a, False) for a in range(0, p, PORTION)]           # (tokens, positions in front, logits wanted)
    if case["family"] == "gguf":
        m, B, f = GGUF_MODELS[case["model"]], case["sequences"], case["fill"]
        per = BYTES_PER_WEIGHT[case["weights"]]
        body = sum(r * c for name, r, c, kind in gguf_shapes(case) if kind == "mat" and name.startswith("blk."))
        head, row = m["vocab"] * m["dim"], case["layers"] * 2 * m["kv"] * m["hs"]
        calls = [(n, a + f, False) for n, a, _ in calls] + [(1, f + p + i, True) for i in range(s)]
        nbytes = flops = 0.0
        for n, a, logits in calls:
            nbytes += body * per + B * (row * 4.0 * (a + 2 * n)) + (head * per + B * m["vocab"] * 4.0 if logits else 0.0)
            flops += B * (2.0 * body * n + 4.0 * case["layers"] * m["heads"] * m["hs"] * n * (a + (n + 1) / 2) + (2.0 * head if logits else 0.0))
        return {"bytes": nbytes, "flops": flops}
    cfg = layer_config(case)
    per = BYTES_PER_WEIGHT[case["dtype"]]
    calls = [(n, a, a + n == p) for n, a, _ in calls] + [(1, p + i, True) for i in range(s)]
    head = cfg["vocab"] * cfg["width"]
    nbytes = flops = 0.0
    shapes = layer_shapes(cfg)
    for n, a, logits in calls:
        for name, shp in shapes.items():
            if name[0] != "l" or len(shp) != 2 or ".hc" in name or name.endswith(".conv"):
                continue
            share = 1.0
            if ".mlp.e" in name:
                share = cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]["top"] / cfg["layers"][int(name[1:name.index(".")])]["mlp"]["router"]["experts"]
            nbytes += shp[0] * shp[1] * per * min(1.0, share * n)
            flops += 2.0 * shp[0] * shp[1] * share * n
        for layer in cfg["layers"]:
            m = layer["mixer"]
            if layer["type"] == "parallel":
                a_, r = m["left"], m["right"]
                span = min(a + (n + 1) / 2, a_["mask"]["size"])
                nbytes += 4.0 * min(a + 2 * n, a_["mask"]["size"] + 2 * n) * a_["kv_heads"] * 2 * a_["dim"] + 8.0 * r["heads"] * r["dim"] * r["vdim"]
                flops += 4.0 * n * span * a_["heads"] * a_["dim"] + 4.0 * n * r["heads"] * r["dim"] * r["vdim"]
            elif layer["type"] in ("mamba2", "mlstm", "lightning"):
                cells = m["heads"] * (m.get("state") or m["dim"]) * m["vdim"]
                nbytes += 8.0 * cells
                flops += 4.0 * n * cells
            else:
                row = m["kv_heads"] * 2 * m["dim"] if layer["type"] == "attention" else m["kv_rank"] + m.get("rot_dim", 0)
                nbytes += 4.0 * row * (a + 2 * n)
                flops += 4.0 * n * (a + (n + 1) / 2) * m["heads"] * m["dim"]
        if logits:
            nbytes += head * per + 4.0 * cfg["vocab"]
            flops += 2.0 * head
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """gguf: bit-exact by contract.  layers: float32 plans differ by float32 sums in another order; bfloat16 plans round every matrix
    product's input, and a sum in another order moves some of these roundings by one place."""
    if case["family"] == "gguf":
        return "exact"
    # against 64 bits: float32 up to 2.9e-6, bfloat16 2.4e-3 to 4.7e-3 (four times that)
    return {"rel": 1.2e-5, "max": 2e-4} if case["dtype"] == "f32" else {"rel": 1.9e-2, "max": 1.5e-1}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------------------------------
def unit_rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def sigmoid(z):
    return 1.0 / (1.0 + torch.exp(-z))


def dequantised(raw, kind, rows, cols):
    if kind == "f32":
        return raw.view(torch.float32).double().view(rows, cols)
    if kind == "f16":
        return raw.view(torch.float16).double().view(rows, cols)
    blk = raw.view(-1, 34 if kind == "q8_0" else 18)
    d = blk[:, :2].contiguous().view(torch.float16).double()
    q = blk[:, 2:].contiguous()
    q = q.view(torch.int8).double() if kind == "q8_0" else torch.cat([(q & 15).double() - 8, (q >> 4).double() - 8], 1)
    return (q * d).view(rows, cols)


def exact_gguf(case, seed):
    m = GGUF_MODELS[case["model"]]
    w = {name: dequantised(raw, kind, r, c) for name, raw, kind, r, c in gguf_tensors(case, seed)}
    tok, hs, H, G, eps = tokens_of(case, seed, m["vocab"]), m["hs"], m["heads"], m["kv"], m["eps"]
    T, B = tok.shape[1], tok.shape[0]

    def mul(name, x):                 # Q8_0: the activation is rounded to int8 per block of 32, as the model's arithmetic is defined
        if case["weights"] == "q8_0":
            b = x.view(x.shape[0], -1, 32)
            d = (b.abs().amax(-1, keepdim=True) / 127.0)
            s = b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
            x = (torch.trunc(s + torch.copysign(torch.full_like(s, 0.5), s)) * d.half().double()).view(x.shape)
        return x @ w[name].T

    freq = (1.0 / np.power(np.float64(m["theta"]), np.arange(0, hs, 2) / np.float64(hs))).astype(np.float32)
    ang = torch.from_numpy((np.arange(T, dtype=np.float32)[:, None] * freq[None]).astype(np.float32)).double().to(DEVICE)[:, None, :]
    c, s = torch.cos(ang), torch.sin(ang)

    def turn(x):                       # adjacent pairs (llama), half-split pairs (qwen3)
        if m["arch"] == 0:
            a, b = x[..., 0::2], x[..., 1::2]
            return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(x.shape)
        a, b = x[..., :hs // 2], x[..., hs // 2:]
        return torch.cat([a * c - b * s, a * s + b * c], -1)

    outs = []
    for row in tok:
        x = w["token_embd.weight"][torch.from_numpy(row).long().to(DEVICE)]
        for i in range(case["layers"]):
            p = "blk.%d." % i
            h = unit_rms(x, eps) * w[p + "attn_norm.weight"]
            q, k, v = (mul(p + "attn_%s.weight" % n, h).view(T, -1, hs) for n in "qkv")
            if m["arch"] == 1:
                q, k = unit_rms(q, eps) * w[p + "attn_q_norm.weight"], unit_rms(k, eps) * w[p + "attn_k_norm.weight"]
            o = softmax_attention(turn(q), turn(k), v, H // G, hs ** -0.5)
            x = x + mul(p + "attn_output.weight", o)
            h = unit_rms(x, eps) * w[p + "ffn_norm.weight"]
            g = mul(p + "ffn_gate.weight", h)
            x = x + mul(p + "ffn_down.weight", g * sigmoid(g) * mul(p + "ffn_up.weight", h))
        y = unit_rms(x[T - case["steps"]:], eps) * w["output_norm.weight"]
        outs.append(mul("token_embd.weight" if m["tied"] else "output.weight", y))
    if B == 1:
        return [outs[0][i] for i in range(case["steps"])]
    return [{"logits": torch.stack([o[i] for o in outs]), "ids": None} for i in range(case["steps"])]


def softmax_attention(q, k, v, per, scale, slopes=None, unit=False, sink=None, seen=None):
    """Causal attention [T, heads * vdim], one head at a time; q [T, H, D], k / v [J, G, .]; slopes: distance penalty per head; unit / sink:
    one more entry of the denominator (score 0, or a score per head); seen [T, J] in place of the causal mask."""
    T, J = q.shape[0], k.shape[0]
    i = torch.arange(T, device=q.device)[:, None]
    j = torch.arange(J, device=q.device)[None, :]
    seen = (j <= i) if seen is None else seen
    out = []
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // per].T) * scale
        if slopes is not None:
            s = s - slopes[h] * (i - j)
        s = torch.where(seen, s, torch.full_like(s, -math.inf))
        m = s.amax(1, keepdim=True)
        extra = 0.0
        if unit or sink is not None:
            z = torch.zeros_like(m) if unit else sink[h].expand_as(m)
            m = torch.maximum(m, z)
            extra = torch.exp(z - m)
        e = torch.exp(s - m)
        out.append((e / (e.sum(1, keepdim=True) + extra)) @ v[:, h // per])
    return torch.stack(out, 1).reshape(T, -1)


def rotated(x, freq, mul=1.0, interleaved=False):
    n = 2 * freq.numel()
    a = torch.arange(x.shape[0], device=x.device, dtype=torch.float64)[:, None, None] * freq
    c, s = torch.cos(a) * mul, torch.sin(a) * mul
    y = x.clone()
    u, v = (x[..., 0:n:2], x[..., 1:n:2]) if interleaved else (x[..., :n // 2], x[..., n // 2:n])
    if interleaved:
        y[..., 0:n:2], y[..., 1:n:2] = u * c - v * s, v * c + u * s
    else:
        y[..., :n // 2], y[..., n // 2:n] = u * c - v * s, v * c + u * s
    return y


def frequencies(rot):
    n = rot["dims"]
    i = torch.arange(n // 2, dtype=torch.float64, device=DEVICE)
    f, sc = float(rot["base"]) ** (-2.0 * i / n), rot.get("scaling") or {}
    if "original" not in sc:
        return f / sc.get("factor", 1.0), 1.0
    where = lambda turns: n * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))  # noqa: E731
    lo, hi = max(math.floor(where(sc["fast"])), 0), min(math.ceil(where(sc["slow"])), n - 1)
    ramp = torch.clamp((i - lo) / max(hi - lo, 0.001), 0.0, 1.0)
    return f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def memory(q, k, v, a, b):
    """o_t = S_t^T q_t with S_t = a_t S_(t-1) + b_t k_t v_t^T per head; a, b: [T, H]."""
    T, H, D = q.shape
    S = torch.zeros((H, D, v.shape[2]), dtype=torch.float64, device=q.device)
    o = torch.empty((T, H, v.shape[2]), dtype=torch.float64, device=q.device)
    for t in range(T):
        S = a[t][:, None, None] * S + (b[t][:, None] * k[t])[:, :, None] * v[t][:, None, :]
        o[t] = torch.bmm(q[t][:, None, :], S)[:, 0]
    return o


def mix_noditar(kind, h, p, c, eps):
    T, H = h.shape[0], c["heads"]
    if kind == "mamba2":
        P, N, G, K = c["vdim"], c["state"], c["groups"], c["conv"]
        inner = H * P
        z, xbc, dt = (h @ p["in"].T).split([inner, inner + 2 * G * N, H], 1)
        pad = torch.cat([torch.zeros((K - 1, xbc.shape[1]), dtype=torch.float64, device=h.device), xbc])
        y = sum(pad[i:i + T] * p["conv"][:, i] for i in range(K)) + p["conv.b"]
        y = y * sigmoid(y)
        x, Bm, Cm = y[:, :inner].reshape(T, H, P), y[:, inner:inner + G * N].reshape(T, G, N), y[:, inner + G * N:].reshape(T, G, N)
        dt = torch.logaddexp(dt + p["dt_bias"], torch.zeros_like(dt))
        o = memory(Cm.repeat_interleave(H // G, 1), Bm.repeat_interleave(H // G, 1), x, torch.exp(-torch.exp(p["A_log"]) * dt), dt) + p["D"][:, None] * x
        o = o.reshape(T, inner) * z * sigmoid(z)
        return (unit_rms(o.view(T, c["norm_groups"], -1), eps).reshape(T, inner) * p["norm"]) @ p["o"].T
    q = (h @ p["q"].T).view(T, H, -1)
    if kind == "attention":
        k, v = ((h @ p[n].T).view(T, c["kv_heads"], -1) for n in "kv")
        slopes = [2.0 ** (-8.0 * (i + 1) / H) for i in range(H)]
        o = softmax_attention(unit_rms(q, eps), unit_rms(k, eps), v, H // c["kv_heads"], c["scale"], slopes, unit=True)
    else:
        lat = unit_rms(h @ p["dkv"].T, eps) * p["dkv.norm"]
        o = softmax_attention(q, (lat @ p["uk"].T).view(T, H, -1), (lat @ p["uv"].T).view(T, H, -1), 1, c["scale"])
    return (o * sigmoid(h @ p["g"].T)) @ p["o"].T


def mix_kosusun(kind, h, p, c, eps):
    T = h.shape[0]
    if kind == "mlstm":
        H, cap = c["heads"], c["gate_cap"]
        q, k, v = (h @ p["q"].T).view(T, H, -1) * c["dim"] ** -0.5, (h @ p["k"].T).view(T, H, -1), (h @ p["v"].T).view(T, H, -1)
        ig = cap * torch.tanh((h @ p["i"].T + p["i.b"]) / cap)
        fz = cap * torch.tanh((h @ p["f"].T + p["f.b"]) / cap)
        fg = -torch.logaddexp(-fz, torch.zeros_like(fz))
        m, top = torch.zeros(H, dtype=torch.float64, device=h.device), []
        for t in range(T):
            top.append(torch.maximum(fg[t] + m, ig[t]))
            m = top[-1]
        m = torch.stack(top)
        a = torch.exp(fg + torch.cat([torch.zeros_like(m[:1]), m[:-1]]) - m)
        ones = torch.ones((T, H, 1), dtype=torch.float64, device=h.device)
        o = memory(q, k, torch.cat([v, ones], 2), a, torch.exp(ig - m))          # last column: q . n
        o = o[..., :-1] / (torch.maximum(o[..., -1].abs(), torch.exp(-m)) + 1e-6)[:, :, None]
        return (unit_rms(o, eps).reshape(T, -1) * p["norm"] * sigmoid(h @ p["g"].T)) @ p["o"].T
    a, r = c["left"], c["right"]
    L = {k[5:]: v for k, v in p.items() if k.startswith("left.")}
    R = {k[6:]: v for k, v in p.items() if k.startswith("right.")}
    f, _ = frequencies(a["rot"])
    q, k = (rotated((unit_rms(h @ L[n].T + L[n + ".b"], eps) * L[n + ".norm"]).view(T, -1, a["dim"]), f, 1.0, True) for n in "qk")
    v = (h @ L["v"].T + L["v.b"]).view(T, a["kv_heads"], -1)
    size, pool = a["mask"]["size"], a["mask"]["pool"]
    nb = T // pool
    i = torch.arange(T, device=h.device)[:, None]
    j = torch.arange(T, device=h.device)[None, :]
    blocks = torch.clamp((i - size + 1).div(pool, rounding_mode="floor"), min=0)
    seen = torch.cat([torch.arange(nb, device=h.device)[None, :] < blocks, (j <= i) & (j > i - size)], 1)
    mean = lambda x: torch.cat([x[:nb * pool].view(nb, pool, x.shape[1], x.shape[2]).mean(1), x])  # noqa: E731
    left = softmax_attention(q, mean(k), mean(v), a["heads"] // a["kv_heads"], a["scale"], sink=L["sink"], seen=seen) @ L["o"].T
    f, _ = frequencies(r["rot"])
    q, k = (rotated((h @ R[n].T).view(T, r["heads"], -1), f) for n in "qk")
    decay = torch.tensor(r["decay"], dtype=torch.float64, device=h.device).expand(T, -1)
    o = memory(q, k * r["dim"] ** -0.5, (h @ R["v"].T).view(T, r["heads"], -1), decay, torch.ones_like(decay))
    g = h @ R["g"].T
    return c["left_scale"] * left + c["right_scale"] * ((unit_rms(o, eps).reshape(T, -1) * g * sigmoid(g)) @ R["o"].T)


def mix_kugadra(kind, h, p, c, eps, cache):
    T, H = h.shape[0], c["heads"]
    if kind == "lightning":
        q, k, v = ((lambda z: z * sigmoid(z))(h @ p[n].T).view(T, H, -1) for n in "qkv")
        decay = torch.tensor(c["decay"], dtype=torch.float64, device=h.device).expand(T, -1)
        o = memory(q, k, v, decay, torch.ones_like(decay))
        return (unit_rms(o.reshape(T, -1), eps) * p["norm"] * sigmoid(h @ p["g"].T)) @ p["o"].T
    R, D = c["kv_rank"], c["dim"]
    f, mul = frequencies(c["rot"])
    if "dkv" in p:
        z = h @ p["dkv"].T
        cache[:] = [unit_rms(z[:, :R], eps) * p["dkv.norm"], rotated(z[:, None, R:], f, mul)]
    lat, kr = cache
    q = ((unit_rms(h @ p["dq"].T, eps) * p["dq.norm"]) @ p["uq"].T).view(T, H, -1)
    q = torch.cat([q[..., :D], rotated(q[..., D:], f, mul)], 2)
    k = torch.cat([(lat @ p["uk"].T).view(T, H, D), kr.expand(T, H, -1)], 2)
    o = softmax_attention(q, k, (lat @ p["uv"].T).view(T, H, -1), 1, c["scale"]).view(T, H, -1)
    return (o * sigmoid(h @ p["g"].T)[:, :, None]).reshape(T, -1) @ p["o"].T


def feed_forward(design, h, p, c):
    if design == "Noditar":
        g, u = torch.clamp(h @ p["gate"].T, max=c["limit"]), torch.clamp(h @ p["up"].T, -c["limit"], c["limit"])
        return (g * sigmoid(1.702 * g) * (u + 1.0)) @ p["down"].T
    if design == "Kosusun":
        g = h @ p["gate"].T
        return (0.5 * g * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (g + 0.044715 * g ** 3))) * (h @ p["up"].T)) @ p["down"].T
    if c["kind"] == "dense":
        return torch.clamp(h @ p["up"].T, min=0.0).square() @ p["down"].T
    def gated(x, e):
        g = x @ p[e + ".gate"].T
        return (g * sigmoid(g) * (x @ p[e + ".up"].T)) @ p[e + ".down"].T
    s = torch.softmax(h @ p["router"].T, -1)
    choice = torch.argsort(s + p["correction"], dim=-1, descending=True, stable=True)[:, :c["router"]["top"]]
    weight = s.gather(1, choice)
    weight = weight / (weight.sum(-1, keepdim=True) + 1e-20) * c["router"]["scale"]
    out = gated(h, "shared")
    for e in range(c["router"]["experts"]):
        row, col = (choice == e).nonzero(as_tuple=True)
        if row.numel():
            out[row] += weight[row, col][:, None] * gated(h[row], "e%d" % e)
    return out


def exact_layers(case, seed):
    cfg = layer_config(case)
    design, eps = cfg["architecture"], cfg["norm"]["eps"]
    weights = layer_tensors(cfg, seed)
    tok = tokens_of(case, seed, cfg["vocab"])[0]
    x = weights["embed"][torch.from_numpy(tok).long().to(DEVICE)].double() * (cfg.get("embedding") or {}).get("scale", 1.0)
    xs = x.expand(cfg.get("streams", 1), -1, -1)
    cache = []
    for i, layer in enumerate(cfg["layers"]):
        w = {k.split(".", 1)[1]: v.double() for k, v in weights.items() if k.startswith("l%d." % i)}
        part = lambda s: {k[len(s):]: v for k, v in w.items() if k.startswith(s)}  # noqa: E731
        mix, ff, kind, c = part("mix."), part("mlp."), layer["type"], layer["mixer"]
        if design == "Noditar":
            for q, fn in ((1, lambda h: mix_noditar(kind, h, mix, c, eps)), (2, lambda h: feed_forward(design, h, ff, layer["mlp"]))):
                if q == 2 and layer["mlp"] is None:
                    continue
                y = fn(unit_rms(torch.tensordot(w["hc%d.in" % q], xs, dims=([0], [0])), eps) * w["norm%d" % q])
                xs = torch.tensordot(w["hc%d.mix" % q].T, xs, dims=([1], [0])) + w["hc%d.out" % q][:, None, None] * y
        elif design == "Kosusun":
            h = unit_rms(xs[0], eps) * w["norm1"]
            xs = xs + cfg["residual_mult"] * (mix_kosusun(kind, h, mix, c, eps) + feed_forward(design, h, ff, layer["mlp"]))
        else:
            xs = xs + unit_rms(mix_kugadra(kind, unit_rms(xs[0], eps) * w["norm1"], mix, c, eps, cache), eps) * w["norm1b"]
            xs = xs + unit_rms(feed_forward(design, unit_rms(xs[0], eps) * w["norm2"], ff, layer["mlp"]), eps) * w["norm2b"]
    x = unit_rms(xs.sum(0)[case["prompt"] - 1:], eps) * weights["final.norm"].double()
    z = x @ weights["head" if "head" in weights else "embed"].double().T * cfg.get("logit_scale", 1.0)
    cap = cfg.get("logit_softcap")
    z = cap * torch.tanh(z / cap) if cap else z
    return [z[i:i + 1] for i in range(z.shape[0])]


def exact(case, seed):
    return exact_gguf(case, seed) if case["family"] == "gguf" else exact_layers(case, seed)
