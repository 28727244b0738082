"""The work whose speed is measured: what a program that serves a qwen35 hybrid model through this library has it do.

Seven kinds of case, each through the public entry points (the C ABI behind rapier_amd, the Engine class):

  gemv     one quantized projection of 1..16 activation columns (Q6_K, Q5_K, Q4_K, Q8_0), plain or with the residual
  ffn      norm, up and gate projections, SwiGLU and the down projection with the residual, as an engine chains them
  head     final norm, vocabulary projection, greedy token and the top-40 list of a serving loop
  gdn      one Gated-DeltaNet layer over 1 (decode), 2 (verify) or up to 16 (prompt chunk) tokens
  attn     one attention layer (per-head norm, RoPE, cache write, split-K decode, gate) over the same token counts
  prefill  a whole prompt through the 9B engine, with the logits that choose the next token
  decode   tokens generated by the 9B engine behind a context, greedy or with draft verification

Sizes are those of the 9B configuration and of the small test configuration, with ragged ones around them.
"""
import ctypes
import math

import numpy as np
import torch

import rapier_amd as rmi
from rapier_amd import engine as rmi_engine

TYPES = {"q6_k": 14, "q5_k": 13, "q4_k": 12, "q8_0": 8}
BLOCK = {"q6_k": (256, 210), "q5_k": (256, 176), "q4_k": (256, 144), "q8_0": (32, 34)}
EPS = 1e-6
S = 128            # GDN state size
HD, ROT = 256, 64  # attention head and rotary dims
THETA = 1e7
TOPK = 40
VOCAB = 248320


def listed():
    return [
        # the k | v rows of one decoded token, plain blocks: the smallest projection, bound by latency and the launch
        {"name": "kv_proj_1tok", "kind": "gemv", "type": "q6_k", "packed": False, "n_in": 4096, "n_out": 2048, "ncols": 1,
         "res": False},
        # the output projection of a verified token pair, in the type mixed files give single matrices
        {"name": "out_proj_2tok_q8_0", "kind": "gemv", "type": "q8_0", "packed": False, "n_in": 4096, "n_out": 4096,
         "ncols": 2, "res": True},
        # the q | k | v projection of a 16-token prompt chunk on the file's own blocks
        {"name": "qkv_16tok", "kind": "gemv", "type": "q6_k", "packed": False, "n_in": 4096, "n_out": 10240, "ncols": 16,
         "res": False},
        # the feed-forward block of a verified pair on packed weights: the largest part of a decode round
        {"name": "ffn_verify", "kind": "ffn", "type": "q6_k", "packed": True, "n_embd": 4096, "n_ff": 12288, "ncols": 2},
        # the same block for one decoded token of a Q5_K file
        {"name": "ffn_decode_q5_k", "kind": "ffn", "type": "q5_k", "packed": False, "n_embd": 4096, "n_ff": 12288,
         "ncols": 1},
        # the same block for a 16-token prompt chunk of a Q4_K file
        {"name": "ffn_chunk_q4_k", "kind": "ffn", "type": "q4_k", "packed": False, "n_embd": 4096, "n_ff": 12288,
         "ncols": 16},
        # the vocabulary head of a verified pair with the serving loop's list
        {"name": "head_2tok", "kind": "head", "n_embd": 4096, "n_vocab": VOCAB, "ncols": 2},
        # one recurrent layer over a prompt chunk
        {"name": "gdn_chunk", "kind": "gdn", "h_k": 16, "h_v": 32, "ntok": 16},
        # one attention layer of a verified pair behind the longest context of the benchmark (its last rows ragged)
        {"name": "attn_verify_64k", "kind": "attn", "n_head": 16, "n_kv": 4, "ntok": 2, "ctx": 65501},
        # one attention layer of a prompt chunk 4K tokens into its prompt
        {"name": "attn_chunk_4k", "kind": "attn", "n_head": 16, "n_kv": 4, "ntok": 16, "ctx": 4001},
        # a prompt, its length no multiple of any chunk
        {"name": "prefill_9b", "kind": "prefill", "tokens": 1999},
        # a burst of generation with draft verification behind a 4K context
        {"name": "decode_9b_mtp", "kind": "decode", "ctx": 4096, "tokens": 32, "mode": "mtp"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "ffn", "ffn", "ffn", "head", "gdn", "gdn", "attn", "attn", "prefill", "decode"])
    if kind == "gemv":
        packed = rng.random() < 0.35
        t = "q6_k" if packed else rng.choice(list(TYPES))
        n_in = 2048 * rng.randint(1, 6) if packed or rng.random() < 0.6 else 256 * rng.randint(4, 48)
        return {"kind": kind, "type": t, "packed": packed, "n_in": n_in, "n_out": _log(rng, 512, 24576),
                "ncols": rng.choice([1, 1, 2, 2, rng.randint(3, 15), 16]), "res": rng.random() < 0.4}
    if kind == "ffn":
        packed = rng.random() < 0.4
        return {"kind": kind, "type": "q6_k" if packed else rng.choice(["q6_k", "q5_k", "q4_k"]), "packed": packed,
                "n_embd": rng.choice([2048, 4096, 4096]), "n_ff": 2048 * rng.randint(2, 6) if packed else 256 * rng.randint(16, 48),
                "ncols": rng.choice([1, 2, rng.randint(3, 15), 16])}
    if kind == "head":
        return {"kind": kind, "n_embd": rng.choice([2048, 4096]), "n_vocab": _log(rng, 5000, VOCAB), "ncols": rng.choice([1, 2])}
    if kind == "gdn":
        h_k = rng.choice([16, rng.randint(2, 15), rng.randint(2, 15)])
        return {"kind": kind, "h_k": h_k, "h_v": 2 * h_k, "ntok": rng.choice([1, 2, rng.randint(3, 15), rng.randint(3, 16)])}
    if kind == "attn":
        n_head, n_kv = rng.choice([(16, 4), (16, 4), (8, 2)])
        ntok = rng.choice([1, 2, rng.randint(3, 15), 16])
        return {"kind": kind, "n_head": n_head, "n_kv": n_kv, "ntok": ntok, "ctx": _log(rng, 40, 65501 if ntok <= 2 else 16000)}
    if kind == "prefill":
        return {"kind": kind, "tokens": _log(rng, 20, 1999)}
    return {"kind": kind, "ctx": _log(rng, 100, 32768), "tokens": rng.randint(8, 32), "mode": rng.choice(["greedy", "mtp"])}


# ---- inputs -----------------------------------------------------------------------------------------------------------
_stream = None


def _side_stream():
    """the stream every call goes to (the library takes no null stream, as an engine has a stream of its own)"""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std + mean


def _weights(g, type_, n_out, n_in):
    """random blocks of a GGUF matrix: uniform codes and sub-scales, block scales so that a row's weights are ~0.02"""
    per, nbytes = BLOCK[type_]
    nb = n_out * (n_in // per)
    w = torch.randint(0, 256, (nb, nbytes), generator=g, device="cuda", dtype=torch.uint8)

    def half(col, v):
        w[:, col:col + 2] = v.to(torch.float16).view(torch.uint8).reshape(nb, 2)

    spread = torch.rand(nb, generator=g, device="cuda") + 0.5
    if type_ == "q6_k":
        half(208, spread * 1.5e-5)
    elif type_ == "q8_0":
        half(0, spread * 2.7e-4)
    else:
        half(0, spread * (4.4e-5 if type_ == "q4_k" else 2.2e-5))
        half(2, spread * 1.6e-4)
    return w.reshape(-1)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _call(name, *args):
    rmi._check(getattr(rmi.lib(), name)(*args))


def _quantize(x, n, ncols, st):
    q = torch.empty(rmi.native_q8_1_bytes(n, ncols), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    rmi.native_quantize_q8_1(x, q, n, ncols, stream=st)
    return q


def _pack(w, n_in, n_out, st, swiglu=False):
    p = torch.empty(rmi.q6_k_packed_bytes(n_in, n_out), dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    if swiglu:
        rmi.q6_k_pack_swiglu(w, p, n_in, n_out // 2, stream=st)
    else:
        rmi.q6_k_pack(w, p, n_in, n_out, stream=st)
    torch.cuda.synchronize()
    return p


def _u8(n):
    return torch.zeros(n, dtype=torch.uint8, device="cuda")


def _f32(*shape):
    return torch.zeros(*shape, dtype=torch.float32, device="cuda")


def _q8_bytes(n):
    return n // 32 * 36


def _gemv_inputs(c, g):
    w = _weights(g, c["type"], c["n_out"], c["n_in"])
    x = _normal(g, c["ncols"], c["n_in"])
    res = _normal(g, c["ncols"], c["n_out"]) if c["res"] else None
    return w, x, res


def _ffn_inputs(c, g):
    e, f = c["n_embd"], c["n_ff"]
    ug, down = _weights(g, c["type"], 2 * f, e), _weights(g, c["type"], e, f)
    return ug, down, _normal(g, e, mean=1.0, std=0.1), _normal(g, c["ncols"], e)


def _head_inputs(c, g):
    return _weights(g, "q6_k", c["n_vocab"], c["n_embd"]), _normal(g, c["n_embd"], mean=1.0, std=0.1), _normal(g, c["ncols"], c["n_embd"])


def _gdn_inputs(c, g):
    hk, hv, n = c["h_k"], c["h_v"], c["ntok"]
    row = 2 * hk * S + 2 * hv * S + 2 * hv
    d = {"x": _normal(g, n, row), "conv_w": _normal(g, 2 * hk * S + hv * S, 4, std=0.5), "dt": _f32(hv),
         "ssm_a": -torch.exp(_normal(g, hv, std=0.5)), "gamma": _normal(g, S, mean=1.0, std=0.1),
         "state": _normal(g, S, hv, S, std=0.05)}
    std = _normal(g, 2 * hk + hv, S, 3, std=0.5)   # history per conv head; value head h sees key head h % h_k
    q = torch.arange(hv, device="cuda") % hk
    d["hist"] = torch.stack([std[q], std[hk + q], std[2 * hk:]], 1).contiguous()
    return d


def _attn_inputs(c, g):
    nh, kv, n, ctx = c["n_head"], c["n_kv"], c["ntok"], c["ctx"]
    rows = (ctx + 63) // 64 * 64
    return {"q3": _normal(g, n, nh * 2 * HD + 2 * kv * HD), "qn": _normal(g, HD, mean=1.0, std=0.1), "kn": _normal(g, HD, mean=1.0, std=0.1),
            "kc": _normal(g, rows, kv, HD).to(torch.float16), "vc": _normal(g, rows, kv, HD).to(torch.float16), "rows": rows}


def _tokens(seed, n, vocab):
    g = torch.Generator()
    g.manual_seed(seed)
    return torch.randint(0, vocab, (n,), generator=g).tolist()


def prepare(case, seed):
    c, kind = case, case["kind"]
    st = _side_stream()
    g = _gen(seed)
    s = {"case": c, "stream": st, "h": ctypes.c_void_p(st.cuda_stream)}
    if kind == "gemv":
        w, x, res = _gemv_inputs(c, g)
        s["w"] = _pack(w, c["n_in"], c["n_out"], st) if c["packed"] else w
        s["xq"] = _quantize(x, c["n_in"], c["ncols"], st)
        s["res"], s["y"] = res, _f32(c["ncols"], c["n_out"])
        s["part"] = _f32(c["ncols"], (c["n_out"] + 3) // 4)
    elif kind == "ffn":
        e, f, n = c["n_embd"], c["n_ff"], c["ncols"]
        ug, down, s["norm"], s["x"] = _ffn_inputs(c, g)
        s["swiglu"] = c["packed"] and e == 4096
        s["ug"] = _pack(ug, e, 2 * f, st, s["swiglu"]) if c["packed"] else ug
        s["down"] = _pack(down, f, e, st) if c["packed"] else down
        s["xpart"] = s["x"].reshape(n, e // 4, 4).square().sum(-1).contiguous()
        s["xq"], s["h8"] = _u8(n * _q8_bytes(e)), _u8(n * _q8_bytes(f))
        s["h32"], s["y"], s["part"] = _f32(n, 2 * f), _f32(n, e), _f32(n, e // 4)
    elif kind == "head":
        v, e, n = c["n_vocab"], c["n_embd"], c["ncols"]
        w, s["norm"], s["x"] = _head_inputs(c, g)
        s["w"] = _pack(w, e, v, st)
        s["xpart"] = s["x"].reshape(n, e // 4, 4).square().sum(-1).contiguous()
        s["xq"], s["logits"] = _u8(n * _q8_bytes(e)), _f32(n, v)
        s["ids"] = torch.zeros(n, dtype=torch.int32, device="cuda")
        s["top"], s["topv"] = torch.zeros(TOPK, dtype=torch.int32, device="cuda"), _f32(TOPK)
        s["ws"], s["tws"] = _u8(rmi.argmax_workspace_bytes(n)), _u8(rmi.topk_workspace_bytes(v))
    elif kind == "gdn":
        s.update(_gdn_inputs(c, g))
        s["state_b"], s["hist_b"] = torch.zeros_like(s["state"]), torch.zeros_like(s["hist"])
        s["sel"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["y"], s["q8"] = _f32(c["ntok"], c["h_v"] * S), _u8(c["ntok"] * _q8_bytes(c["h_v"] * S))
        s["xch"] = _u8(rmi.gdn_exchange_bytes(c["h_v"]))
    elif kind == "attn":
        s.update(_attn_inputs(c, g))
        nh, kv, n = c["n_head"], c["n_kv"], c["ntok"]
        s["pos"] = torch.arange(c["ctx"] - n, c["ctx"], dtype=torch.int32, device="cuda")
        s["nsub"] = max(2, min(64, -(-s["rows"] // (64 * (256 // kv)))))   # the engine's: a workgroup per compute unit
        s["qbuf"], s["y"], s["q8"] = _f32(n, nh * HD), _f32(n, nh * HD), _u8(n * _q8_bytes(nh * HD))
        s["ws"] = _u8(rmi.gqa_workspace_bytes(s["rows"], kv, s["nsub"]))
    else:
        cfg = rmi_engine.qwen35_9b_config()
        prompt = c.get("ctx", c.get("tokens"))
        e = s["engine"] = rmi_engine.Engine(cfg, seed=seed + 1, max_ctx=prompt + 64 + c["tokens"], stream=st)
        if kind == "prefill":
            s["tokens"] = _tokens(seed, c["tokens"], cfg.n_vocab)
        else:
            s["cur"] = e.synth_context(c["ctx"], seed, _tokens(seed, 1, cfg.n_vocab)[0])
            s["pos"] = e.state()[0]
            e.save_state()
    torch.cuda.synchronize()
    return s


# ---- one pass ---------------------------------------------------------------------------------------------------------
def _gemv(s, type_, packed, w, xq, y, n_in, n_out, n):
    if packed:
        _call("rmi_native_q6_k_mmvq_packed", _ptr(w), _ptr(xq), _ptr(y), n_in, n_out, n, s["h"])
    else:
        _call("rmi_native_mmvq", TYPES[type_], _ptr(w), _ptr(xq), _ptr(y), n_in, n_out, n, s["h"])


def _gemv_res(s, type_, packed, w, xq, y, res, part, n_in, n_out, n):
    name = "rmi_native_q6_k_mmvq_packed_res_n" if packed else "rmi_native_%s_mmvq_res_n" % type_
    _call(name, _ptr(w), _ptr(xq), _ptr(y), _ptr(res), _ptr(part), n_in, n_out, n, s["h"])


def run(s):
    c, kind, st = s["case"], s["case"]["kind"], s["stream"]
    if kind == "gemv":
        if not c["res"]:
            _gemv(s, c["type"], c["packed"], s["w"], s["xq"], s["y"], c["n_in"], c["n_out"], c["ncols"])
            return {"y": s["y"]}
        _gemv_res(s, c["type"], c["packed"], s["w"], s["xq"], s["y"], s["res"], s["part"], c["n_in"], c["n_out"], c["ncols"])
        return {"y": s["y"], "part": s["part"]}
    if kind == "ffn":
        e, f, n = c["n_embd"], c["n_ff"], c["ncols"]
        if s["swiglu"] and n <= 2:
            rmi.native_q6_k_swiglu_packed_norm(s["ug"], s["x"], s["norm"], s["xpart"], EPS, s["h8"], e, f, n, stream=st)
        else:
            rmi.rms_quant_apply(s["x"], s["norm"], s["xpart"], s["xq"], e, EPS, n, stream=st)
            _gemv(s, c["type"], c["packed"], s["ug"], s["xq"], s["h32"], e, 2 * f, n)
            if s["swiglu"]:
                rmi.swiglu_quant_interleaved(s["h32"], s["h8"], f, n, 2 * f, stream=st)
            else:
                rmi.swiglu_quant(s["h32"], s["h32"][0, f:], s["h8"], f, n, 2 * f, stream=st)
        _gemv_res(s, c["type"], c["packed"], s["down"], s["h8"], s["y"], s["x"], s["part"], f, e, n)
        return {"y": s["y"], "part": s["part"]}
    if kind == "head":
        v, e, n = c["n_vocab"], c["n_embd"], c["ncols"]
        rmi.rms_quant_apply(s["x"], s["norm"], s["xpart"], s["xq"], e, EPS, n, stream=st)
        _gemv(s, "q6_k", True, s["w"], s["xq"], s["logits"], e, v, n)
        rmi.argmax(s["logits"], v, s["ids"], s["ws"], n, v, stream=st)
        rmi.topk(s["logits"], v, TOPK, s["top"], s["topv"], s["tws"], stream=st)
        return {"logits": s["logits"], "ids": s["ids"], "top": s["top"], "topv": s["topv"]}
    if kind == "gdn":
        hk, hv, n = c["h_k"], c["h_v"], c["ntok"]
        qkvz, row = 2 * hk * S + 2 * hv * S, 2 * hk * S + 2 * hv * S + 2 * hv
        rmi.gdn_layer_tokens_x(s["state"], s["state_b"], s["hist"], s["hist_b"], s["sel"], s["x"], row, s["x"][0, qkvz:], row, s["conv_w"],
                               s["dt"], s["ssm_a"], s["gamma"], EPS, s["y"], hv * S, s["q8"], _q8_bytes(hv * S), hk, hv, n, s["xch"],
                               stream=st)
        return {"y": s["y"], "q8": s["q8"], "state": s["state"], "hist": s["hist"]}
    if kind == "attn":
        nh, kv, n, rows = c["n_head"], c["n_kv"], c["ntok"], s["rows"]
        stride, q8s, scale = nh * 2 * HD + 2 * kv * HD, _q8_bytes(nh * HD), 1.0 / math.sqrt(HD)
        if n <= 2:
            rmi.gqa_flash_decode_prep(s["q3"], stride, s["qn"], s["kn"], s["kc"], s["vc"], s["pos"], s["y"], nh * HD, s["q8"], q8s, s["ws"],
                                      nh, kv, HD, ROT, THETA, 1.0, 262144.0, EPS, n, rows, s["nsub"], scale, stream=st)
        else:
            rmi.attn_prep(s["q3"], stride, s["qn"], s["kn"], s["kc"], s["vc"], s["pos"], s["qbuf"], nh, kv, HD, ROT, THETA, EPS, n, rows,
                          stream=st)
            rmi.gqa_flash_decode(s["qbuf"], s["kc"], s["vc"], s["pos"], s["q3"], stride, s["y"], nh * HD, s["q8"], q8s, s["ws"], nh, kv, HD,
                                 n, rows, s["nsub"], scale, stream=st)
        new = slice(c["ctx"] - n, c["ctx"])   # what the call adds to the caches
        return {"y": s["y"], "q8": s["q8"], "k": s["kc"][new], "v": s["vc"][new]}
    e = s["engine"]
    if kind == "prefill":
        ids = [e.prefill(s["tokens"])]
    else:
        e.restore_state(s["pos"], s["cur"])
        ids, _ = e.generate(c["tokens"], rmi_engine.MTP if c["mode"] == "mtp" else rmi_engine.GREEDY)
    top = e.topk(TOPK)
    logits = e.read(rmi_engine.BUF_LOGITS, 0, 4 * e.cfg.n_vocab).view("<f4")
    hidden = e.read(rmi_engine.BUF_HIDDEN, 0, 4 * e.cfg.n_embd).view("<f4")
    return {"ids": np.array(ids), "top": np.array([i for i, _ in top]), "logits": logits, "hidden": hidden}


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def _w_bytes(type_, n_out, n_in):
    per, nbytes = BLOCK[type_]
    return n_out * (n_in // per) * nbytes


def work(case):
    c, kind = case, case["kind"]
    if kind == "gemv":
        n, i, o = c["ncols"], c["n_in"], c["n_out"]
        return {"bytes": _w_bytes(c["type"], o, i) + n * (_q8_bytes(i) + 4 * o + ((4 * o + o) if c["res"] else 0)), "flops": 2 * n * i * o}
    if kind == "ffn":
        n, e, f = c["ncols"], c["n_embd"], c["n_ff"]
        return {"bytes": _w_bytes(c["type"], 2 * f, e) + _w_bytes(c["type"], e, f) + 4 * e + n * 10 * e, "flops": 6 * n * e * f}
    if kind == "head":
        n, e, v = c["ncols"], c["n_embd"], c["n_vocab"]
        return {"bytes": _w_bytes("q6_k", v, e) + 4 * e + n * (5 * e + 4 * v), "flops": 2 * n * e * v}
    if kind == "gdn":
        hk, hv, n = c["h_k"], c["h_v"], c["ntok"]
        state, hist = 4 * S * hv * S, 4 * hv * 3 * S * 3
        row = 2 * hk * S + 2 * hv * S + 2 * hv
        return {"bytes": (3 if n == 2 else 2) * (state + hist) + 16 * (2 * hk + hv) * S + n * (4 * row + hv * S * 4 + _q8_bytes(hv * S)),
                "flops": n * hv * S * S * 8}
    if kind == "attn":
        nh, kv, n, ctx = c["n_head"], c["n_kv"], c["ntok"], c["ctx"]
        return {"bytes": ctx * kv * HD * 4 + n * (4 * (2 * nh + 2 * kv) * HD + 4 * nh * HD + _q8_bytes(nh * HD)),
                "flops": 4 * n * nh * HD * (ctx - (n - 1) / 2)}
    e, f, rows, q3 = 4096, 12288, 12352, 10240
    ffn = 3 * e * f
    gdn, att = rows * e + e * e + ffn, q3 * e + e * e + ffn
    trunk, draft, lm = 24 * gdn + 8 * att, 2 * e * e + att, VOCAB * e
    b = 210 / 256
    if kind == "prefill":
        n = c["tokens"]
        return {"bytes": b * (trunk + draft + lm) + 9 * 4096 * n, "flops": 2 * n * (trunk + draft) + 2 * lm + 9 * 2 * n * n * 16 * HD}
    n, ctx = c["tokens"], c["ctx"]
    if c["mode"] == "greedy":
        return {"bytes": n * (b * (trunk + lm) + 8 * 4096 * ctx), "flops": 2 * n * (trunk + lm)}
    r = (n + 1) // 2   # every draft accepted: two tokens a round
    return {"bytes": r * (b * (trunk + draft + 2 * lm) + 9 * 4096 * ctx), "flops": 4 * r * (trunk + draft + 2 * lm)}


def tolerance(case):
    # About four times what the paths measured against the 64-bit results.  A projection of given Q8_1 columns differs
    # by the order of its 32-bit sums (9e-8 of the norm).  Blocks that quantize between two projections differ where a
    # value falls on the other side of an 8-bit code's boundary (up to 9e-5 measured, a code flipped ahead of the up and
    # gate projections).  The recurrent layer and attention: 1.6e-7 and 3.3e-7;
    # fp16 cache rows and Q8_1 bytes may round to the neighbouring value.
    if case["kind"] == "gemv":
        return {"rel": 5e-7, "max": 2e-5}
    if case["kind"] in ("ffn", "head"):
        return {"rel": 4e-4, "max": 5e-3, "differ": 0.01}
    if case["kind"] == "gdn":
        return {"rel": 1e-6, "max": 1e-4, "differ": 2e-3}
    if case["kind"] == "attn":
        return {"rel": 2e-5, "max": 2e-3, "differ": 2e-3}
    # a whole model: a code that flips in one layer travels through all that follow
    return {"rel": 0.03, "max": 0.3, "differ": 0.01}


# ---- 64-bit results, from the formats' and layers' definitions ----------------------------------------------------------
def _q8(x):
    """the values a Q8_1 column stands for: blocks of 32, d = amax / 127 as fp16, codes rounded half away from zero"""
    b = x.to(torch.float32).reshape(*x.shape[:-1], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    v = torch.where(d > 0, b / torch.where(d > 0, d, torch.ones_like(d)), torch.zeros_like(b))
    q = torch.sign(v) * torch.floor(v.abs().double() + 0.5)
    return (q.double() * d.clamp(max=65504).to(torch.float16).double()).reshape(x.shape)


def _rows(type_, w, n_in):
    """[rows, n_in] in float64 of the blocks w: uint8 [rows, row bytes]"""
    per, nbytes = BLOCK[type_]
    b = w.reshape(-1, n_in // per, nbytes)

    def half(lo):
        return b[..., lo:lo + 2].contiguous().view(torch.float16).double()

    if type_ == "q8_0":
        return (half(0) * b[..., 2:].contiguous().view(torch.int8).double()).reshape(-1, n_in)
    if type_ == "q6_k":
        ql, qh = b[..., :128].reshape(*b.shape[:2], 2, 2, 32), b[..., 128:192].reshape(*b.shape[:2], 2, 1, 32)
        sc = b[..., 192:208].contiguous().view(torch.int8).double().reshape(*b.shape[:2], 2, 4, 2, 1)
        lo = torch.cat([ql & 15, ql >> 4], -2)                                       # quarters 0..3 of each half
        hi = torch.cat([(qh >> (2 * k)) & 3 for k in range(4)], -2)
        q = ((lo | (hi << 4)).double() - 32).reshape(*b.shape[:2], 2, 4, 2, 16)
        return (half(208)[..., None, None, None] * sc * q).reshape(-1, n_in)
    s = b[..., 4:16].to(torch.int32)
    sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], -1).double()
    mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1).double()
    qs = b[..., -128:].reshape(*b.shape[:2], 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], -2).reshape(*b.shape[:2], 8, 32)
    if type_ == "q5_k":
        qh = b[..., 16:48].reshape(*b.shape[:2], 1, 32)
        q = q | (torch.cat([(qh >> j) & 1 for j in range(8)], -2) << 4)
    return (half(0)[..., None] * sc[..., None] * q.double() - half(2)[..., None] * mn[..., None]).reshape(-1, n_in)


def _matmul(type_, w, n_in, x):
    """x [cols, n_in] float64 times the matrix, some rows at a time"""
    per, nbytes = BLOCK[type_]
    w = w.reshape(-1, n_in // per * nbytes)
    step = max(1, (1 << 24) // n_in)
    return torch.cat([torch.mm(x, _rows(type_, w[i:i + step], n_in).t().contiguous()) for i in range(0, w.shape[0], step)], 1)


def _partials(y):
    pad = -y.shape[1] % 4
    return torch.nn.functional.pad(y, (0, pad)).reshape(y.shape[0], -1, 4).square().sum(-1)


def _norm(x, w):
    x = x.double()
    return x * w.double() / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)


def _silu(x):
    return x * torch.sigmoid(x)


def _exact_gdn(c, d):
    hk, hv, n = c["h_k"], c["h_v"], c["ntok"]
    d = {k: v.double() for k, v in d.items()}
    q = torch.arange(hv, device="cuda") % hk
    qk, ch = 2 * hk * S, 2 * hk * S + hv * S
    rows = torch.cat([d["x"][:, :qk].reshape(n, 2, hk, S)[:, :, q], d["x"][:, qk:ch].reshape(n, 1, hv, S)], 1)   # [n, 3, hv, S]
    taps = torch.stack([d["conv_w"][:hk * S].reshape(hk, S, 4)[q], d["conv_w"][hk * S:qk].reshape(hk, S, 4)[q],
                        d["conv_w"][qk:].reshape(hv, S, 4)])
    past = d["hist"].permute(3, 1, 0, 2)
    line = torch.cat([past, rows])
    conv = _silu(sum(line[t:t + n] * taps[..., t] for t in range(4)))
    qs, ks = (v / torch.sqrt(v.square().sum(-1, keepdim=True) + EPS) for v in (conv[:, 0], conv[:, 1]))
    z = d["x"][:, ch:ch + hv * S].reshape(n, hv, S)
    beta = torch.sigmoid(d["x"][:, ch + hv * S:ch + hv * S + hv])
    g = torch.exp(torch.nn.functional.softplus(d["x"][:, ch + hv * S + hv:] + d["dt"]) * d["ssm_a"])
    st, ys = d["state"], []
    for t in range(n):
        kv = (st * ks[t].t()[..., None]).sum(0)
        delta = (conv[t, 2] - g[t][:, None] * kv) * beta[t][:, None]
        st = g[t][None, :, None] * st + ks[t].t()[..., None] * delta[None]
        o = (st * qs[t].t()[..., None]).sum(0) / math.sqrt(S)
        ys.append(o / torch.sqrt(o.square().mean(-1, keepdim=True) + EPS) * d["gamma"] * _silu(z[t]))
    return {"y": torch.stack(ys).reshape(n, -1), "q8": None, "state": st, "hist": line[-3:].permute(2, 1, 3, 0).contiguous()}


def _rope(x, pos):
    """NEOX rotation of the first ROT dims of [n, heads, HD] at positions [n]"""
    half = ROT // 2
    ang = pos.double()[:, None, None] * THETA ** (-2.0 * torch.arange(half, device="cuda", dtype=torch.float64) / ROT)
    a, b = x[..., :half], x[..., half:ROT]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos(), x[..., ROT:]], -1)


def _exact_attn(c, d):
    nh, kv, n, ctx = c["n_head"], c["n_kv"], c["ntok"], c["ctx"]
    pos = torch.arange(ctx - n, ctx, device="cuda")
    qg = d["q3"][:, :nh * 2 * HD].reshape(n, nh, 2, HD)
    k, v = d["q3"][:, nh * 2 * HD:].reshape(n, 2, kv, HD).unbind(1)
    q = _rope(_norm(qg[:, :, 0], d["qn"]), pos)
    k = _rope(_norm(k, d["kn"]), pos)
    kc, vc = d["kc"][:ctx].clone(), d["vc"][:ctx].clone()
    kc[ctx - n:], vc[ctx - n:] = k.to(torch.float16), v.to(torch.float16)
    y = torch.empty(n, nh, HD, dtype=torch.float64, device="cuda")
    seen = torch.arange(ctx, device="cuda")[None] <= pos[:, None]
    for h in range(nh):
        kh, vh = kc[:, h // (nh // kv)].double().contiguous(), vc[:, h // (nh // kv)].double().contiguous()
        sc = torch.mm(q[:, h].contiguous(), kh.t().contiguous()) / math.sqrt(HD)
        y[:, h] = torch.mm(torch.softmax(sc.masked_fill(~seen, -math.inf), -1), vh)
    y = (y * torch.sigmoid(qg[:, :, 1].double())).reshape(n, -1)
    return {"y": y, "q8": None, "k": kc[ctx - n:].double(), "v": vc[ctx - n:].double()}


def exact(case, seed):
    c, kind = case, case["kind"]
    g = _gen(seed)
    if kind == "gemv":
        w, x, res = _gemv_inputs(c, g)
        y = _matmul(c["type"], w, c["n_in"], _q8(x))
        if not c["res"]:
            return {"y": y}
        y = y + res.double()
        return {"y": y, "part": _partials(y)}
    if kind == "ffn":
        ug, down, norm, x = _ffn_inputs(c, g)
        h = _matmul(c["type"], ug, c["n_embd"], _q8(_norm(x, norm)))
        up, gate = h[:, :c["n_ff"]], h[:, c["n_ff"]:]
        y = x.double() + _matmul(c["type"], down, c["n_ff"], _q8(_silu(gate) * up))
        return {"y": y, "part": _partials(y)}
    if kind == "head":
        w, norm, x = _head_inputs(c, g)
        y = _matmul("q6_k", w, c["n_embd"], _q8(_norm(x, norm)))
        return {"logits": y, "ids": None, "top": None, "topv": torch.sort(y[0], descending=True)[0][:TOPK].clone()}
    if kind == "gdn":
        return _exact_gdn(c, _gdn_inputs(c, g))
    if kind == "attn":
        return _exact_attn(c, _attn_inputs(c, g))
    return None
