"""The work this framework is measured at: prompts and decode steps of its decoders through their public entry points, from
one row of a small decoder to packed prompts of a wide one, and the cached attention operators by themselves.

A case is a dict of plain values.  "path" says what a pass is:

  prefill   packed prompts in, logits and filled caches out
  decode    greedy steps of a resident session over caches that an earlier prefill left (a serving loop's steady state)
  serve     prefill, then greedy steps of a resident session (one request from start to end)
  sample    generate(): prefill, then sampled steps
  portions  slots continued by portions of prompts and single tokens (continuous batching)
  attend    K/V append and cached attention of one decode step, layer by layer, through the backend's operators

and "arch" whose decoder it is.  Weights keep the variance of what passes through them, and the LM head is a permutation of the
embedding, so that predictions are as peaked as a trained model's and no greedy pick is a tie.  (Girirax has no head of its
own: it predicts the token that it was given.)
"""
import ctypes
import importlib.util
import json
import math
import os
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _package():
    """The repository's package; its folder's name is not one that an import statement could hold."""
    name = "gradients_c_amd"
    if name not in sys.modules:
        path = os.path.join(ROOT, "gradients.c_amd", "__init__.py")
        spec = importlib.util.spec_from_file_location(name, path, submodule_search_locations=[os.path.dirname(path)])
        sys.modules[name] = module = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(module)
    return sys.modules[name]


def _decoders():
    _package()
    from gradients_c_amd import decoder
    return decoder


# ---- the cases ------------------------------------------------------------------------------------------------------

#: the two gpt_lm decoders of bench.py, the wide one with four of its 24 layers (a layer's work does not depend on the others')
SMALL = dict(arch="gpt", vocab=2048, layers=3, heads=8, head_dim=64, ff=1536)
WIDE = dict(arch="gpt", vocab=32768, layers=4, heads=16, head_dim=128, ff=5632)
#: layer lists of perf_layer_lists.py with fewer layers
GIRIRAX = dict(arch="girirax", vocab=32768, layers=4, dtype="bfloat16")
BONATAR = dict(arch="bonatar", vocab=32768, layers=4, dtype="bfloat16", experts=16)


def listed():
    return [
        # one user, one short question to the small decoder: everything is launches and latency
        dict(SMALL, name="gpt-serve-1", path="serve", batch=1, low=32, high=32, new=64, window=0, block=0),
        # the throughput of a server of the small decoder, caches nearly full, one new token per row and step
        dict(SMALL, name="gpt-decode-64", path="decode", batch=64, low=300, high=479, new=32, window=0, block=0),
        # the reference program's own use: sampled text, attention through its default window of 256 tokens
        dict(SMALL, name="gpt-sample-16", path="sample", batch=16, low=20, high=400, new=48, window=256, block=0),
        # the small decoder's packed prompts under its second architecture: attention over picked blocks of 128 tokens
        dict(SMALL, name="blocks-prefill-8", path="prefill", batch=8, low=500, high=4096, new=0, window=0, block=128),
        # long ragged conversations of a wide decoder: weights and caches stream from HBM
        dict(WIDE, name="wide-decode-16", path="decode", batch=16, low=1024, high=4000, new=16, window=0, block=0),
        # ragged prompts of a wide decoder: the matrix cores' work
        dict(WIDE, name="wide-prefill-32", path="prefill", batch=32, low=64, high=2048, new=0, window=0, block=0),
        # a decode step's attention over very uneven caches, as an engine that brings its own projections calls it
        dict(name="attend-32", path="attend", arch="operators", layers=4, batch=32, heads=8, kv_heads=8, head_dim=64, low=1, high=4095,
             window=0),
        # prompts of a decoder with recurrent and latent-attention layers
        dict(GIRIRAX, name="girirax-prefill-16", path="prefill", width=2048, ff=5632, kv_rank=512, batch=16, low=64, high=2048, new=0),
        # many short requests to it, from prompt to answer: state and latent caches of 64 rows
        dict(GIRIRAX, name="girirax-serve-64", path="serve", width=1024, ff=2816, kv_rank=256, batch=64, low=40, high=300, new=48),
        # the same in 32 bits, prompts in portions between other sequences' single tokens: a replay that has to be exact
        dict(GIRIRAX, name="girirax-portions-f32", path="portions", width=1024, ff=2816, kv_rank=256, batch=6, low=100, high=500,
             new=0, rounds=6, portion=128, layers=2, dtype="float32"),
        # long prompts of a decoder with grouped attention and experts, wide enough for whole tiles of every expert
        dict(BONATAR, name="bonatar-prefill-12", path="prefill", width=4096, layers=2, ff=11264, experts=8, heads=32, kv_heads=8,
             chunk=8192, batch=12, low=500, high=4000, new=0),
        # conversations with it: few rows per expert, chunks of 2048 positions
        dict(BONATAR, name="bonatar-serve-16", path="serve", width=2048, ff=5632, heads=16, kv_heads=4, chunk=2048, batch=16, low=300,
             high=1900, new=64),
    ]


def _between(rng, low, high):
    """A whole number, spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _gpt_draw(rng, path):
    wide = rng.random() < 0.4
    if wide:
        c = dict(WIDE, layers=rng.randint(1, 4), vocab=_between(rng, 4000, 32768), heads=rng.choice([8, 12, 16]))
    else:
        c = dict(SMALL, layers=rng.randint(1, 4), vocab=_between(rng, 300, 8192), heads=rng.randint(4, 12))
    c.update(path=path, window=rng.choice([0, 0, 0, 256]), block=0, new=0)
    c["ff"] = (c["heads"] * c["head_dim"] * rng.randint(20, 32) // 10) // 32 * 32
    if path == "prefill":
        if not wide and rng.random() < 0.4:
            c.update(block=128, window=0)
        c.update(batch=_between(rng, 1, 32), low=_between(rng, 5, 200))
        c["high"] = max(c["low"], _between(rng, 100, 2048 if wide else 4096))
    elif path == "decode":
        c.update(batch=_between(rng, 1, 32 if wide else 96), low=_between(rng, 10, 1000), new=rng.randint(8, 24))
        c["high"] = max(c["low"], _between(rng, 100, 3000 if wide else 1000))
    else:
        c.update(layers=min(c["layers"], 3), batch=_between(rng, 1, 24), low=_between(rng, 5, 40), new=rng.randint(16, 64))
        c["high"] = max(c["low"], _between(rng, 30, 400))
    return c


def draw(rng):
    kind = rng.choice(["gpt prefill", "gpt prefill", "gpt decode", "gpt decode", "gpt serve", "gpt sample", "attend", "girirax", "bonatar",
                       "girirax", "bonatar", "portions"])
    if kind.startswith("gpt"):
        return _gpt_draw(rng, kind.split()[1])
    if kind == "attend":
        kv_heads = rng.choice([1, 2, 4, 8, 8, 16])
        low = _between(rng, 1, 1000)
        return dict(path="attend", arch="operators", layers=rng.randint(1, 4), batch=_between(rng, 1, 64), heads=kv_heads * rng.choice([1, 1, 4]),
                    kv_heads=kv_heads, head_dim=rng.choice([64, 128]), low=low, high=max(low, _between(rng, 50, 4095)),
                    window=rng.choice([0, 0, 0, 256, 1000]))
    width = rng.choice([512, 1024, 2048])
    if kind == "portions":
        c = dict(rng.choice([GIRIRAX, BONATAR]), dtype=rng.choice(["bfloat16", "float32"]), path="portions", layers=2, width=width // 2,
                 batch=rng.randint(1, 8), low=_between(rng, 20, 100), high=_between(rng, 100, 500), new=0, rounds=rng.randint(3, 7),
                 portion=_between(rng, 16, 256), vocab=_between(rng, 500, 8000))
    else:
        c = dict(GIRIRAX if kind == "girirax" else BONATAR, path=rng.choice(["prefill", "serve"]), layers=rng.choice([2, 4]), width=width,
                 batch=_between(rng, 1, 32), low=_between(rng, 10, 300), vocab=_between(rng, 500, 32768), new=0)
        c["high"] = max(c["low"], _between(rng, 100, 1500))
        if c["path"] == "serve":
            c.update(new=rng.randint(16, 48), batch=_between(rng, 1, 64), high=max(c["low"], c["high"] // 4))
    c["ff"] = c["width"] * rng.randint(16, 28) // 10 // 64 * 64
    if c["arch"] == "girirax":
        c["kv_rank"] = rng.choice([128, 256, 512])
    else:
        heads = c["width"] // 128
        c.update(heads=heads, kv_heads=max(1, heads // 4), chunk=rng.choice([512, 2048, 8192]), experts=rng.choice([4, 16]))
    return c


# ---- inputs from a seed -----------------------------------------------------------------------------------------------

def _lengths(case, seed):
    rng = np.random.default_rng([seed, 1])
    lens = rng.integers(case["low"], case["high"] + 1, case["batch"])
    return lens, np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)


def _tokens(case, seed, n, stream=2):
    return np.random.default_rng([seed, stream]).integers(0, case["vocab"], n).astype(np.int32)


def _successor(case, seed):
    """What the model says behind a token."""
    if case["arch"] == "girirax":
        return np.arange(case["vocab"])
    return np.random.default_rng([seed, 3]).permutation(case["vocab"])


def _width(case):
    return case["width"] if "width" in case else case["heads"] * case["head_dim"]


class _Random:
    """Tensors on the GPU, drawn one after the other from a seed."""

    def __init__(self, seed, dtype):
        self.g, self.dtype = torch.Generator("cuda").manual_seed(seed), dtype

    def normal(self, *shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(self.dtype)

    def uniform(self, n, low, high):
        return (torch.rand(n, generator=self.g, device="cuda") * (high - low) + low).to(self.dtype)


def _head_of(embed, case, seed, peak=14.0):
    """The head that says _successor: logits of about `peak` for it, about 0 +- peak / sqrt(width) for the others."""
    head = torch.empty_like(embed)
    head[torch.from_numpy(_successor(case, seed)).cuda()] = (embed.float() * (peak / _width(case))).to(embed.dtype)
    return head


def _gpt_weights(case, seed):
    """name, layer -> F16 tensor, as gd_gpt_decoder_tensor names them."""
    r, D, F, w = _Random(seed, torch.float16), _width(case), case["ff"], {}
    w["embed", 0] = r.normal(case["vocab"], D)
    w["lm_head", 0] = _head_of(w["embed", 0], case, seed)
    w["lm_bias", 0] = r.normal(case["vocab"], std=0.1)
    w["final_norm", 0] = r.normal(D, std=0.1, mean=1.0)
    for l in range(case["layers"]):
        w["attn_norm", l], w["mlp_norm", l] = r.normal(D, std=0.1, mean=1.0), r.normal(D, std=0.1, mean=1.0)
        w["w_qkv", l], w["b_qkv", l] = r.normal(3 * D, D, std=D ** -0.5), r.normal(3 * D, std=0.1)
        w["w_attn", l], w["b_attn", l] = r.normal(D, D, std=0.5 * D ** -0.5), r.normal(D, std=0.05)
        w["w_upgate", l], w["b_upgate", l] = r.normal(2 * F, D, std=D ** -0.5), r.normal(2 * F, std=0.1)
        w["w_down", l], w["b_down", l] = r.normal(F, D, std=0.5 * F ** -0.5), r.normal(D, std=0.05)
    return w


def _girirax_config(c):
    W = c["width"]
    ssm = {"heads": W // 32, "vdim": 64, "state": 128, "groups": 1, "norm_groups": 1, "conv": 4}
    latent = {"heads": max(1, W // 128), "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": W * 3 // 8, "kv_rank": c["kv_rank"],
              "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}
    return {"architecture": "Girirax", "vocab": c["vocab"], "width": W, "norm": {"eps": 1e-5}, "residual_mult": 0.5,
            "embedding": {"scale": 4.0},
            "layers": [{"type": "mamba2" if i % 2 == 0 else "latent_attention", "mixer": ssm if i % 2 == 0 else latent,
                        "mlp": {"kind": "dense", "ff": c["ff"]}} for i in range(c["layers"])]}


def _bonatar_config(c):
    mixer = {"heads": c["heads"], "kv_heads": c["kv_heads"], "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": c["chunk"]},
             "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "original": 8192, "fast": 32.0, "slow": 1.0}}}
    mlps = [{"kind": "dense", "ff": c["ff"] * 3 // 2},
            {"kind": "moe", "router": {"experts": c["experts"], "top": 2}, "expert": {"ff": c["ff"] // 4, "limit": 7.0},
             "shared": {"ff": c["ff"] // 2, "limit": 7.0}}]
    return {"architecture": "Bonatar", "vocab": c["vocab"], "width": c["width"], "norm": {"eps": 1e-5}, "embedding": {"scale": 4.0},
            "layers": [{"type": "attention", "mixer": mixer, "mlp": mlps[i % 2]} for i in range(c["layers"])]}


def _config(case):
    return (_girirax_config if case["arch"] == "girirax" else _bonatar_config)(case)


def _list_weights(case, seed):
    """name -> BF16 tensor (tables: I32), as model.safetensors holds them."""
    r, W, w, cfg = _Random(seed, torch.bfloat16), case["width"], {}, _config(case)

    def mat(name, rows, cols, gain=1.0):
        w[name] = r.normal(rows, cols, std=gain * cols ** -0.5)

    first = 0.0 if case["arch"] == "bonatar" else 1.0  # Bonatar's norm weights lie around zero
    w["embed"] = r.normal(case["vocab"], W, std=0.25)
    if case["arch"] == "bonatar":
        w["head"] = _head_of(w["embed"], case, seed, 56.0)
    w["final.norm"] = r.normal(W, std=0.1, mean=first)
    for i, l in enumerate(cfg["layers"]):
        p, m, f = "l%d." % i, l["mixer"], l["mlp"]
        w[p + "norm1"], w[p + "norm2"] = r.normal(W, std=0.1, mean=first), r.normal(W, std=0.1, mean=first)
        if l["type"] == "mamba2":
            inner, ch = m["heads"] * m["vdim"], m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"]
            mat(p + "mix.in", inner + ch + m["heads"], W)
            w[p + "mix.conv"], w[p + "mix.conv.b"] = r.normal(ch, m["conv"], std=0.5), r.normal(ch, std=0.1)
            w[p + "mix.dt_bias"], w[p + "mix.A_log"] = r.uniform(m["heads"], -4.6, -2.3), r.uniform(m["heads"], 0.0, 2.7)
            w[p + "mix.D"], w[p + "mix.norm"] = r.uniform(m["heads"], 0.5, 1.5), r.normal(inner, std=0.1, mean=1.0)
            mat(p + "mix.o", W, inner)
        elif l["type"] == "latent_attention":
            H = m["heads"]
            mat(p + "mix.dq", m["q_rank"], W)
            mat(p + "mix.uq", H * (m["dim"] + m["rot_dim"]), m["q_rank"])
            mat(p + "mix.dkv", m["kv_rank"] + m["rot_dim"], W)
            mat(p + "mix.uk", H * m["dim"], m["kv_rank"])
            mat(p + "mix.uv", H * m["vdim"], m["kv_rank"])
            w[p + "mix.dq.norm"], w[p + "mix.dkv.norm"] = r.normal(m["q_rank"], std=0.1, mean=1.0), r.normal(m["kv_rank"], std=0.1, mean=1.0)
            mat(p + "mix.g", H * m["vdim"], W)
            mat(p + "mix.o", W, H * m["vdim"])
        else:
            mat(p + "mix.q", m["heads"] * m["dim"], W)
            mat(p + "mix.k", m["kv_heads"] * m["dim"], W)
            mat(p + "mix.v", m["kv_heads"] * m["vdim"], W)
            mat(p + "mix.g", m["heads"], W)
            mat(p + "mix.o", W, m["heads"] * m["vdim"], 0.5)
        if case["arch"] == "girirax":
            for part, rows, cols in (("gate", f["ff"], W), ("up", f["ff"], W), ("down", W, f["ff"])):
                mat(p + "mlp." + part, rows, cols)
                w[p + "mlp." + part + ".b"] = r.normal(rows, std=0.1)
        elif f["kind"] == "dense":
            mat(p + "mlp.up", f["ff"], W)
            mat(p + "mlp.down", W, f["ff"], 0.4)
        else:
            for name, ff in [("e%d." % e, f["expert"]["ff"]) for e in range(f["router"]["experts"])] + [("shared.", f["shared"]["ff"])]:
                mat(p + "mlp." + name + "gate", ff, W)
                mat(p + "mlp." + name + "up", ff, W)
                mat(p + "mlp." + name + "down", W, ff, 0.4)
            picks = torch.rand(case["vocab"], f["router"]["experts"], generator=r.g, device="cuda").argsort(1)[:, :f["router"]["top"]]
            w[p + "mlp.table"] = picks.to(torch.int32)
    return w


def _save(folder, config, weights):
    """config.json and model.safetensors."""
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump(config, f)
    header, at = {}, 0
    for name, t in weights.items():
        n = t.numel() * t.element_size()
        header[name] = {"dtype": "I32" if t.dtype == torch.int32 else "BF16", "shape": list(t.shape), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(header).encode()
    with open(os.path.join(folder, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for t in weights.values():
            f.write(t.contiguous().view(torch.uint8).cpu().numpy().data)


# ---- what a user's program holds -----------------------------------------------------------------------------------------

_KINDS = {1: ("<i2", torch.float16), 2: ("<i2", torch.bfloat16), 3: ("<f4", torch.float32)}


class _Owner:
    """A decoder, or a backend and its buffers, closed when nobody holds them or memory of theirs any more."""

    def __init__(self, held):
        self.held = held

    def __del__(self):
        self.held.close()


class _Region:
    """Device memory of the library, for torch.as_tensor: the tensor keeps it, and it keeps the memory's owner."""

    def __init__(self, pointer, shape, kind, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": _KINDS[kind][0], "data": (pointer, False), "version": 3}


def _seen(owner, buffer, offset, shape, kind):
    """The library's memory as a torch tensor that shares it."""
    base = _package().lib().gd_backend_buffer_device_ptr(buffer)
    return torch.as_tensor(_Region(base + offset, shape, kind, owner), device="cuda").view(_KINDS[kind][1])


class State:
    owner = decoder = backend = None


def _decoder_tensor(s, name, layer=0):
    t = s.decoder.tensor(name, layer)
    return _seen(s.owner, t.storage.buffer, t.storage.offset + t.view_offset, [t.shape[i] for i in range(t.rank)], t.dtype)


def _max_seq(case):
    return -(-(case["high"] + case["new"] + 1) // 64) * 64


def _open_gpt(s, case, seed, rows):
    D = _decoders()
    cfg = D.gpt_config(case["vocab"], _width(case), case["layers"], case["heads"], case["head_dim"], case["ff"], _max_seq(case),
                       case["batch"], window=case["window"], tie_lm_head=False, seed=seed,
                       minimax_m3=(case["block"], 4, 1, 1) if case["block"] else None)
    s.decoder = D.GptDecoder(cfg, max_prefill_tokens=rows)
    s.owner = _Owner(s.decoder)
    for (name, layer), t in _gpt_weights(case, seed).items():
        s.decoder.write_tensor(name, layer, t.cpu().numpy())
        if name == "w_down":
            s.decoder.write_tensor("w_down_t", layer, t.t().contiguous().cpu().numpy())
    for l in range(case["layers"]):
        s.outputs["k%d" % l], s.outputs["v%d" % l] = _decoder_tensor(s, "k_cache", l), _decoder_tensor(s, "v_cache", l)


def _open_list(s, case, seed, rows):
    D = _decoders()
    folder = tempfile.mkdtemp()
    try:
        _save(folder, _config(case), _list_weights(case, seed))
        model = D.Model(folder)
        try:
            s.decoder = model.decoder(max_seq=_max_seq(case), batch=case["batch"], max_step_tokens=max(rows, case["batch"]),
                                      compute=case["dtype"])
        finally:
            model.close()
    finally:
        shutil.rmtree(folder)
    s.owner = _Owner(s.decoder)
    for l, layer in enumerate(_config(case)["layers"]):
        for name in {"mamba2": ["states"], "latent_attention": ["cache"], "attention": ["k_cache", "v_cache"]}[layer["type"]]:
            s.outputs["%s%d" % (name, l)] = _decoder_tensor(s, name, l)


def _portions(case, seed):
    """The calls of a "portions" pass: per round, sequence -> (first, count) of its tokens."""
    lens, _ = _lengths(case, seed)
    rng = np.random.default_rng([seed, 5])
    held, rounds = np.zeros(case["batch"], int), []
    for _ in range(case["rounds"]):
        take = np.where(held < lens, np.minimum(lens - held, rng.integers(1, case["portion"] + 1, case["batch"])), 1)
        rounds.append({b: (int(held[b]), int(take[b])) for b in range(case["batch"])})
        held += take
    return rounds, held


def _prepare_attend(s, case, seed):
    gd = _package()
    s.backend = gd.Backend()
    s.owner = _Owner(s.backend)
    B, H, G, D = case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    T = _attend_rows(case)
    s.arena = s.backend.buffer(case["layers"] * (2 * B * T * G * D * 2 + 2 * B * (H + G) * D * 2 + (1 << 12)) + (1 << 16))
    inputs, s.calls = _attend_inputs(case, seed), []
    s.pos = s.arena.from_numpy(inputs["pos"])
    for l in range(case["layers"]):
        t = {}
        for name in ("k", "v", "q", "kn", "vn"):
            source = inputs[name][l]
            t[name] = s.arena.alloc(source.shape, gd.F16)
            _seen(s.owner, s.arena.handle, t[name].offset, source.shape, gd.F16).copy_(source)
        t["out"] = s.arena.alloc((B, 1, H, D), gd.F16)
        s.outputs["k%d" % l] = _seen(s.owner, s.arena.handle, t["k"].offset, t["k"].shape, gd.F16)
        s.outputs["v%d" % l] = _seen(s.owner, s.arena.handle, t["v"].offset, t["v"].shape, gd.F16)
        s.outputs["out%d" % l] = _seen(s.owner, s.arena.handle, t["out"].offset, t["out"].shape, gd.F16)
        s.calls.append({n: x.view() for n, x in t.items()})
    s.pos_view = s.pos.view()
    s.append_args, s.decode_args = gd.KvAppendArgs(0), gd.SdpaDecodeArgs(D ** -0.5, case["window"], 0, 0)
    torch.cuda.synchronize()
    s.backend.scope_begin()


def _attend_rows(case):
    return -(-(case["high"] + 1) // 256) * 256


def _attend_inputs(case, seed):
    r = _Random(seed, torch.float16)
    B, H, G, D, T, L = case["batch"], case["heads"], case["kv_heads"], case["head_dim"], _attend_rows(case), range(case["layers"])
    lens, _ = _lengths(case, seed)
    return {"pos": lens.astype(np.int32), "k": [r.normal(B, T, G, D) for _ in L], "v": [r.normal(B, T, G, D) for _ in L],
            "q": [r.normal(B, 1, H, D) for _ in L], "kn": [r.normal(B, 1, G, D) for _ in L], "vn": [r.normal(B, 1, G, D) for _ in L]}


def prepare(case, seed):
    s = State()
    s.case, s.outputs = case, {}
    if case["path"] == "attend":
        _prepare_attend(s, case, seed)
        return s
    s.lens, s.cu = _lengths(case, seed)
    if case["path"] == "portions":
        s.rounds, held = _portions(case, seed)
        rows = max(sum(n for _, n in r.values()) for r in s.rounds)
        s.ids = [_tokens(case, seed, int(n), 100 + b) for b, n in enumerate(held)]
    else:
        rows = int(s.cu[-1])
        s.ids = _tokens(case, seed, rows)
    (_open_gpt if case["arch"] == "gpt" else _open_list)(s, case, seed, rows)
    if case["path"] == "decode":
        s.decoder.prefill(s.ids, s.cu, want_logits=False)
        s.first = _tokens(case, seed, case["batch"], 4)
    if case["path"] in ("decode", "serve", "sample"):
        s.outputs["logits"] = _decoder_tensor(s, "last_logits")
    torch.cuda.synchronize()
    return s


# ---- one pass ------------------------------------------------------------------------------------------------------------

def _greedy(d, first, steps):
    d.resident_begin(first, steps, keep_logits=True)
    d.resident_run(steps - 1)
    return d.resident_end()


def run(state):
    case, d, out = state.case, state.decoder, dict(state.outputs)
    if case["path"] == "prefill":
        out["logits"], out["next"], out["gap"] = d.prefill(state.ids, state.cu)
    elif case["path"] == "decode":
        d.positions[:] = state.lens
        out["tokens"], out["gap"] = _greedy(d, state.first, case["new"])
    elif case["path"] == "serve":
        _, first, _ = d.prefill(state.ids, state.cu, want_logits=False)
        out["tokens"], out["gap"] = _greedy(d, first, case["new"])
    elif case["path"] == "sample":
        out["tokens"] = d.generate(state.ids, state.cu, case["new"], temperature=0.8, min_p=0.05, repetition_penalty=1.3,
                                   logits_softcap=20.0, rng_state=11)
    elif case["path"] == "portions":
        slots = [d.acquire() for _ in range(case["batch"])]
        for i, r in enumerate(state.rounds):
            counts = [n for _, n in r.values()]
            out["logits%d" % i] = d.extend({slots[b]: state.ids[b][at:at + n] for b, (at, n) in r.items()}, want=np.cumsum(counts) - 1)
        for slot in slots:
            d.release(slot)
    else:
        call, by = state.backend.call, ctypes.byref
        for v in state.calls:
            for status in (call("gd_backend_kv_cache_append_positions", v["k"], v["v"], state.pos_view, v["kn"], v["vn"], by(state.append_args)),
                           call("gd_backend_sdpa_decode_positions", v["q"], v["k"], v["v"], state.pos_view, v["out"], by(state.decode_args))):
                if status != 0:
                    raise RuntimeError("status %d" % status)
    return out


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------

def _layer_sizes(case):
    """Per layer: (weights a token multiplies with, weights that a step of many rows reads, values a token leaves in the caches,
    operations of attention per visible pair, operations of a recurrence per token, F32 state values of a sequence)."""
    W = _width(case)
    if case["arch"] == "gpt":
        n = 4 * W * W + 3 * W * case["ff"]
        return [(n, n, 2 * W, 4 * W, 0, 0)] * case["layers"]
    sizes = []
    for l in _config(case)["layers"]:
        m, f = l["mixer"], l["mlp"]
        if l["type"] == "mamba2":
            inner, bc = m["heads"] * m["vdim"], 2 * m["groups"] * m["state"]
            mixer, keep, pair, token, state = W * (3 * inner + bc + m["heads"]), 0, 0, 4 * inner * m["state"], inner * m["state"]
        elif l["type"] == "latent_attention":
            H, keep, token, state = m["heads"], m["kv_rank"] + m["rot_dim"], 0, 0
            mixer = W * (m["q_rank"] + keep + 2 * H * m["vdim"]) + m["q_rank"] * H * (m["dim"] + m["rot_dim"]) + \
                m["kv_rank"] * H * (m["dim"] + m["vdim"])
            pair = 2 * H * (m["dim"] + m["rot_dim"] + m["vdim"])
        else:
            H, G, token, state = m["heads"], m["kv_heads"], 0, 0
            mixer, keep, pair = W * (2 * H * 128 + 2 * G * 128 + H), 2 * G * 128, 4 * H * 128
        if f["kind"] == "moe":
            e, shared = 3 * W * f["expert"]["ff"], 3 * W * f["shared"]["ff"]
            used, held = f["router"]["top"] * e + shared, f["router"]["experts"] * e + shared
        else:
            used = held = W * f["ff"] * (3 if case["arch"] == "girirax" else 2)
        sizes.append((mixer + used, mixer + held, keep, pair, token, state))
    return sizes


def _visible(case, first, count):
    """Keys that the rows first .. first + count - 1 of a sequence see in a layer's attention."""
    if case["arch"] == "bonatar" and case["chunk"] < first + count:
        return int(sum(i % case["chunk"] + 1 for i in range(first, first + count)))
    if case["arch"] == "gpt" and case["window"]:
        return int(sum(min(i + 1, case["window"]) for i in range(first, first + count)))
    if case["arch"] == "gpt" and case["block"]:
        return int(sum(min(i + 1, 3 * case["block"] + i % case["block"] + 1) for i in range(first, first + count)))
    return count * first + count * (count + 1) // 2


def _pass_work(case, first, count, picks):
    """One forward over count[b] rows behind first[b] rows of each sequence, with the logits of `picks` rows."""
    es, W = 4 if case.get("dtype") == "float32" else 2, _width(case)
    rows, n_bytes, flops = sum(count), 0, 0
    pairs = sum(_visible(case, f, c) for f, c in zip(first, count))
    for used, held, keep, pair, token, state in _layer_sizes(case):
        if held > used and case["arch"] == "bonatar":  # the experts that these rows choose
            held = used + (held - used) * (1 - (1 - 1 / case["experts"]) ** max(0, 2 * rows - 2))
        n_bytes += es * held + es * keep * (sum(first) + rows) + 8 * state * len(count)
        flops += 2 * used * rows + pair * pairs + token * rows
    n_bytes += es * (case["vocab"] * W + min(rows, case["vocab"]) * W + picks * case["vocab"])
    return n_bytes, flops + 2 * picks * W * case["vocab"]


def work(case):
    lens = _lengths(case, 0)[0].tolist()
    B, total = case["batch"], [0.0, 0.0]

    def add(first, count, picks):
        for i, x in enumerate(_pass_work(case, first, count, picks)):
            total[i] += x

    if case["path"] == "attend":
        seen = sum(min(n + 1, case["window"] or n + 1) for n in lens)
        row = case["kv_heads"] * case["head_dim"]
        total = [case["layers"] * (4 * row * (seen + B) + 4 * B * case["heads"] * case["head_dim"]),
                 case["layers"] * 4 * seen * case["heads"] * case["head_dim"]]
    elif case["path"] == "portions":
        for r in _portions(case, 0)[0]:
            add([at for at, _ in r.values()], [n for _, n in r.values()], B)
    else:
        if case["path"] != "decode":
            add([0] * B, lens, B)
        steps = case["new"] - (1 if case["path"] == "sample" else 0)
        for i in range(steps if case["path"] != "prefill" else 0):
            add([n + i for n in lens], [1] * B, B)
    return {"bytes": float(total[0]), "flops": float(total[1])}


def tolerance(case):
    """About four times what the outputs differ from exact() by; other orders of the sums in a layer move the roundings of all
    that follow, so that two correct passes are as far apart as each is from exact()."""
    if case.get("dtype") == "float32":
        return {"rel": 1e-5, "max": 1e-3}                    # 1.2e-6
    if case["path"] == "attend":
        return {"rel": 1e-3, "max": 1e-2}                    # 2.1e-4: F16 outputs of F32 sums
    if case["arch"] == "gpt" and case["block"]:
        return {"rel": 1e-2, "max": 0.5, "differ": 0.002}    # a rounding can change which block is picked
    if case["arch"] == "gpt":
        return {"rel": 3e-3, "max": 0.05, "differ": 0.002}   # 8e-4: F16 between the operators
    return {"rel": 2e-2, "max": 0.3, "differ": 0.002}        # 5e-3: BF16 between the operators


# ---- the same in 64 bits ------------------------------------------------------------------------------------------------------

def _rms(x, weight, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * weight


def _rotated(x, positions, freq, mult=1.0, neighbours=False):
    """x [T, H, D]; pairs (i, i + D/2), or (2i, 2i + 1)."""
    angle = positions[:, None, None] * freq
    cos, sin, n = angle.cos() * mult, angle.sin() * mult, len(freq)
    if neighbours:
        u, v = x[..., 0::2], x[..., 1::2]
        return torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2)
    u, v = x[..., :n], x[..., n:]
    return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)


def _powers(base, dims):
    return torch.tensor(base, dtype=torch.float64, device="cuda") ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device="cuda") / dims)


def _attention(q, k, v, scale, window=0, chunk=0):
    """q [T, H, D] of the last T positions, k [S, G, D], v [S, G, E] -> [T, H, E], a slice of queries at a time."""
    H, G, S, T, out = q.shape[1], k.shape[1], k.shape[0], q.shape[0], []
    k, v = (x.repeat_interleave(H // G, 1).transpose(0, 1) for x in (k, v))
    j = torch.arange(S, device="cuda")
    for at in range(0, T, 1024):
        part = q[at:at + 1024].transpose(0, 1)
        i = torch.arange(S - T + at, S - T + at + part.shape[1], device="cuda")[:, None]
        seen = (j <= i) & ((i - j) < (window or S)) & ((i // (chunk or S + 1)) == (j // (chunk or S + 1)))
        p = ((part @ k.transpose(1, 2)) * scale).masked_fill(~seen, -math.inf).softmax(-1)
        out.append((p @ v).transpose(0, 1))
    return torch.cat(out)


def _gpt_exact(case, seed, ids, cu):
    """Packed sequences -> (the last norm's output of every row, the layers' keys, the layers' values)."""
    w = {k: v.double() for k, v in _gpt_weights(case, seed).items()}
    H, D, F = case["heads"], case["head_dim"], case["ff"]
    runs, keys, values = [(int(a), int(b)) for a, b in zip(cu[:-1], cu[1:])], [], []
    x, freq = w["embed", 0][torch.from_numpy(ids).cuda().long()], _powers(10000.0, D)
    pos = torch.cat([torch.arange(b - a, device="cuda", dtype=torch.float64) for a, b in runs])
    for l in range(case["layers"]):
        qkv = (_rms(x, w["attn_norm", l], 1e-5) @ w["w_qkv", l].t() + w["b_qkv", l]).view(-1, 3, H, D)
        q, k, v = _rotated(qkv[:, 0], pos, freq), _rotated(qkv[:, 1], pos, freq), qkv[:, 2]
        keys.append(k)
        values.append(v)
        a = torch.cat([_attention(q[i:j], k[i:j], v[i:j], D ** -0.5, case["window"]) for i, j in runs]).reshape(-1, H * D)
        x = x + a @ w["w_attn", l].t() + w["b_attn", l]
        up = _rms(x, w["mlp_norm", l], 1e-5) @ w["w_upgate", l].t() + w["b_upgate", l]
        x = x + (up[:, :F] * torch.nn.functional.silu(up[:, F:])) @ w["w_down", l] + w["b_down", l]
    return _rms(x, w["final_norm", 0], 1e-5), keys, values, lambda h: h @ w["lm_head", 0].t() + w["lm_bias", 0]


def _ssm_exact(h, w, p, m, eps, runs):
    inner, N, H, P = m["heads"] * m["vdim"], m["state"], m["heads"], m["vdim"]
    z, xbc, dt = (h @ w[p + "in"].t()).split([inner, inner + 2 * N, H], -1)
    K, T, B = m["conv"], max(j - i for i, j in runs), len(runs)
    u = torch.zeros(B, T + K - 1, inner + 2 * N, dtype=torch.float64, device="cuda")
    step = torch.zeros(B, T, H, dtype=torch.float64, device="cuda")  # rows behind a sequence's end change nothing
    for b, (i, j) in enumerate(runs):
        u[b, K - 1:K - 1 + j - i] = xbc[i:j]
        step[b, :j - i] = torch.nn.functional.softplus(dt[i:j] + w[p + "dt_bias"])
    u = torch.nn.functional.silu(sum(u[:, k:k + T] * w[p + "conv"][:, k] for k in range(K)) + w[p + "conv.b"])
    x, b_, c_ = u[..., :inner].reshape(B, T, H, P), u[..., inner:inner + N], u[..., inner + N:]
    decay, state = torch.exp(-torch.exp(w[p + "A_log"]) * step), torch.zeros(B, H, N, P, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    for t in range(T):
        state = state * decay[:, t, :, None, None] + b_[:, t, None, :, None] * (step[:, t, :, None] * x[:, t])[:, :, None, :]
        y[:, t] = (state * c_[:, t, None, :, None]).sum(2)
    y = (y + w[p + "D"][:, None] * x).reshape(B, T, inner)
    y = torch.cat([y[b, :j - i] for b, (i, j) in enumerate(runs)])
    return _rms(y * torch.nn.functional.silu(z), w[p + "norm"], eps) @ w[p + "o"].t(), state


def _latent_exact(h, w, p, m, eps, runs, pos):
    H, D, R, V = m["heads"], m["dim"], m["rot_dim"], m["vdim"]
    freq = _powers(m["rot"]["base"], R)
    q = (_rms(h @ w[p + "dq"].t(), w[p + "dq.norm"], eps) @ w[p + "uq"].t()).view(-1, H, D + R)
    q = torch.cat([q[..., :D], _rotated(q[..., D:], pos, freq)], -1)
    c, rot = (h @ w[p + "dkv"].t()).split([m["kv_rank"], R], -1)
    c = _rms(c, w[p + "dkv.norm"], eps)
    k = torch.cat([(c @ w[p + "uk"].t()).view(-1, H, D), _rotated(rot[:, None], pos, freq).expand(-1, H, R)], -1)
    v = (c @ w[p + "uv"].t()).view(-1, H, V)
    a = torch.cat([_attention(q[i:j], k[i:j], v[i:j], m["scale"]) for i, j in runs]).reshape(-1, H * V)
    return (a * torch.sigmoid(h @ w[p + "g"].t())) @ w[p + "o"].t()


def _grouped_exact(h, w, p, m, runs, pos):
    H, G, s = m["heads"], m["kv_heads"], m["rot"]["scaling"]
    f, i = _powers(m["rot"]["base"], 128), torch.arange(64, device="cuda", dtype=torch.float64)
    lo, hi = (128 * math.log(s["original"] / (2 * math.pi * t)) / (2 * math.log(m["rot"]["base"])) for t in (s["fast"], s["slow"]))
    lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), 127)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    f, mult = f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1
    q = _rotated((h @ w[p + "q"].t()).view(-1, H, 128), pos, f, mult, True)
    k = _rotated((h @ w[p + "k"].t()).view(-1, G, 128), pos, f, mult, True)
    v = (h @ w[p + "v"].t()).view(-1, G, 128)
    a = torch.cat([_attention(q[i:j], k[i:j], v[i:j], m["scale"], 0, m["mask"]["size"]) for i, j in runs])
    return (a * torch.sigmoid(h @ w[p + "g"].t())[:, :, None]).reshape(-1, H * 128) @ w[p + "o"].t()


def _expert(h, w, p, limit):
    g, u = (h @ w[p + "gate"].t()).clamp(max=limit), (h @ w[p + "up"].t()).clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w[p + "down"].t()


def _list_exact(case, seed, ids, cu):
    """Packed sequences -> (the last norm's output of every row, layer -> final recurrent states, rows -> logits)."""
    cfg, w = _config(case), {k: v.double() if v.dtype == torch.bfloat16 else v for k, v in _list_weights(case, seed).items()}
    runs, eps, states = [(int(a), int(b)) for a, b in zip(cu[:-1], cu[1:])], cfg["norm"]["eps"], {}
    tokens = torch.from_numpy(ids).cuda().long()
    x = w["embed"][tokens] * cfg["embedding"]["scale"]
    pos = torch.cat([torch.arange(b - a, device="cuda", dtype=torch.float64) for a, b in runs])
    for i, l in enumerate(cfg["layers"]):
        p, m, f = "l%d." % i, l["mixer"], l["mlp"]
        if case["arch"] == "girirax":
            if l["type"] == "mamba2":
                y, states[i] = _ssm_exact(x, w, p + "mix.", m, eps, runs)
            else:
                y = _latent_exact(x, w, p + "mix.", m, eps, runs, pos)
            x = x + cfg["residual_mult"] * _rms(y, w[p + "norm1"], eps)
            y = torch.nn.functional.gelu(x @ w[p + "mlp.gate"].t() + w[p + "mlp.gate.b"], approximate="tanh") * \
                (x @ w[p + "mlp.up"].t() + w[p + "mlp.up.b"])
            x = x + cfg["residual_mult"] * _rms(y @ w[p + "mlp.down"].t() + w[p + "mlp.down.b"], w[p + "norm2"], eps)
            continue
        x = x + _grouped_exact(_rms(x, 1 + w[p + "norm1"], eps), w, p + "mix.", m, runs, pos)
        h = _rms(x, 1 + w[p + "norm2"], eps)
        if f["kind"] == "dense":
            x = x + (h @ w[p + "mlp.up"].t()).relu().square() @ w[p + "mlp.down"].t()
            continue
        x, table = x + _expert(h, w, p + "mlp.shared.", f["shared"]["limit"]), w[p + "mlp.table"].long()[tokens]
        for e in range(f["router"]["experts"]):
            rows = (table == e).any(1).nonzero()[:, 0]
            x[rows] += _expert(h[rows], w, p + "mlp.e%d." % e, f["expert"]["limit"]) / f["router"]["top"]
    head, off = (w["embed"], 0) if case["arch"] == "girirax" else (w["head"], 1)
    return _rms(x, off + w["final.norm"], eps), states, lambda h: h @ head.t()


def _exact_attend(case, seed):
    t, out = _attend_inputs(case, seed), {}
    for l in range(case["layers"]):
        k, v, rows = t["k"][l].double(), t["v"][l].double(), []
        for b, n in enumerate(t["pos"].tolist()):
            k[b, n], v[b, n] = t["kn"][l][b, 0].double(), t["vn"][l][b, 0].double()
            rows.append(_attention(t["q"][l][b].double(), k[b, :n + 1], v[b, :n + 1], case["head_dim"] ** -0.5, case["window"]))
        out.update({"k%d" % l: k, "v%d" % l: v, "out%d" % l: torch.stack(rows)})
    return out


def _fed(case, seed):
    """The sequences that a pass has seen at its end, and the places whose logits say the tokens of each step."""
    lens, cu = _lengths(case, seed)
    ids, after = _tokens(case, seed, int(cu[-1])), _successor(case, seed)
    rows = [ids[a:b] for a, b in zip(cu[:-1], cu[1:])]
    if case["path"] == "decode":
        new = [[t] for t in _tokens(case, seed, case["batch"], 4)]
    else:
        new = [[after[r[-1]]] for r in rows]
    for _ in range(case["new"] - 1):
        for n in new:
            n.append(after[n[-1]])
    if case["path"] == "prefill":
        new = [[] for _ in rows]
    elif case["path"] == "sample":  # the last pick is not fed
        new = [n[:-1] for n in new]
    rows = [np.concatenate([r, np.array(n, np.int32)]).astype(np.int32) for r, n in zip(rows, new)]
    ends = np.cumsum([len(r) for r in rows])
    return np.concatenate(rows), np.concatenate([[0], ends]).astype(np.int32), ends - 1, lens


def exact(case, seed):
    if case["path"] == "attend":
        return _exact_attend(case, seed)
    if case.get("block"):
        return None  # which blocks a row attends to is a choice that rounding decides
    if case["path"] == "portions":
        rounds, held = _portions(case, seed)
        cu = np.concatenate([[0], np.cumsum(held)]).astype(np.int32)
        ids = np.concatenate([_tokens(case, seed, int(n), 100 + b) for b, n in enumerate(held)])
        h, _, head = _list_exact(case, seed, ids, cu)
        return {"logits%d" % i: head(h[torch.tensor([int(cu[b]) + at + n - 1 for b, (at, n) in r.items()]).cuda()])
                for i, r in enumerate(rounds)}
    ids, cu, last, lens = _fed(case, seed)
    out = {}
    if case["arch"] == "gpt":
        h, keys, values, head = _gpt_exact(case, seed, ids, cu)
        for l, (k, v) in enumerate(zip(keys, values)):
            for name, x in (("k", k), ("v", v)):
                cache = torch.zeros(case["batch"], _max_seq(case), case["heads"], case["head_dim"], dtype=torch.float64, device="cuda")
                for b, (i, j) in enumerate(zip(cu[:-1].tolist(), cu[1:].tolist())):
                    cache[b, :j - i] = x[i:j]
                out["%s%d" % (name, l)] = cache
    else:
        h, states, head = _list_exact(case, seed, ids, cu)
        out.update({"states%d" % i: s for i, s in states.items()})
    if case["path"] == "sample":  # the kept logits are the prompts' own
        out["logits"] = head(h[torch.from_numpy(cu[:-1] + lens - 1).cuda().long()])
        return out
    out["logits"] = head(h[torch.from_numpy(last).cuda().long()])
    if case["path"] == "prefill":
        top = out["logits"].topk(2, 1)
        out["next"], out["gap"] = top.indices[:, 0].int(), top.values[:, 0] - top.values[:, 1]
    return out
