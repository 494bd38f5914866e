"""What lumen is timed on: LoRA training steps, prompts and decode steps of served models, through
the engine a user's program drives (``ZeroEngine``, ``LLMEngine`` and its runner).

A case is a plain dict: ``path`` (train | prefill | decode), ``model`` (llama2-7b: the shapes of
Llama-2-7B; llama: the grouped-query Llama of ``lumen.bench.hybrid_bench``; the other names: that
bench's per-layer-mixer stacks), ``width``, ``layers``, ``batch`` sequences of up to ``tokens``
tokens (``ragged``: from an eighth of that on), ``dtype``, ``kv`` (cache element type), ``dropout``
(adapters).  Depth is cut to 4 - 6 layers, as in that bench: a layer costs the same at any depth.

``prepare`` makes weights and token ids from the seed, builds the engine and, for decoding, runs
the prompts and one decode step; ``run`` is one training step, one prompt step or one decode step.
``exact`` recomputes the same pass in float64 with plain torch, from the weights and token ids.

Routed experts get the confident router a trained model has: every expert owns a direction that the
embeddings of its tokens carry, so its choice does not hang on the last bit of a 16-bit row.
"""
from __future__ import annotations

import math
import os
from types import SimpleNamespace

import torch
import torch.nn.functional as F

F64 = torch.float64
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
BLOCK = 16                  # tokens per cache block (the engine's default)
CONTEXT = 4096              # max_model_len (the engine's default)
SEQUENCES = 256             # max_num_seqs (the engine's default)
CHUNK = 8192                # prompt rows per step while a decode case is prepared
STACKS = ("gedatar", "dalavik", "silonex", "tazulix")


def case(name, path, model, width, layers, batch, tokens, ragged=False, dtype="bf16", kv="auto",
         dropout=0.0):
    c = dict(path=path, model=model, width=width, layers=layers, batch=batch, tokens=tokens,
             ragged=ragged, dtype=dtype, kv=kv, dropout=dropout)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the headline training step of bench.py (8 x 512 tokens, r = 16 on q, k, v, o), 6 layers
        case("train_8x512", "train", "llama2-7b", 4096, 6, 8, 512, dropout=0.05),
        # the one run the reference published: micro-batch 1, 512 tokens, fp16 with loss scaling
        case("train_1x512_fp16", "train", "llama2-7b", 4096, 4, 1, 512, dtype="fp16"),
        # rows of 64 - 509 tokens packed back to back, grouped-query heads
        case("train_packed", "train", "llama", 2048, 4, 14, 509, ragged=True),
        # one prefill step of a burst of unequal prompts (a 4096-token scheduling budget)
        case("prefill_7b_ragged", "prefill", "llama2-7b", 4096, 4, 14, 509, ragged=True),
        # one chat user: batch-1 decode latency
        case("decode_7b_1", "decode", "llama2-7b", 4096, 4, 1, 387),
        # a full server: 256 streams in the middle of their answers
        case("decode_7b_256", "decode", "llama2-7b", 4096, 4, 256, 576, ragged=True),
        # the per-layer-mixer bench's default family: 8 prompts of 512 tokens; a few streams
        case("prefill_gedatar_8", "prefill", "gedatar", 2048, 4, 8, 512),
        case("decode_gedatar_8", "decode", "gedatar", 2048, 4, 8, 512),
        # latent attention: unequal prompts; a busy server
        case("prefill_dalavik_ragged", "prefill", "dalavik", 2048, 4, 14, 509, ragged=True),
        case("decode_dalavik_64", "decode", "dalavik", 2048, 4, 64, 512, ragged=True),
        # first token of one prompt on an idle server (window attention, three recurrences)
        case("prefill_silonex_1", "prefill", "silonex", 4096, 4, 1, 512),
        # one stream through routed experts: the smallest step
        case("decode_tazulix_1", "decode", "tazulix", 2048, 4, 1, 331),
    ]


def _log(rng, lo, hi):
    return min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choice(("train", "prefill", "decode"))
    if path == "train":
        model, width = rng.choice((("llama2-7b", 4096), ("llama", 2048), ("llama", 4096)))
        batch = _log(rng, 1, 16)
        return case(None, path, model, width, 4, batch, _log(rng, 64, max(65, 4096 // batch)),
                    rng.random() < 0.5, rng.choice(("bf16", "bf16", "fp16")))
    model = rng.choice(("llama2-7b", "llama") + STACKS)
    if model == "llama2-7b":
        width = 4096
    else:
        width = rng.choice((1024, 1536, 2048, 3072, 4096))
    dtype = rng.choice(("bf16", "bf16", "bf16", "fp16")) if model.startswith("llama") else "bf16"
    if path == "prefill":
        batch = _log(rng, 1, 32)
        rows = 4096 if width <= 2048 else 2048
        return case(None, path, model, width, 4, batch, _log(rng, 24, max(25, rows // batch)),
                    rng.random() < 0.7, dtype)
    llama = model.startswith("llama")
    batch = _log(rng, 1, 256 if llama else 64)
    return case(None, path, model, width, 4, batch, _log(rng, 17, 1023 if batch <= 64 else 576),
                rng.random() < 0.7, dtype, rng.choice(("auto", "auto", "fp8")) if llama else "auto")


def lengths(c):
    """Tokens of every sequence: all ``tokens``, or spread evenly from an eighth of it to it."""
    b, t = c["batch"], c["tokens"]
    if not c["ragged"] or b == 1:
        return [t] * b
    return [t - (t - max(1, t // 8)) * i // (b - 1) for i in range(b)]


def config(c):
    from lumen.bench import hybrid_bench
    from lumen.models import get_config

    if c["model"] == "llama2-7b":
        cfg = get_config("llama2-7b")
        cfg.num_hidden_layers = c["layers"]
        return cfg
    if c["model"] == "llama":
        return hybrid_bench.llama_config(c["width"], c["layers"])
    return getattr(hybrid_bench, c["model"] + "_config")(c["width"])


# ---- inputs ----------------------------------------------------------------------------------------
def token_ids(c, vocab, seed):
    """[batch, longest + 2] token ids on the GPU."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 1)
    return torch.randint(3, vocab, (c["batch"], c["tokens"] + 2), device="cuda", generator=g)


def llama_shapes(cfg):
    H, V, I, D = cfg.hidden_size, cfg.vocab_size, cfg.intermediate_size, cfg.head_dim
    nh, nkv = cfg.num_attention_heads, cfg.num_key_value_heads
    out = {"embed": (V, H), "norm": (H,), "head": (V, H)}
    for i in range(cfg.num_hidden_layers):
        out.update({f"{i}.n1": (H,), f"{i}.n2": (H,), f"{i}.qkv": ((nh + 2 * nkv) * D, H),
                    f"{i}.o": (H, nh * D), f"{i}.gu": (2 * I, H), f"{i}.down": (H, I)})
    return out


def _fill(name, v, g, cfg):
    """The distribution of one tensor: projections Normal(0, 1 / fan in), norm weights near 1,
    decays from slow to fast, the residual copies mostly kept."""
    leaf = name.rsplit(".", 1)[-1]
    n = v.numel()
    v.normal_(generator=g)
    if v.dim() == 0:                                                   # slope of a tanh norm
        return 0.5 + 0.5 * torch.sigmoid(v)
    if name == "embed" or name.endswith(".embed"):
        return v / (cfg.embedding_scale if cfg.arch == "tazulix" else 1.0)
    if leaf == "talk":
        return 0.2 * v + torch.eye(v.shape[0], device=v.device)
    if leaf == "mix" and ".hc" in name:
        return 0.1 * v + 0.9 * torch.eye(v.shape[0], device=v.device)
    if leaf in ("in", "out") and ".hc" in name:
        return 0.1 * v + 1.0 / v.shape[0]
    if name == "loop.in":                                              # keeps what it is given
        eye = torch.eye(v.shape[0], device=v.device)
        return 0.3 * v / math.sqrt(v.shape[1]) + 0.7 * torch.cat([eye, eye], 1)
    if leaf == "canon1":
        return 0.3 * v
    if leaf == "u" and v.dim() == 2:
        return 0.5 * v
    if v.dim() == 2:
        return v / math.sqrt(v.shape[1])
    if leaf == "w0":
        return torch.linspace(-3.0, 1.0, n, device=v.device)[
            torch.randperm(n, device=v.device, generator=g)]
    if leaf == "A_log":
        return torch.log(torch.linspace(0.5, 8.0, n, device=v.device))
    if leaf == "dt_bias":
        return v - 2.0
    if leaf in ("b", "sink"):
        return (1.0 if leaf == "sink" else 0.1) * v
    if leaf == "r1":
        return 0.3 * v.abs()
    if leaf == "r2":
        return 0.05 + 0.25 * v.abs()
    if ".mu." in name:
        return torch.sigmoid(v)
    return 1.0 + 0.1 * v                                               # norm weights, D


def weights(c, cfg, seed):
    """{name: 16-bit tensor on the GPU}: Llama's by ``llama_shapes``, a stack's by its own names."""
    dt = DTYPES[c["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 2)
    if cfg.arch == "llama":
        return {n: _fill(n, torch.empty(s, device="cuda"), g, cfg).to(dt)
                for n, s in llama_shapes(cfg).items()}
    import importlib

    shapes = importlib.import_module("lumen.models." + cfg.arch).tensor_shapes(cfg)
    w = {n: _fill(n, torch.empty(s, device="cuda"), g, cfg).to(dt) for n, s in shapes.items()}
    routers = [n for n in w if n.endswith(".router")]
    if routers:                                     # expert e's direction, and its tokens' share of it
        E, W = w[routers[0]].shape
        top = next(L["mlp"]["router"]["top"] for L in cfg.layer_specs
                   if "router" in (L.get("mlp") or {}))
        u = torch.randint(0, 2, (E, W), device="cuda", generator=g) * 2.0 - 1.0
        pick = torch.rand(cfg.vocab_size, E, device="cuda", generator=g).topk(top, 1).indices
        share = torch.zeros(cfg.vocab_size, E, device="cuda").scatter_(
            1, pick, 0.6 + 0.2 * torch.rand(cfg.vocab_size, top, device="cuda", generator=g))
        w["embed"] = (w["embed"].float() + share @ u / cfg.embedding_scale).to(dt)
        for n in routers:
            w[n] = (4.0 * u / W + w[n].float() / 20.0).to(dt)
    return w


def adapters(cfg, seed, r=16):
    """[(A, B) of q|k|v, (A, B) of o] per layer, fp32: an adapter in the middle of its training."""
    g = torch.Generator(device="cuda").manual_seed(seed * 7919 + 3)
    H, D = cfg.hidden_size, cfg.head_dim
    nh, nkv = cfg.num_attention_heads, cfg.num_key_value_heads
    out = []
    for _ in range(cfg.num_hidden_layers):
        for seg, rows, k in ((3, (nh + 2 * nkv) * D, H), (1, H, nh * D)):
            out.append((torch.randn(seg * r, k, device="cuda", generator=g) / math.sqrt(3 * k),
                        0.01 * torch.randn(rows, r, device="cuda", generator=g)))
    return out


def build(c, cfg, w):
    from lumen.models import MODEL_CLASSES

    model = MODEL_CLASSES[cfg.arch](cfg, dtype=DTYPES[c["dtype"]], device=torch.device("cuda"))
    with torch.no_grad():
        if cfg.arch != "llama":
            for n, v in w.items():
                model.tensor(n).copy_(v)
            return model
        model.embed_tokens.weight.copy_(w["embed"])
        model.norm.weight.copy_(w["norm"])
        model.lm_head.weight.copy_(w["head"])
        for i, L in enumerate(model.layers):
            for n, p in (("n1", L.input_layernorm.weight), ("n2", L.post_attention_layernorm.weight),
                         ("qkv", L.self_attn.qkv_proj.weight), ("o", L.self_attn.o_proj.weight),
                         ("gu", L.mlp.gate_up_proj.weight), ("down", L.mlp.down_proj.weight)):
                p.copy_(w[f"{i}.{n}"])
    return model


def train_batch(c, ids):
    """The rows as the collators lay them out: [batch, tokens], or packed back to back."""
    lens, rows, labels = lengths(c), [], []
    for i, n in enumerate(lens):
        rows.append(ids[i, :n])
        labels.append(torch.cat([ids[i, 1:n], ids.new_full((1,), -100)]))
    b = {"n_valid": sum(lens) - len(lens)}
    if not c["ragged"]:
        return dict(b, input_ids=torch.stack(rows), labels=torch.stack(labels))
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    pos = torch.cat([torch.arange(n, dtype=torch.int32, device="cuda") for n in lens])
    return dict(b, input_ids=torch.cat(rows).view(1, -1), labels=torch.cat(labels).view(1, -1),
                pos=pos, cu_seqlens=tuple(cu))


def prepare(case, seed):
    from lumen.utils.gemm_tuning import load_tuned_gemms

    torch.cuda.set_device(0)
    load_tuned_gemms()
    cfg = config(case)
    w = weights(case, cfg, seed)
    ids = token_ids(case, cfg.vocab_size, seed)
    model = build(case, cfg, w)
    del w
    if case["path"] == "train":
        return _prepare_train(case, cfg, model, ids, seed)
    return _prepare_serve(case, cfg, model, ids, seed)


def _prepare_train(c, cfg, model, ids, seed):
    from lumen.lora import LoraConfig, apply_lora
    from lumen.parallel.dist import init
    from lumen.train.config import load_ds_config
    from lumen.train.engine import ZeroEngine

    torch.manual_seed(seed)
    name = "ds_config_zero2.json" if c["dtype"] == "fp16" else "ds_config_zero3_mi355x.json"
    ds = load_ds_config(os.path.join(ROOT, "configs", name), c["batch"], 1, 1, 2e-4)
    apply_lora(model, LoraConfig(r=16, lora_dropout=c["dropout"]))
    with torch.no_grad():
        for (_, m), (A, B) in zip(model.lora_modules(), adapters(cfg, seed)):
            m.lora.lora_A.copy_(A)
            m.lora.lora_B.copy_(B)
    model.train()
    engine = ZeroEngine(model, ds, init())
    params = [p for _, m in model.lora_modules() for p in (m.lora.lora_A, m.lora.lora_B)]
    moments = []
    for p in params:
        _, o, n = engine.flat.index[id(p)]
        moments.append(engine.opt.m[o:o + n].view_as(p))
    return SimpleNamespace(path="train", engine=engine, batch=train_batch(c, ids),
                           params=[p.detach() for p in params], moments=moments)


def _prepare_serve(c, cfg, model, ids, seed):
    from lumen.ops.segments import SegBatch
    from lumen.serve.engine import EngineConfig, LLMEngine
    from lumen.serve.model_runner import StepInput

    lens = lengths(c)
    need = [(n + 2 + BLOCK - 1) // BLOCK for n in lens]
    engine = LLMEngine(EngineConfig(
        model=cfg.name, dtype=c["dtype"], max_model_len=CONTEXT, block_size=BLOCK,
        num_blocks=sum(need) + 1, max_num_seqs=SEQUENCES, kv_cache_dtype=c["kv"],
        async_scheduling=False), model=model, tokenizer=SimpleNamespace(eos_token_id=None))
    g = torch.Generator().manual_seed(seed)
    free = torch.randperm(sum(need), generator=g).tolist()           # blocks in a server's disorder
    tables = torch.zeros(c["batch"], max(need), dtype=torch.int32)
    for i, n in enumerate(need):
        tables[i, :n] = torch.tensor([free.pop() for _ in range(n)], dtype=torch.int32)
    tables = tables.cuda()
    i32 = dict(dtype=torch.int32, device="cuda")
    hybrid = engine.hybrid

    def slots(seg, pos):
        return tables[seg, (pos // BLOCK).long()].long() * BLOCK + pos.long() % BLOCK

    def prompts(i0, i1):
        part = lens[i0:i1]
        cu = [0]
        for n in part:
            cu.append(cu[-1] + n)
        pos = torch.cat([torch.arange(n, **i32) for n in part])
        row = torch.cat([torch.full((n,), i, **i32) for i, n in enumerate(part)])
        cuts = torch.tensor(cu, **i32)
        inp = StepInput("mixed", torch.cat([ids[i0 + i, :n] for i, n in enumerate(part)]), pos,
                        slots(row.long() + i0, pos), cu, kv_lens=list(part),
                        kv_lens_t=torch.tensor(part, **i32), prefill_tables=tables[i0:i1],
                        sample_rows=cuts[1:].long() - 1)
        if hybrid:
            from lumen.ops.segments import TILE_ROWS, tile_list

            inp.seg = SegBatch(cuts, torch.arange(i0, i1, **i32), torch.zeros(i1 - i0, **i32), row,
                               pos, tables[i0:i1], inp.slots,
                               torch.tensor(tile_list(cu, i1 - i0), **i32).view(-1, 2), cu[-1],
                               TILE_ROWS)
        return inp

    def token(step):
        pos = torch.tensor([n + step for n in lens], **i32)
        seq = torch.arange(c["batch"], **i32)
        inp = StepInput("decode", ids[seq.long(), pos.long()], pos, slots(seq.long(), pos), [0],
                        block_tables=tables, context_lens=pos + 1, max_context=max(lens) + step + 1)
        if hybrid:
            inp.seg = SegBatch(torch.arange(c["batch"] + 1, **i32), seq, pos, seq, pos, tables,
                               inp.slots)
        return inp

    s = SimpleNamespace(path=c["path"], engine=engine, runner=engine.runner)
    if c["path"] == "prefill":
        s.input = prompts(0, c["batch"])
        s.kept = _caches(engine.runner, c["batch"])
        return s
    i = 0
    while i < c["batch"]:
        j, rows = i, 0
        while j < c["batch"] and (j == i or rows + lens[j] <= CHUNK):
            rows += lens[j]
            j += 1
        engine.runner.execute(prompts(i, j))
        i = j
    engine.runner.decode(token(0))
    s.input = token(1)
    s.kept = _states(engine.runner, c["batch"])
    return s


def _caches(runner, batch):
    """What a prompt step leaves behind: the paged caches and the recurrent state."""
    st = getattr(runner, "state", None)
    if st is None:
        return {"k": runner.k_cache, "v": runner.v_cache}
    out = {}
    for n in ("keys", "lat", "k", "v"):
        for i, t in enumerate(getattr(st, n, None) or []):
            if t is not None:
                out[f"{n}{i}"] = t
    return dict(out, **_states(runner, batch))


def _states(runner, batch):
    """The recurrent states of the running sequences (slots 0 .. batch - 1)."""
    st = getattr(runner, "state", None)
    return {f"S{i}": t[:batch] for i, t in enumerate(getattr(st, "S", None) or []) if t is not None}


def run(state):
    if state.path == "train":
        loss = state.engine.forward(state.batch)
        state.engine.backward(loss)
        state.engine.step()
        return {"loss": loss.detach(), "params": state.params, "moments": state.moments}
    step = state.runner.execute if state.path == "prefill" else state.runner.decode
    return {"logits": step(state.input), "kept": state.kept}


# ---- what a pass cannot do without -------------------------------------------------------------------
def _layer_sizes(cfg):
    """Per layer (weights every row multiplies, weights of one routed expert, experts, top,
    attention entries of a row's scores and values, cache entries per token, state entries)."""
    if cfg.arch == "llama":
        D, nh, nkv = cfg.head_dim, cfg.num_attention_heads, cfg.num_key_value_heads
        H = cfg.hidden_size
        dense = (2 * nh + 2 * nkv) * D * H + 3 * H * cfg.intermediate_size
        return [(dense, 0, 0, 0, 2 * nh * D, 2 * nkv * D, 0)] * cfg.num_hidden_layers
    import importlib

    shapes = importlib.import_module("lumen.models." + cfg.arch).tensor_shapes(cfg)
    out = []
    for i, L in enumerate(cfg.layer_specs):
        m, f = L["mixer"], L.get("mlp") or {}
        one = sum(math.prod(s) for n, s in shapes.items() if n.startswith(f"l{i}.mlp.e0."))
        E, top = (f["router"]["experts"], f["router"]["top"]) if f.get("kind") == "moe" else (0, 0)
        every = sum(math.prod(s) for n, s in shapes.items() if n.startswith(f"l{i}."))
        att = cache = state = 0
        if L["type"] == "latent_attention":
            att = m["heads"] * (2 * m["kv_rank"] + m["rot_dim"])
            cache = m["kv_rank"] + m["rot_dim"]
        elif L["type"] == "attention":
            att = m["heads"] * (m["dim"] + m["vdim"])
            cache = m["kv_heads"] * (m["dim"] + (0 if cfg.arch == "gedatar" else m["vdim"]))
        elif L["type"] == "parallel":
            a, r = m["left"], m["right"]
            att, cache = 2 * a["heads"] * a["dim"], 2 * a["kv_heads"] * a["dim"]
            state = r["heads"] * r["dim"] * r["vdim"]
        elif L["type"] == "mamba2":
            state = m["heads"] * m["vdim"] * m["state"]
        else:
            state = m["heads"] * m["dim"] * m.get("vdim", m["dim"])
        out.append((every - E * one, one, E, top, att, cache, state))
    return out


def work(case):
    cfg, lens = config(case), lengths(case)
    sizes = _layer_sizes(cfg)
    T, B, W, V = sum(lens), len(lens), cfg.hidden_size, cfg.vocab_size
    rows = B if case["path"] == "decode" else T
    seen = sum(n + 2 for n in lens) if case["path"] == "decode" else sum(n * (n + 1) // 2 for n in lens)
    kv = 1 if case["kv"] == "fp8" else 2
    flops = bytes_ = 0
    for dense, one, E, top, att, cache, state in sizes:
        used = dense + min(E, rows * top) * one
        flops += 2 * rows * (dense + top * one) + 2 * seen * att + 6 * rows * state
        bytes_ += 2 * used + 8 * B * state
        bytes_ += kv * cache * (sum(lens) + 2 * B if case["path"] == "decode" else T)
    if case["path"] == "train":
        lora = cfg.num_hidden_layers * 16 * (4 * W + 2 * cfg.q_size + 2 * cfg.kv_size + 2 * W)
        head = 2 * T * V * W
        # forward and input gradients (attention backward: 2.5 x its forward); weights read twice,
        # the adapters, their gradients and both moments once
        att = sum(2 * seen * s[4] for s in sizes)
        return {"bytes": 2 * bytes_ + 4 * V * W + 2 * T * W + 32 * lora,
                "flops": 2 * (flops - att) + 3.5 * att + 2 * head + 6 * T * lora}
    return {"bytes": bytes_ + 2 * V * W + 2 * rows * W + 2 * B * V, "flops": flops + 2 * B * V * W}


def tolerance(case):
    # 16-bit weights and activations through 4 - 6 layers.  Distance from ``exact``, measured: bf16
    # logits and states 0.3 - 0.9 %, bf16 adapter moments 0.9 - 1.3 %; fp16 moments 0.1 - 0.15 % (and
    # two runs of one training step, whose gradients are summed by atomics: bf16 0.25 %, fp16 0.1 %)
    if case["dtype"] == "fp16" and case["kv"] == "auto":
        return {"rel": 0.006, "max": 0.1}
    return {"rel": 0.03, "max": 0.5}


# ---- the same pass in float64 ------------------------------------------------------------------------
def unit_rms(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def layer_norm(x, w, b, eps):
    return F.layer_norm(x, x.shape[-1:], w, b, eps)


def relu2(x):
    return torch.relu(x).square()


def turn(x, pos, freq, amp=1.0, pairs=False):
    """Rotary on the first 2 * len(freq) entries of x [B, T, n, D]: entry i pairs with i + half, or
    (``pairs``) 2i with 2i + 1."""
    a = pos[:, None].to(F64) * freq
    cs, sn = (amp * torch.cos(a))[:, None], (amp * torch.sin(a))[:, None]
    h = freq.numel()
    u, v = (x[..., 0:2 * h:2], x[..., 1:2 * h:2]) if pairs else (x[..., :h], x[..., h:2 * h])
    p, q = u * cs - v * sn, v * cs + u * sn
    y = torch.stack([p, q], -1).flatten(-2) if pairs else torch.cat([p, q], -1)
    return torch.cat([y, x[..., 2 * h:]], -1)


def base_freq(dims, base):
    return torch.tensor([float(base) ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F64,
                        device="cuda")


def attend(q, k, v, score, mask, sink=None):
    """q [B, T, H, D], k, v [B, T, G, .] -> [B, T, H * Dv]; ``score`` shapes the products
    [H, T, T]; ``sink`` [H]: a score that joins the denominator."""
    B, T, H, _ = q.shape
    out = []
    for b in range(B):
        kb = k[b].repeat_interleave(H // k.shape[2], 1).transpose(0, 1)
        vb = v[b].repeat_interleave(H // v.shape[2], 1).transpose(0, 1)
        s = score(q[b].transpose(0, 1) @ kb.transpose(1, 2)).masked_fill(~mask, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.view(H, 1, 1).expand(H, T, 1)], -1)
        p = torch.softmax(s, -1)[..., :T]
        out.append((p @ vb).transpose(0, 1).reshape(T, -1))
    return torch.stack(out)


def scan(q, k, v, decay, beta=None, unit=None, bonus=None, removal=None):
    """Matrix-state recurrences over the second axis; q, k, decay [B, T, H, D or 1], v [B, T, H, Dv].
    S <- decay S [- removal], S <- S + k v^T; the read-out S^T q.  Returns (read-outs, last state)."""
    B, T, H, D = k.shape
    S = torch.zeros(B, H, D, v.shape[-1], dtype=F64, device=k.device)
    out = []
    for t in range(T):
        kt, vt, qt = k[:, t, ..., None], v[:, t, :, None], q[:, t, :, None]
        old = S
        S = decay[:, t, ..., None] * S
        if removal is not None:                     # along the unit key, from the state before decay
            un = unit[:, t, :, None]
            S = S - (removal[:, t] * unit[:, t])[..., None] * (un @ old)
        if beta is not None:                        # delta rule: write what the key does not hold yet
            vt = beta[:, t, :, None, None] * (vt - kt.transpose(-1, -2) @ S)
        add = kt * vt
        if bonus is not None:                       # read-out before the write, plus a bonus on it
            out.append((qt @ (old + bonus[..., None] * add))[:, :, 0])
            S = S + add
        else:
            S = S + add
            out.append((qt @ S)[:, :, 0])
    return torch.stack(out, 1), S


def causal(T, window=0):
    d = torch.arange(T, device="cuda")
    d = d[:, None] - d[None]
    return (d >= 0) & (d < window if window else d >= 0)


def short_conv(x, taps, bias=None):
    """Causal depthwise convolution of x [B, T, C]; the last tap multiplies the row itself."""
    K = taps.shape[1]
    y = sum(taps[:, K - 1 - j] * F.pad(x, (0, 0, j, 0))[:, :x.shape[1]] for j in range(K))
    return y if bias is None else y + bias


class Llama:
    def __init__(self, cfg, w, lora=None, scale=2.0):
        self.cfg, self.w, self.lora, self.scale = cfg, w, lora, scale

    def proj(self, h, i, n):
        y = h @ self.w[f"{i}.{n}"].T
        if self.lora is not None:
            A, B = self.lora[2 * i + (n == "o")]
            z = h @ A.T
            r, rows = 16, 0
            cuts = [B.shape[0]] if n == "o" else [self.cfg.q_size, self.cfg.kv_size,
                                                  self.cfg.kv_size]
            parts = []
            for s, m in enumerate(cuts):
                parts.append(z[..., s * r:(s + 1) * r] @ B[rows:rows + m].T)
                rows += m
            y = y + self.scale * torch.cat(parts, -1)
        return y

    def __call__(self, ids):
        """Token ids [B, T] -> (the normed last rows [B, T, W], {kept: [B, T, ...]})."""
        cfg, w, eps = self.cfg, self.w, self.cfg.rms_norm_eps
        nh, nkv, D = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
        B, T = ids.shape
        pos, mask = torch.arange(T, device="cuda"), causal(T)
        f = base_freq(D, cfg.rope_theta)
        x, kept = w["embed"][ids], {}
        for i in range(cfg.num_hidden_layers):
            h = unit_rms(x, eps) * w[f"{i}.n1"]
            q, k, v = self.proj(h, i, "qkv").split([nh * D, nkv * D, nkv * D], -1)
            q, k, v = q.view(B, T, nh, D), k.view(B, T, nkv, D), v.view(B, T, nkv, D)
            q, k = turn(q, pos, f), turn(k, pos, f)
            kept[f"k{i}"], kept[f"v{i}"] = k, v
            o = attend(q, k, v, lambda s: s / math.sqrt(D), mask)
            x = x + self.proj(o, i, "o")
            g, u = (unit_rms(x, eps) * w[f"{i}.n2"] @ w[f"{i}.gu"].T).chunk(2, -1)
            x = x + (F.silu(g) * u) @ w[f"{i}.down"].T
        return unit_rms(x, eps) * w["norm"], kept

    def logits(self, h):
        return h @ self.w["head"].T


class Stack:
    def __init__(self, cfg, w):
        self.cfg, self.w, self.eps = cfg, w, cfg.rms_norm_eps

    def lin(self, h, name):
        y = h @ self.w[name].T
        return y + self.w[name + ".b"] if name + ".b" in self.w else y


class Gedatar(Stack):
    def norm(self, x, n):
        w = self.w
        return torch.tanh(w[n + ".alpha"] * x) * w[n] + w[n + ".b"]

    def mixer(self, i, L, h, kept):
        w, m, p, eps = self.w, L["mixer"], f"l{i}.mix.", self.eps
        B, T, _ = h.shape
        heads = lambda x: x.view(B, T, -1, m["dim"])  # noqa: E731
        if L["type"] == "attention":
            q, k = heads(h @ w[p + "q"].T), heads(h @ w[p + "k"].T)
            kept[f"keys{i}"] = k
            at = torch.arange(T, device="cuda") // m["mask"]["size"]
            o = attend(unit_rms(q, eps), unit_rms(k, eps), k, lambda s: s * m["scale"],
                       causal(T) & (at[:, None] == at[None]),
                       torch.zeros(m["heads"], dtype=F64, device="cuda"))
            return o @ w[p + "o"].T
        if L["type"] == "wkv":
            prev = F.pad(h, (0, 0, 1, 0))[:, :T]
            r, k, v, g, d = (h + (prev - h) * w[p + "mu." + s] for s in "rkvgw")
            decay = torch.exp(-torch.exp(torch.tanh(d @ w[p + "w1"].T) @ w[p + "w2"].T + w[p + "w0"]))
            o, S = scan(heads(r @ w[p + "r"].T), heads(k @ w[p + "k"].T), heads(v @ w[p + "v"].T),
                        heads(decay), bonus=w[p + "u"])
            gate = F.silu(g @ w[p + "g"].T)
        else:
            r, k, v, g = (h @ w[p + s].T for s in "rkvg")
            d = torch.tanh(h @ w[p + "w1"].T) @ w[p + "w2"].T + w[p + "w0"]
            decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(d))
            k = heads(k)
            unit = k / torch.sqrt(k.square().sum(-1, keepdim=True) + 1e-6)
            o, S = scan(heads(r), k, heads(v), heads(decay), unit=unit,
                        removal=heads(torch.sigmoid(self.lin(h, p + "a"))))
            gate = torch.sigmoid(g)
        kept[f"S{i}"] = S
        return (unit_rms(o, eps).flatten(2) * w[p + "norm"] * gate) @ w[p + "o"].T

    def ff(self, f, p, h):
        w = self.w
        one = lambda q, x: (F.silu(x @ w[q + "gate"].T) * (x @ w[q + "up"].T)) @ w[q + "down"].T  # noqa: E731
        if f["kind"] == "dense":
            return one(p, h)
        z, idx = (h @ w[p + "router"].T + w[p + "router.b"]).topk(f["router"]["top"], -1)
        r = torch.zeros(*h.shape[:-1], f["router"]["experts"], dtype=F64, device="cuda")
        r.scatter_(-1, idx, torch.softmax(z, -1))
        y = one(p + "shared.", h)
        for e in range(r.shape[-1]):
            y = y + r[..., e:e + 1] * one(p + f"e{e}.", h)
        return y

    def __call__(self, ids):
        x, kept = self.w["embed"][ids], {}
        for i, L in enumerate(self.cfg.layer_specs):
            p = f"l{i}."
            h = self.norm(x, p + "norm1")
            x = x + self.norm(self.mixer(i, L, h + short_conv(h, self.w[p + "canon1"]), kept),
                              p + "norm1b")
            x = x + self.norm(self.ff(L["mlp"], p + "mlp.", self.norm(x, p + "norm2")), p + "norm2b")
        return self.norm(x, "final.norm"), kept

    def logits(self, h):
        return h @ self.w["head"].T


class Dalavik(Stack):
    def group(self, x, n):
        g = self.cfg.norm_groups
        return unit_rms(x.unflatten(-1, (g, -1)), self.eps).flatten(-2) * self.w[n]

    def mixer(self, i, L, x, kept):
        w, m, p, eps = self.w, L["mixer"], f"l{i}.mix.", self.eps
        B, T, _ = x.shape
        pos, mask, H, D = torch.arange(T, device="cuda"), causal(T), m["heads"], m["dim"]
        if L["type"] == "latent_attention":
            R, f = m["kv_rank"], base_freq(m["rot"]["dims"], m["rot"]["base"])
            if m.get("kv_from") is None:
                z = x @ w[p + "dkv"].T
                kr = turn(z[..., None, R:], pos, f, pairs=True)[:, :, 0]
                kept[f"lat{i}"] = torch.cat([unit_rms(z[..., :R], eps) * w[p + "dkv.norm"], kr], -1)
            row = kept[f"lat{m.get('kv_from', i)}"]
            q = (unit_rms(x @ w[p + "dq"].T, eps) * w[p + "dq.norm"]) @ w[p + "uq"].T
            q = q.view(B, T, H, -1)
            q = torch.cat([q[..., :D], turn(q[..., D:], pos, f, pairs=True)], -1)
            k = (row[..., :R] @ w[p + "uk"].T).view(B, T, H, D)
            k = torch.cat([k, row[:, :, None, R:].expand(B, T, H, -1)], -1)
            v = (row[..., :R] @ w[p + "uv"].T).view(B, T, H, -1)
            return attend(q, k, v, lambda s: s * m["scale"], mask) @ w[p + "o"].T
        q, k, v = (self.lin(x, p + n).view(B, T, -1, D) for n in "qkv")
        q, k = unit_rms(q, eps) * w[p + "q.norm"], unit_rms(k, eps) * w[p + "k.norm"]
        kept[f"k{i}"], kept[f"v{i}"] = k, v
        qt = m["q_temp"]
        q = q * (1.0 + qt["coef"] * torch.log(torch.floor((pos.to(F64) + 1) / qt["every"]) + 1.0)
                 ).view(T, 1, 1)
        far = torch.log1p(w[p + "r2"].view(H, 1, 1) * (pos[:, None] - pos).clamp(min=0).to(F64))

        def score(s):
            s = m["softcap"] * torch.tanh(s * m["scale"] / m["softcap"])
            s = s - w[p + "r1"].view(H, 1, 1) * far
            return (w[p + "talk"] @ s.view(H, -1)).view(H, T, T)

        return attend(q, k, v, score, mask, w[p + "sink"]) @ w[p + "o"].T

    def __call__(self, ids):
        w, x, kept, sd = self.w, self.w["embed"][ids], {}, self.cfg.token_side_dim
        for i, L in enumerate(self.cfg.layer_specs):
            p = f"l{i}."
            x = x + self.group(self.mixer(i, L, x, kept), p + "norm1")
            y = torch.relu(x @ w[p + "mlp.gate"].T) * (x @ w[p + "mlp.up"].T)
            x = x + self.group(y @ w[p + "mlp.down"].T, p + "norm2")
            e = w["side.embed"][ids][..., i * sd:(i + 1) * sd]
            y = (F.gelu(x @ w[p + "side.gate"].T, approximate="tanh") * e) @ w[p + "side.proj"].T
            x = x + unit_rms(y, self.eps) * w[p + "side.norm"]
        return self.group(x, "final.norm"), kept

    def logits(self, h):
        return h @ self.w["embed"].T


class Silonex(Stack):
    def mixer(self, i, L, h, kept):
        w, m, p, eps = self.w, L["mixer"], f"l{i}.mix.", self.eps
        B, T, _ = h.shape
        heads = lambda x, n: x.view(B, T, n, -1)  # noqa: E731
        if L["type"] == "lightning":
            return lightning(w, p, m, h, eps, kept, i)
        if L["type"] == "mamba2":
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            z, c, dt = (h @ w[p + "in"].T).split([H * P, H * P + 2 * G * N, H], -1)
            c = F.silu(short_conv(c, w[p + "conv"], w[p + "conv.b"]))
            x, b, c = c.split([H * P, G * N, G * N], -1)
            x = heads(x, H)
            b, c = (heads(t, G).repeat_interleave(H // G, 2) for t in (b, c))
            dt = F.softplus(dt + w[p + "dt_bias"])[..., None]
            y, kept[f"S{i}"] = scan(c, b, dt * x, torch.exp(-torch.exp(w[p + "A_log"])[:, None] * dt))
            y = (y + w[p + "D"][:, None] * x).flatten(2) * F.silu(z)
            y = unit_rms(y.unflatten(-1, (m["norm_groups"], -1)), eps).flatten(-2) * w[p + "norm"]
            return y @ w[p + "o"].T
        a, q_ = m["left"], p + "left."
        q = unit_rms(heads(h @ w[q_ + "q"].T, a["heads"]), eps) * w[q_ + "q.norm"]
        k = unit_rms(heads(h @ w[q_ + "k"].T, a["kv_heads"]), eps) * w[q_ + "k.norm"]
        v = unit_rms(heads(h @ w[q_ + "v"].T, a["kv_heads"]), eps)
        f, sc = base_freq(a["rot"]["dims"], a["rot"]["base"]), a["rot"]["scaling"]
        wave = 2.0 * math.pi / f
        keep = ((sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        f = (1.0 - keep) * f / sc["factor"] + keep * f
        pos = torch.arange(T, device="cuda")
        q, k = turn(q, pos, f), turn(k, pos, f)
        kept[f"k{i}"], kept[f"v{i}"] = k, v
        cap = a["softcap"]
        left = attend(q, k, v, lambda s: cap * torch.tanh(s * a["scale"] / cap),
                      causal(T, a["mask"]["size"])) @ w[q_ + "o"].T
        r, q_ = m["right"], p + "right."
        H, G = r["heads"], r["kv_heads"]
        q, k, v = (F.silu(short_conv(h @ w[q_ + n].T, w[q_ + n + ".conv"])) for n in "qkv")
        unit = lambda x: x / torch.sqrt(x.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k = (unit(heads(t, G)).repeat_interleave(H // G, 2) for t in (q, k))
        decay = torch.exp(-torch.exp(w[q_ + "A_log"]) * F.softplus(h @ w[q_ + "a"].T + w[q_ + "dt_bias"]))
        o, kept[f"S{i}"] = scan(q * r["dim"] ** -0.5, k, heads(v, H), decay[..., None],
                                beta=torch.sigmoid(h @ w[q_ + "b"].T))
        o = unit_rms(o, eps) * w[q_ + "norm"] * F.silu(heads(h @ w[q_ + "g"].T, H))
        right = o.flatten(2) @ w[q_ + "o"].T
        return 0.5 * (unit_rms(left, eps) * w[p + "left.out"] + unit_rms(right, eps) * w[p + "right.out"])

    def sub(self, xs, p, n, fn):
        w = self.w
        h = torch.einsum("s,sbtw->btw", w[p + f"hc{n}.in"], xs)
        y = fn(layer_norm(h, w[p + f"norm{n}"], w[p + f"norm{n}.b"], self.eps))
        return (torch.einsum("st,sbcw->tbcw", w[p + f"hc{n}.mix"], xs)
                + w[p + f"hc{n}.out"].view(-1, 1, 1, 1) * y)

    def __call__(self, ids):
        w, kept = self.w, {}
        xs = w["embed"][ids].expand(self.cfg.streams, -1, -1, -1)
        for i, L in enumerate(self.cfg.layer_specs):
            p = f"l{i}."
            ff = lambda h: (F.silu(h @ w[p + "mlp.gate"].T) * (h @ w[p + "mlp.up"].T)) @ w[p + "mlp.down"].T  # noqa: E731
            xs = self.sub(xs, p, 1, lambda h: self.mixer(i, L, h, kept))
            xs = self.sub(xs, p, 2, ff)
        return layer_norm(xs.sum(0), w["final.norm"], w["final.norm.b"], self.eps), kept

    def logits(self, h):
        return h @ self.w["embed"].T


def lightning(w, p, m, h, eps, kept, i):
    B, T, _ = h.shape
    q, k, v = (F.silu(h @ w[p + n].T).view(B, T, m["heads"], -1) for n in "qkv")
    decay = torch.tensor(m["decay"], dtype=F64, device="cuda").view(1, 1, -1, 1).expand(B, T, -1, 1)
    o, kept[f"S{i}"] = scan(q, k, v, decay)
    o = unit_rms(o.flatten(2), eps) * w[p + "norm"] * torch.sigmoid(h @ w[p + "g"].T)
    return o @ w[p + "o"].T


class Tazulix(Stack):
    def attention(self, i, m, h, kept):
        w, p, eps = self.w, f"l{i}.mix.", self.eps
        B, T, _ = h.shape
        q = (unit_rms(self.lin(h, p + "q"), eps) * w[p + "q.norm"]).view(B, T, m["heads"], -1)
        k = (unit_rms(self.lin(h, p + "k"), eps) * w[p + "k.norm"]).view(B, T, m["kv_heads"], -1)
        v = self.lin(h, p + "v").view(B, T, m["kv_heads"], -1)
        r = m["rot"]
        sc, n, f = r["scaling"], r["dims"], base_freq(r["dims"], r["base"])
        at = lambda turns: n * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(r["base"]))  # noqa: E731
        lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), n - 1)
        ramp = ((torch.arange(n // 2, device="cuda", dtype=F64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        f, amp = f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
        pos = torch.arange(T, device="cuda")
        q, k = turn(q, pos, f, amp), turn(k, pos, f, amp)
        kept[f"k{i}"], kept[f"v{i}"] = k, v
        return attend(q, k, v, lambda s: s * m["scale"], causal(T)) @ w[p + "o"].T

    def ff(self, f, p, h):
        w = self.w
        if f["kind"] == "dense":
            return relu2(h @ w[p + "up"].T) @ w[p + "down"].T

        def one(q, x, limit):
            g = (x @ w[q + "gate"].T).clamp(max=limit)
            u = (x @ w[q + "up"].T).clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[q + "down"].T

        s = torch.sigmoid(h @ w[p + "router"].T)
        val, idx = s.topk(f["router"]["top"], -1)
        r = torch.zeros_like(s).scatter_(-1, idx, val)
        y = one(p + "shared.", h, f["shared"]["limit"])
        for e in range(s.shape[-1]):
            on = (r[..., e:e + 1] > 0).to(F64)
            y = y + on * one(p + f"e{e}.", r[..., e:e + 1] * h, f["expert"]["limit"])
        return y

    def __call__(self, ids):
        w, eps, kept = self.w, self.eps, {}
        x0 = w["embed"][ids] * self.cfg.embedding_scale
        x, lp = x0, self.cfg.loop
        for i, L in enumerate(self.cfg.layer_specs):
            p = f"l{i}."
            if i == lp["start"]:                                     # one pass through the loop
                x = torch.cat([x, x0], -1) @ w["loop.in"].T
            h = unit_rms(x, eps) * w[p + "norm1"]
            x = x + (self.attention(i, L["mixer"], h, kept) if L["type"] == "attention" else
                     lightning(w, p + "mix.", L["mixer"], h, eps, kept, i))
            x = x + self.ff(L["mlp"], p + "mlp.", unit_rms(x, eps) * w[p + "norm2"])
        return unit_rms(x, eps) * w["final.norm"], kept

    def logits(self, h):
        return h @ self.w["head"].T


def exact(case, seed):
    c, cfg = case, config(case)
    lens = lengths(c)
    ids = token_ids(c, cfg.vocab_size, seed)
    w = {n: v.to(F64) for n, v in weights(c, cfg, seed).items()}
    if c["path"] == "train":
        return _exact_train(c, cfg, w, ids, lens, seed)
    net = Llama(cfg, w) if cfg.arch == "llama" else {
        "gedatar": Gedatar, "dalavik": Dalavik, "silonex": Silonex, "tazulix": Tazulix}[cfg.arch](cfg, w)
    more = 2 if c["path"] == "decode" else 0
    logits, states = [], {}
    with torch.no_grad():
        # sequences of like length together; a state is read at its own sequence's end, so unequal
        # sequences of a recurrent stack go one by one
        group = 8 if len(set(lens)) == 1 or cfg.arch in ("llama", "dalavik") else 1
        for i in range(0, len(lens), group):
            n = max(lens[i:i + group]) + more
            h, kept = net(ids[i:i + group, :n])
            last = torch.tensor([m + more - 1 for m in lens[i:i + group]], device="cuda")
            logits.append(net.logits(h[torch.arange(h.shape[0], device="cuda"), last]))
            for name, t in kept.items():
                if name[0] == "S":
                    states.setdefault(name, []).append(t)
    # (the paged caches hold the projections of every token: what the logits and states come from)
    return {"logits": torch.cat(logits), "kept": {n: torch.cat(t) for n, t in states.items()}}


def _exact_train(c, cfg, w, ids, lens, seed):
    if c["dropout"] > 0:           # the mask is drawn inside the step
        return None
    lora = [(A.to(F64).requires_grad_(), B.to(F64).requires_grad_()) for A, B in adapters(cfg, seed)]
    net = Llama(cfg, w, lora)
    total, n_valid = 0.0, sum(lens) - len(lens)
    for i, n in enumerate(lens):
        h, _ = net(ids[i:i + 1, :n])
        loss = F.cross_entropy(net.logits(h[0, :n - 1]), ids[i, 1:n], reduction="sum") / n_valid
        loss.backward()
        total = total + loss.detach()
    flat = [p for pair in lora for p in pair]
    norm = torch.sqrt(sum(p.grad.square().sum() for p in flat))
    clip = torch.clamp(1.0 / (norm + 1e-6), max=1.0)
    # the first step of the warm-up runs at learning rate 0: parameters stay, the moments move
    return {"loss": total, "params": [p.detach() for p in flat],
            "moments": [0.1 * clip * p.grad for p in flat]}
