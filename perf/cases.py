"""The framework's measured workloads: what a speculative-decoding program has it do, through the public entry
points (``SubnetworkDraftModel.forward`` / ``forward_rows``, the vocabulary head, the sampler).

Model cases run blocks of a model -- one to three layers at a Llama shape the repository serves (1B, 8B, 70B) -- with the
vocabulary of the few prompt cases that end in a head cut in proportion (8192 rows beside two layers is what 128256
is beside thirty-two), so that a layer's and the head's shares of a pass are those of the whole model.
"""

import math
import os
import sys

import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "subnetwork-speculative-decoding_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

BF16 = torch.bfloat16
# hidden, q heads, kv heads, head_dim, MLP width
SHAPES = {"1b": (2048, 32, 8, 64, 8192), "8b": (4096, 32, 8, 128, 14336), "70b": (8192, 64, 8, 128, 28672)}
EPS, THETA, BLOCK_VOCAB = 1e-5, 500000.0, 8192
TOP_K = 4


# ------------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # The prompt's target forward before decoding starts: a long document, a chat turn with history, a short
        # question to the small model (odd length), and the shortest kind of prompt.
        dict(name="prompt_8b_4096", kind="prompt", shape="8b", layers=2, tokens=4096),
        dict(name="prompt_8b_512", kind="prompt", shape="8b", layers=2, tokens=512),
        dict(name="prompt_1b_300", kind="prompt", shape="1b", layers=4, tokens=300),
        dict(name="prompt_8b_100", kind="prompt", shape="8b", layers=2, tokens=100),
        # One autoregressive step of the small model: one row, the latency of its launches.
        dict(name="step_1b", kind="rows", mode="ar", shape="1b", layers=4, rows=1, context=512),
        # One drafted level: 12 tree rows through two sub-network layers and the bridge between them.
        dict(name="draft_8b", kind="rows", mode="draft", shape="8b", layers=3, rows=12, context=4096),
        # The verify forward of a 24-node tree (25 rows) at an ordinary and at a long context.
        dict(name="verify_8b", kind="rows", mode="tree", shape="8b", layers=2, rows=25, context=4096),
        dict(name="verify_70b_16k", kind="rows", mode="tree", shape="70b", layers=1, rows=25, context=16384),
        # One step of batched generation: a row of each of 32 sequences of different lengths.
        dict(name="batch_8b", kind="rows", mode="batch", shape="8b", layers=2, rows=32, context=1024),
        # Greedy verification's head: each row's argmax over the vocabulary.
        dict(name="argmax_8b", kind="head", hidden=4096, vocab=128256, rows=25, k=1, mode=0),
        # Sampled decoding: the draft distribution and the children drawn from it for one level, and the
        # acceptance of the whole tree (depth 3, branch 3-2-1: 16 rows).
        dict(name="propose", kind="propose", vocab=128256, rows=6, k=2, temperature=0.7, top_p=0.9),
        dict(name="accept", kind="accept", vocab=128256, branch="3,2,1", temperature=0.7, top_p=0.9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prompt", "prompt", "rows", "rows", "rows", "head", "propose", "accept"])
    if kind == "prompt":
        shape = rng.choice(["1b", "8b"])
        return dict(kind=kind, shape=shape, layers=2, tokens=_log(rng, 24, 4000 if shape == "1b" else 2600))
    if kind == "rows":
        mode = rng.choice(["ar", "draft", "tree", "tree", "batch"])
        shape = rng.choice(["1b", "8b", "8b", "70b"]) if mode in ("ar", "tree") else rng.choice(["1b", "8b"])
        rows = 1 if mode == "ar" else _log(rng, 3, 24) if mode == "draft" else _log(rng, 5, 64)
        context = _log(rng, 48, 2500) if mode == "batch" else _log(rng, 48, 16000)
        return dict(kind=kind, mode=mode, shape=shape, layers=1 if shape == "70b" else 3 if mode == "draft" else 2,
                    rows=rows, context=context)
    vocab = rng.choice([32768, 128256])
    if kind == "head":
        k = rng.randint(1, TOP_K)
        return dict(kind=kind, hidden=rng.choice([2048, 4096]), vocab=vocab, rows=_log(rng, 1, 64), k=k,
                    mode=int(k > 1))
    temperature, top_p = round(rng.uniform(0.5, 1.2), 2), rng.choice([0.8, 0.9, 0.95, 1.0])
    if kind == "propose":
        return dict(kind=kind, vocab=vocab, rows=_log(rng, 1, 24), k=rng.randint(1, TOP_K), temperature=temperature,
                    top_p=top_p)
    branch = rng.choice(["4", "4,5", "3,2,1", "3,2,2", "2,2,2,1", "1,1,1,1", "4,2,1,1"])
    return dict(kind=kind, vocab=vocab, branch=branch, temperature=temperature, top_p=top_p)


# ------------------------------------------------------------------------------------------------- inputs
class _Rand:
    """Tensors of one case, each from its own seeded generator on the GPU."""

    def __init__(self, seed):
        self.seed, self.n = seed, 0

    def gen(self):
        self.n += 1
        return torch.Generator(device="cuda").manual_seed(self.seed * 1009 + self.n)

    def normal(self, *size, std=1.0, mean=0.0, dtype=BF16):
        t = torch.randn(*size, generator=self.gen(), device="cuda", dtype=dtype)
        return t.mul_(std).add_(mean) if mean else t.mul_(std)

    def ints(self, n, hi):
        return torch.randint(0, hi, (n,), generator=self.gen(), device="cuda")


def _model_tensors(case, r):
    """State-dict tensors of the case's model (HF names); matrices N(0, 0.02), norm weights around 1."""
    d, heads, kv, hd, inter = SHAPES[case["shape"]]
    sd = {"model.embed_tokens.weight": r.normal(BLOCK_VOCAB, d, std=0.02)}
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        for name, n, k in (("self_attn.q_proj", heads * hd, d), ("self_attn.k_proj", kv * hd, d),
                           ("self_attn.v_proj", kv * hd, d), ("self_attn.o_proj", d, heads * hd),
                           ("mlp.gate_proj", inter, d), ("mlp.up_proj", inter, d), ("mlp.down_proj", d, inter)):
            sd[p + name + ".weight"] = r.normal(n, k, std=0.02)
        for name in ("input_layernorm", "post_attention_layernorm"):
            sd[p + name + ".weight"] = r.normal(d, std=0.1, mean=1.0)
    sd["model.norm.weight"] = r.normal(d, std=0.1, mean=1.0)
    sd["lm_head.weight"] = r.normal(BLOCK_VOCAB, d, std=0.02)
    return sd


def _bridge_tensors(case, r):
    """The one bridge of a draft case: layers 0 and 2 of three are selected, so it leads into layer 2."""
    d = SHAPES[case["shape"]][0]
    p = "into_2."
    return {p + "norm.weight": r.normal(d, std=0.1, mean=1.0).float(),
            p + "mlp.body.0.weight": r.normal(d, d, std=d ** -0.5).float(), p + "mlp.body.0.bias": r.normal(d, std=0.1).float(),
            p + "mlp.out_proj.weight": r.normal(d, d, std=0.01).float(),
            p + "mlp.out_proj.bias": r.normal(d, std=0.01).float()}


def _row_table(case, seed):
    """Host lists of a forward's rows: position, slot, prefix, ancestor slots, and the committed lengths per row."""
    g = torch.Generator().manual_seed(seed)
    m, ctx = case["rows"], case["context"]
    if case["mode"] == "batch":  # lengths between half the context and all of it
        lens = [ctx] + torch.randint(ctx // 2, ctx + 1, (m - 1,), generator=g).tolist()
        return lens, lens, [c + 1 for c in lens], [[] for _ in lens], lens
    if case["mode"] == "ar":
        return [ctx], [ctx], [ctx + 1], [[]], [ctx]
    # row 0 the root at the first free slot, row i a node whose parent is one of the rows before it (depth <= 6)
    paths = [[]]
    for i in range(1, m):
        ok = [j for j, p in enumerate(paths) if len(p) < 6]
        paths.append(paths[ok[int(torch.randint(max(0, len(ok) - 8), len(ok), (1,), generator=g))]] + [ctx + i])
    return [ctx + len(p) for p in paths], [ctx + i for i in range(m)], [ctx + 1] * m, paths, [ctx] * m


def _kv_tensors(case, r):
    """The committed K and V of each layer [layers, sequences, kv heads, context, head_dim] (K after its rotation)."""
    _, _, kv, hd, _ = SHAPES[case["shape"]]
    n_seq = case["rows"] if case["mode"] == "batch" else 1
    size = (case["layers"], n_seq, kv, case["context"], hd)
    return r.normal(*size, std=1.3), r.normal(*size, std=1.3)


def _sampled_logits(case, r, rows):
    """Target rows spread like a language model's, draft rows the same with an error of their own."""
    ld = (case["vocab"] + 7) // 8 * 8
    target = r.normal(rows, ld, std=2.5)
    return target, (target.float() + r.normal(rows, ld, dtype=torch.float32)).to(BF16)


def _warp64(logits, temperature, top_p):
    """softmax(logits / T) with the nucleus cut (ties: lower columns first), in 64 bits."""
    p = torch.softmax(logits.double() / temperature, -1)
    if top_p < 1.0:
        s, i = torch.sort(p, descending=True, stable=True)
        keep = torch.zeros_like(p, dtype=torch.bool).scatter_(-1, i, s.cumsum(-1) - s <= top_p)
        p = torch.where(keep, p, torch.zeros_like(p))
    return p / p.sum(-1, keepdim=True)


def _tree_parents(branch):
    """Parents (-1 the root), child ranks and depths of the whole tree, level by level."""
    parents, ranks, depths, level = [], [], [], [-1]
    for d, b in enumerate(branch):
        nxt = []
        for p in level:
            for k in range(b):
                parents.append(p)
                ranks.append(k)
                depths.append(d + 1)
                nxt.append(len(parents) - 1)
        level = nxt
    return parents, ranks, depths


# ------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"prompt": _prepare_prompt, "rows": _prepare_rows, "head": _prepare_head, "propose": _prepare_propose,
            "accept": _prepare_accept}[case["kind"]](case, _Rand(seed), seed)


def _build(case, r):
    from ssd.models.llama import LlamaShape, MI355XLlama

    d, heads, kv, hd, inter = SHAPES[case["shape"]]
    shape = LlamaShape(d, case["layers"], heads, kv, hd, inter, BLOCK_VOCAB, EPS, THETA)
    return MI355XLlama.from_state_dict(_model_tensors(case, r), shape)


def _prepare_prompt(case, r, seed):
    from ssd.engine.speculative import TargetRunner

    target = TargetRunner(_build(case, r))
    ids = r.ints(case["tokens"], BLOCK_VOCAB).cpu()[None]
    return dict(case=case, target=target, ids=ids, cache=target.new_cache(case["tokens"] + 64))


def _prepare_rows(case, r, seed):
    from ssd import ops
    from ssd.config import BridgeConfig
    from ssd.engine.kv_cache import KVCache
    from ssd.engine.speculative import TargetRunner
    from ssd.models.subnetwork_draft import Rows, SubnetworkDraftModel

    base = _build(case, r)
    if case["mode"] == "draft":
        model = SubnetworkDraftModel(base, [0, 2], BridgeConfig())
        model.bridges.load_state_dict(_bridge_tensors(case, r))
        model.place_bridges()
    else:
        model = TargetRunner(base)
    s, m, ctx = base.shape, case["rows"], case["context"]
    ids = r.ints(m, BLOCK_VOCAB).to(torch.int32)
    k, v = _kv_tensors(case, r)
    pos, slot, prefix, anc, _ = _row_table(case, seed)
    cap = (ctx + m + 1 + 63) // 64 * 64
    n_seq = k.shape[1]
    arenas = []
    for t, which in ((k, "k"), (v, "v")):
        plain = torch.zeros(n_seq, s.layers, s.kv_heads, cap, s.head_dim, dtype=BF16, device="cuda")
        plain[:, :, :, :ctx] = t.transpose(0, 1)
        arena = torch.empty(n_seq, s.layers, s.kv_heads, cap * s.head_dim, dtype=BF16, device="cuda")
        for i in range(n_seq):
            arena[i] = ops.kv_tile(plain[i], which)
        arenas.append(arena)
    cache = KVCache(s.layers, cap)
    cache.kv_heads, cache.head_dim, cache.device = s.kv_heads, s.head_dim, base.device
    cache.k, cache.vt = arenas[0][0], arenas[1][0]
    rows = Rows(64, base.device)
    rows.upload(ids.cpu(), pos, slot, prefix, [len(a) for a in anc], anc)
    if case["mode"] == "batch":
        rows.set_kv_offsets(torch.arange(n_seq, dtype=torch.int64, device="cuda") * arenas[0][0].numel())
        p_min = 0  # rows of different sequences share no keys
    else:
        p_min = min(prefix)
    l_max = max(p + len(a) for p, a in zip(prefix, anc))
    ws = model.workspace()
    torch.cuda.synchronize()
    return dict(case=case, model=model, rows=rows, cache=cache, arenas=arenas, ws=ws, p_min=p_min, l_max=l_max)


def _head_tensors(case, r):
    return (r.normal(case["rows"], case["hidden"], std=1.0), r.normal(case["vocab"], case["hidden"], std=0.02),
            r.normal(case["hidden"], std=0.1, mean=1.0))


def _prepare_head(case, r, seed):
    from ssd import ops

    m, n, k = case["rows"], case["vocab"], case["k"]
    h, w, norm = _head_tensors(case, r)
    return dict(case=case, h=h, w=ops.pack_weight(w, col_scale=norm),
                parts=torch.empty(ops.gemm_topk_bytes(m, n), dtype=torch.uint8, device="cuda"),
                tok=torch.zeros(m * k, dtype=torch.int32, device="cuda"),
                val=torch.zeros(m * k, dtype=torch.float32, device="cuda"))


def _prepare_propose(case, r, seed):
    from ssd import ops

    m, v, k = case["rows"], case["vocab"], case["k"]
    return dict(case=case, logits=_sampled_logits(case, r, m)[0], seed=seed,
                q=torch.zeros(m, (v + 3) // 4 * 4, dtype=torch.float32, device="cuda"),
                tok=torch.zeros(m * k, dtype=torch.int32, device="cuda"),
                lp=torch.zeros(m * k, dtype=torch.float32, device="cuda"),
                ws=torch.empty(ops.sample_ws_bytes(m, v), dtype=torch.uint8, device="cuda"))


def _prepare_accept(case, r, seed):
    from ssd.engine.sampling import Sampler
    from ssd.engine.tree_drafter import DeviceTree

    branch = [int(b) for b in case["branch"].split(",")]
    parents, ranks, depths = _tree_parents(branch)
    n, v = len(parents), case["vocab"]
    target, draft = _sampled_logits(case, r, n + 1)
    sampler = Sampler(case["temperature"], case["top_p"], v, "cuda", 1 + n, 1 + n, seed)
    sampler.max_kids, sampler.counter = max(branch), 1
    q = _warp64(draft[:, :v], case["temperature"], case["top_p"]).float()
    sampler.Q[:, :v] = q
    tokens = []
    for p in dict.fromkeys(parents):  # children in order, drawn without replacement from their parent's row
        b = parents.count(p)
        tokens += torch.multinomial(q[p + 1], b, generator=r.gen()).tolist()
    tree = DeviceTree("cuda", cap=n)
    i32 = dict(dtype=torch.int32, device="cuda")
    for dst, src in ((tree.vtokens, tokens), (tree.vparents, parents), (tree.vranks, ranks), (tree.vdepths, depths),
                     (tree.vorig, list(range(n)))):
        dst[:n] = torch.tensor(src, **i32)
    tree.vmeta[0] = n
    depth = len(branch)
    return dict(case=case, sampler=sampler, tree=tree, logits=target[:, :v], rows=n + 1,
                result=torch.zeros(depth + 3, **i32), keep=torch.zeros(depth + 2, **i32), n_keep=torch.zeros(1, **i32),
                root=torch.zeros(1, **i32))


# ------------------------------------------------------------------------------------------------- run
def run(state):
    from ssd import ops

    c = state["case"]
    if c["kind"] == "prompt":
        state["cache"].reset()
        out = state["target"](state["ids"], past_key_values=state["cache"], logits_to_keep=1)
        return {"logits": out.logits, "hidden": out.hidden_states, "k": state["cache"].k, "v": state["cache"].vt}
    if c["kind"] == "rows":
        ws = state["ws"]
        state["model"].forward_rows(state["rows"], c["rows"], state["p_min"], state["l_max"], state["cache"], ws,
                                    head_rows=0)
        return {"h": ws.h[:c["rows"]], "k": state["arenas"][0], "v": state["arenas"][1]}
    if c["kind"] == "head":
        m, n, k, mode = c["rows"], c["vocab"], c["k"], c["mode"]
        s = ops.gemm_topk(state["h"], m, state["w"], n, c["hidden"], k, mode, state["parts"], norm_eps=EPS)
        ops.row_topk_merge(state["parts"], m, s, k, mode, None, state["tok"], state["val"])
        return {"tokens": state["tok"], "values": state["val"]}
    if c["kind"] == "propose":
        m, v = c["rows"], c["vocab"]
        ops.warp_probs(state["logits"], m, v, c["temperature"], c["top_p"], state["q"], ws=state["ws"])
        ops.gumbel_topk(state["q"], m, v, c["k"], state["seed"], 1, state["tok"], state["lp"], ws=state["ws"])
        return {"tokens": state["tok"], "logprobs": state["lp"], "q": state["q"]}
    state["sampler"].accept(state["tree"], state["logits"], state["rows"], 0, state["result"], state["keep"],
                            state["n_keep"], state["root"])
    return {"result": state["result"], "keep": state["keep"], "n_keep": state["n_keep"], "root": state["root"],
            "p": state["sampler"].P}


# ------------------------------------------------------------------------------------------------- work
def _layer_weights(shape):
    d, heads, kv, hd, inter = SHAPES[shape]
    return d * (heads + 2 * kv) * hd + d * heads * hd + 3 * d * inter


def work(case):
    if case["kind"] in ("prompt", "rows"):
        d, heads, kv, hd, _ = SHAPES[case["shape"]]
        layers = 2 if case.get("mode") == "draft" else case["layers"]
        weights = layers * _layer_weights(case["shape"]) + (2 * d * d if case.get("mode") == "draft" else 0)
        if case["kind"] == "prompt":
            m = case["tokens"]
            read, seen = 0, m * (m + 1) // 2
            head = BLOCK_VOCAB * d
            out = m * d + BLOCK_VOCAB
        else:
            m = case["rows"]
            _, _, _, anc, lens = _row_table(case, 0)
            read = sum(lens) if case["mode"] == "batch" else lens[0]
            seen, head, out = sum(c + 1 + len(a) for c, a in zip(lens, anc)), 0, m * d
        kv_bytes = layers * 2 * kv * hd * 2 * (read + m)
        return {"bytes": 2 * (weights + head + m * d + out) + kv_bytes,
                "flops": 2 * m * weights + 2 * head + 4 * seen * heads * hd * layers}
    m, v = case.get("rows", 0), case["vocab"]
    if case["kind"] == "head":
        return {"bytes": 2 * case["hidden"] * (v + m) + 8 * m * case["k"], "flops": 2 * m * v * case["hidden"]}
    if case["kind"] == "propose":  # logits read, probabilities written; a draw reads nothing more
        return {"bytes": m * v * (2 + 4) + 8 * m * case["k"], "flops": 10 * m * v}
    parents = _tree_parents([int(b) for b in case["branch"].split(",")])[0]
    m, inner = 1 + len(parents), len(set(parents))
    # logits read, target rows written, the draft rows of the nodes with children read
    return {"bytes": m * v * (2 + 4) + inner * v * 4, "flops": 10 * (m + inner) * v}


def tolerance(case):
    if case["kind"] in ("prompt", "rows"):
        # a bf16 residual stream through two to four layers: the same prompts through the prefill kernels and, 64 rows
        # at a time, through the decode kernels differ by 0.010-0.014 (largest 0.07 of a value or of the rms)
        return {"rel": 0.025, "max": 0.3}
    if case["kind"] == "head":
        return {"rel": 4e-3}  # logits rounded to bf16: 0.0012-0.0017 from the 64-bit ones
    return {"rel": 2e-6, "max": 1e-5, "differ": 0.01}  # 32-bit softmax rows (3e-7 from the 64-bit ones); draws from them


# ------------------------------------------------------------------------------------------------- in 64 bits
def _norm64(h, w):
    return h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, pos):
    """x [rows, heads, hd] rotated to its positions."""
    hd = x.shape[-1]
    ang = pos.double()[:, None] / THETA ** (torch.arange(0, hd, 2, dtype=torch.float64, device="cuda") / hd)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    lo, hi = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([lo * c - hi * s, hi * c + lo * s], -1)


def _layer64(h, sd, i, case, pos, attend):
    """One layer on h [rows, d] in 64 bits; ``attend(q, k, v)`` mixes the rows' values."""
    d, heads, kv, hd, _ = SHAPES[case["shape"]]

    def lin(x, name):
        return x @ sd[f"model.layers.{i}.{name}.weight"].double().T

    x = _norm64(h, sd[f"model.layers.{i}.input_layernorm.weight"])
    q = _rope64(lin(x, "self_attn.q_proj").view(-1, heads, hd), pos)
    k = _rope64(lin(x, "self_attn.k_proj").view(-1, kv, hd), pos)
    v = lin(x, "self_attn.v_proj").view(-1, kv, hd)
    h = h + lin(attend(q, k, v).reshape(h.shape[0], heads * hd), "self_attn.o_proj")
    x = _norm64(h, sd[f"model.layers.{i}.post_attention_layernorm.weight"])
    return h + lin(torch.nn.functional.silu(lin(x, "mlp.gate_proj")) * lin(x, "mlp.up_proj"), "mlp.down_proj")


def _exact_prompt(case, r):
    heads, kv, hd = SHAPES[case["shape"]][1:4]
    sd = _model_tensors(case, r)
    ids = r.ints(case["tokens"], BLOCK_VOCAB)
    m = case["tokens"]
    pos = torch.arange(m, device="cuda")
    hidden_from = pos[None, :] > pos[:, None]

    def attend(q, k, v):
        out = torch.empty_like(q)
        for j in range(heads):
            s = q[:, j] @ k[:, j * kv // heads].T / math.sqrt(hd)
            out[:, j] = torch.softmax(s.masked_fill_(hidden_from, -math.inf), -1) @ v[:, j * kv // heads]
        return out

    h = sd["model.embed_tokens.weight"][ids].double()
    for i in range(case["layers"]):
        h = _layer64(h, sd, i, case, pos, attend)
    hidden = _norm64(h, sd["model.norm.weight"])
    return {"logits": (hidden[-1:] @ sd["lm_head.weight"].double().T)[None], "hidden": hidden[None], "k": None, "v": None}


def _exact_rows(case, r, seed):
    heads, kv, hd = SHAPES[case["shape"]][1:4]
    sd = _model_tensors(case, r)
    bridge = _bridge_tensors(case, r) if case["mode"] == "draft" else None
    ids = r.ints(case["rows"], BLOCK_VOCAB)
    k_all, v_all = _kv_tensors(case, r)
    pos, slot, _, anc, lens = _row_table(case, seed)
    ctx = case["context"]
    h = sd["model.embed_tokens.weight"][ids].double()
    for i in [0, 2] if case["mode"] == "draft" else range(case["layers"]):
        if i == 2 and bridge is not None:
            b = {n.split(".", 1)[1]: t.double() for n, t in bridge.items()}
            x = _norm64(h, b["norm.weight"])
            x = torch.nn.functional.silu(x @ b["mlp.body.0.weight"].T + b["mlp.body.0.bias"])
            h = h + x @ b["mlp.out_proj.weight"].T + b["mlp.out_proj.bias"]

        def attend(q, k, v):
            out = torch.empty_like(q)
            for t in range(q.shape[0]):
                seq = t if case["mode"] == "batch" else 0
                # the committed keys, then this call's rows: itself in a batch, the root and its ancestors in a tree
                new = [t] if case["mode"] == "batch" else [0] + [a - ctx for a in anc[t]]
                kk = torch.cat([k_all[i, seq, :, :lens[t]].double(), k[new].transpose(0, 1)], 1)
                vv = torch.cat([v_all[i, seq, :, :lens[t]].double(), v[new].transpose(0, 1)], 1)
                qq = q[t].view(kv, heads // kv, hd)
                p = torch.softmax(qq @ kk.transpose(1, 2) / math.sqrt(hd), -1)
                out[t] = (p @ vv).view(heads, hd)
            return out

        h = _layer64(h, sd, i, case, torch.tensor(pos, device="cuda"), attend)
    return {"h": h, "k": None, "v": None}


def exact(case, seed):
    r = _Rand(seed)
    if case["kind"] == "prompt":
        return _exact_prompt(case, r)
    if case["kind"] == "rows":
        return _exact_rows(case, r, seed)
    if case["kind"] == "head":
        h, w, norm = _head_tensors(case, r)
        z = _norm64(h.double(), norm) @ w.double().T
        val = z.topk(case["k"], -1).values
        return {"tokens": None, "values": (val - torch.logsumexp(z, -1, keepdim=True) if case["mode"] else val).reshape(-1)}
    v = case["vocab"]
    if case["kind"] == "propose":
        q = _warp64(_sampled_logits(case, r, case["rows"])[0][:, :v], case["temperature"], case["top_p"])
        return {"tokens": None, "logprobs": None, "q": q}
    n = len(_tree_parents([int(b) for b in case["branch"].split(",")])[0])
    p = _warp64(_sampled_logits(case, r, n + 1)[0][:, :v], case["temperature"], case["top_p"])
    return {"result": None, "keep": None, "n_keep": None, "root": None, "p": p}
