"""The attention calls whose speed matters, as a user's program makes them.

Each case is one pass through the public entry points of `intra_amd`: a forward call
(`intra_llm_attn`, `intra_image_attn`) or a training step of one attention layer
(`intra_llm_attn_func`, `intra_image_attn_func` with their gradients).  The sizes are those of this
repository's benchmark and tests: language-model prefill at 32 query / 8 kv heads from a few hundred
tokens to 64 K, FLUX-style images of 1024^2 (64 x 64 latents) and 2048^2 (128 x 128) at 24 heads.
"""
import torch

from intra_amd import intra_image_attn, intra_image_attn_func, intra_llm_attn, intra_llm_attn_func

HEAD_DIM = 128
TEXT_LEN = 512
DEVICE = "cuda"


def _llm(name, mode, pattern, S, B=1, H=32, Hkv=8, layout="bshd", lse=False, softmax="", **args):
    return {"name": name, "family": "llm", "mode": mode, "pattern": pattern, "B": B, "S": S, "H": H, "Hkv": Hkv,
            "layout": layout, "lse": lse, "softmax": softmax, **args}


def _image(name, mode, pattern, width, B=1, H=24, layout="bhsd", lse=False, softmax=""):
    return {"name": name, "family": "image", "mode": mode, "pattern": pattern, "B": B,
            "S": TEXT_LEN + width * width, "H": H, "Hkv": H, "layout": layout, "lse": lse, "softmax": softmax,
            "width": width}


def listed():
    return [
        # The smallest call: a short prompt on one kv head group (what one GPU holds of a model
        # whose heads are spread over eight); latency of the call itself.
        _llm("fwd_scatter8_s1024_h4", "fwd", "scatter", 1024, H=4, Hkv=1, group_num=8),
        # Two prompts of a few thousand tokens, ragged, through a local layer, cut out of the
        # projection's fused q/k/v rows.
        _llm("fwd_window576_s3000_b2", "fwd", "window", 3000, B=2, layout="fused", window=576),
        # Middle prefill length, the gathered-segments layer.
        _llm("fwd_gather1_s8192", "fwd", "gather1", 8192, group_num=8),
        # The benchmark's headline call.
        _llm("fwd_scatter8_s32768", "fwd", "scatter", 32768, group_num=8),
        # The layer that a g2s4 model has 28 of 32 times, at a long prompt.
        _llm("fwd_window576_s32768", "fwd", "window", 32768, window=576),
        # Its other four layers at the longest prompt of the benchmark: the largest forward call.
        _llm("fwd_scatter2_s65536", "fwd", "scatter", 65536, group_num=2),
        # The two alternating layers of image generation, one at each image size, on the
        # (batch, head, token, dim) storage that the image model's processor holds.
        _image("fwd_image_scatter_1024", "fwd", "scatter", 64),
        _image("fwd_image_gather0_2048", "fwd", "gather0", 128),
        # Training (forward with log-sum-exp, backward): the headline layer at full length ...
        _llm("train_scatter8_s32768", "train", "scatter", 32768, group_num=8),
        # ... the local layer with sinks of the long-context fine-tuning setting ...
        _llm("train_window_sink_s8192", "train", "window_sink", 8192, window=575, n_sink=64),
        # ... its global layer with a stripe offset at a length that fits no tile ...
        _llm("train_block_scatter2_s6000", "train", "block_scatter", 6000, group_num=2, block=256, offset=1, n_sink=64),
        # ... and image distillation.
        _image("train_image_gather0_1024", "train", "gather0", 64),
    ]


# Work of the largest listed case; drawn cases stay below it.
_MAX_FLOPS = 4 * HEAD_DIM * 1073774592 * 32


def draw(rng):
    """One more case of the same ranges: both families, both directions, every pattern."""
    mode = rng.choice(["fwd", "fwd", "train"])
    softmax = rng.choice(["", "", "", "exact", "scaled"]) if mode == "fwd" else ""
    lse = mode == "fwd" and rng.random() < 0.25
    if rng.random() < 0.3:
        H = rng.choice([3, 6, 12, 16, 24, 24])
        case = _image("", mode, rng.choice(["scatter", "gather0"]), rng.choice([64, 128]),
                      B=1 if H > 12 else rng.choice([1, 2]), H=H, layout=rng.choice(["bhsd", "bshd"]), lse=lse,
                      softmax=softmax)
        del case["name"]
        return case
    H, Hkv = rng.choice([(4, 1), (8, 2), (16, 4), (32, 8), (32, 8), (32, 8), (32, 32), (16, 8), (8, 1), (28, 4)])
    B = rng.choice([1, 1, 1, 2, 3])
    pattern = rng.choice(["scatter", "gather1", "window", "block_scatter", "window_sink"])
    args = {}
    if pattern == "scatter":
        args = {"group_num": rng.choice([2, 2, 3, 4, 8, 8, 16])}
    elif pattern == "gather1":
        args = {"group_num": 8}
    elif pattern == "window":
        args = {"window": rng.choice([576, 576, 320, 1000, 1088, 2112])}
    elif pattern == "block_scatter":
        args = {"group_num": rng.choice([2, 2, 4, 8]), "block": 256, "offset": rng.choice([0, 1]),
                "n_sink": rng.choice([0, 64, 64])}
    else:
        args = {"window": rng.choice([575, 575, 255, 1023]), "n_sink": rng.choice([4, 64, 64])}
    S = int(256 * 256.0 ** rng.random())
    if pattern == "gather1" or rng.random() < 0.25:
        S = max(64, S // 64 * 64)
    while True:
        case = _llm("", mode, pattern, S, B=B, H=H, Hkv=Hkv, layout=rng.choice(["bshd", "bshd", "fused", "bhsd"]),
                    lse=lse, softmax=softmax, **args)
        del case["name"]
        if work(case)["flops"] <= _MAX_FLOPS:
            return case
        S = S // 128 * 64


def _qkv(case, gen):
    """q, k, v ~ N(0, 1) in bf16, (B, S, heads, 128) views of the storage that `layout` names."""
    B, S, H, Hkv = case["B"], case["S"], case["H"], case["Hkv"]

    def normal(*shape):
        return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.bfloat16)

    if case["layout"] == "fused":  # one row per token: query heads, key heads, value heads
        rows = normal(B, S, H + 2 * Hkv, HEAD_DIM)
        return rows[:, :, :H], rows[:, :, H:H + Hkv], rows[:, :, H + Hkv:]
    if case["layout"] == "bhsd":
        return tuple(normal(B, h, S, HEAD_DIM).transpose(1, 2) for h in (H, Hkv, Hkv))
    return tuple(normal(B, S, h, HEAD_DIM) for h in (H, Hkv, Hkv))


def _call_args(case):
    """Keyword arguments of the entry points (those of the forward calls that name an option too)."""
    if case["family"] == "image":
        args = {"pattern": case["pattern"], "width": case["width"]}
    else:
        args = {"pattern": case["pattern"]}
        args.update({n: case[n] for n in ("group_num", "window", "block", "offset", "n_sink") if n in case})
    return args


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    q, k, v = _qkv(case, gen)
    state = {"family": case["family"], "mode": case["mode"], "args": _call_args(case)}
    if case["mode"] == "train":
        q, k, v = (x.requires_grad_() for x in (q, k, v))
        state["dout"] = torch.randn(q.shape, generator=gen, device=DEVICE, dtype=torch.bfloat16)
    else:
        if case["lse"]:
            state["args"]["return_lse"] = True
        if case["softmax"]:
            state["args"]["softmax"] = case["softmax"]
    state["qkv"] = (q, k, v)
    return state


def run(state):
    q, k, v = state["qkv"]
    if state["mode"] == "train":
        func = intra_image_attn_func if state["family"] == "image" else intra_llm_attn_func
        out = func(q, k, v, **state["args"])
        return (out.detach(),) + torch.autograd.grad(out, (q, k, v), state["dout"])
    attn = intra_image_attn if state["family"] == "image" else intra_llm_attn
    with torch.no_grad():
        return attn(q, k, v, **state["args"])


def _pairs(case):
    """Visible (query, key) pairs per query head and batch entry."""
    S = case["S"]
    if case["family"] == "image":
        image = case["width"] ** 2
        scatter_row = TEXT_LEN + image // 8
        if case["pattern"] == "scatter":
            return S * scatter_row
        return TEXT_LEN * scatter_row + image * (TEXT_LEN + 256)
    pattern = case["pattern"]
    if pattern in ("scatter", "gather1"):
        G = case["group_num"]
        sizes = [len(range(g, S, G)) for g in range(G)] if pattern == "scatter" else [S // G] * G
        return sum(n * (n + 1) // 2 for n in sizes)
    if pattern == "window":
        return sum(t - max(t // 64 * 64 - (case["window"] - 64), 0) + 1 for t in range(S))
    if pattern == "window_sink":
        W, sinks = case["window"], case["n_sink"]
        return sum(min(t + 1, W) + min(sinks, max(t - W + 1, 0)) for t in range(S))
    G, blk, off, sinks = case["group_num"], case["block"], case["offset"], case["n_sink"]
    total = 0
    for qb in range((S + blk - 1) // blk):
        nq = min(blk, S - qb * blk)
        source = (qb + off) % G
        earlier = len(range(source, qb, G))
        total += nq * earlier * blk
        if off != 0 or source == qb % G:
            total += nq * (nq + 1) // 2
        if source != 0 and qb > 0:  # sinks that lie in no visible block
            total += nq * min(sinks, blk)
    return total


def work(case):
    B, S, H, Hkv = case["B"], case["S"], case["H"], case["Hkv"]
    pair_heads = _pairs(case) * H * B
    q_bytes, kv_bytes = 2 * B * S * H * HEAD_DIM, 2 * B * S * Hkv * HEAD_DIM
    if case["mode"] == "fwd":  # q, k, v, out; two products
        return {"bytes": 2 * q_bytes + 2 * kv_bytes + (4 * B * S * H if case["lse"] else 0),
                "flops": 4 * HEAD_DIM * pair_heads}
    # q, k, v, dout read; out, dq, dk, dv written; two products forward, five backward
    return {"bytes": 4 * q_bytes + 4 * kv_bytes, "flops": 14 * HEAD_DIM * pair_heads}


def tolerance(case):
    # Measured against the same pass in float64 (S = 2048 and 4608, every pattern): outputs 2.1e-3 to
    # 2.3e-3, gradients 2.3e-3 to 2.7e-3, which is what rounding weights and results to bf16 gives;
    # four times that.
    return {"rel": 1e-2}


def _visible(case, rows):
    """Mask of the query positions `rows` against every key position."""
    i, j = rows[:, None], torch.arange(case["S"], device=rows.device)[None, :]
    pattern = case["pattern"]
    if case["family"] == "image":
        W = case["width"]

        def group(t):  # text chunks of 64 tokens ride with groups 0..7
            return torch.where(t < TEXT_LEN, t // 64, (t - TEXT_LEN) // W % 2 * 4 + (t - TEXT_LEN) % W % 4)

        scattered = (j < TEXT_LEN) | (group(i) == group(j))
        if pattern == "scatter":
            return scattered

        def in_window(query, key):  # 16 rows or columns around the query's patch of 8, inside the grid
            start = (query // 8 * 8 - 4).clamp(0, W - 16)
            return (key >= start) & (key < start + 16)

        qi, kj = i - TEXT_LEN, j - TEXT_LEN
        window = in_window(qi // W, kj // W) & in_window(qi % W, kj % W)
        return torch.where(i < TEXT_LEN, scattered, (j < TEXT_LEN) | window)
    causal = j <= i
    if pattern == "scatter":
        return causal & (i % case["group_num"] == j % case["group_num"])
    if pattern == "gather1":
        G = case["group_num"]
        return causal & (i // G % G == j // G % G)
    if pattern == "window":
        return causal & (j >= i // 64 * 64 - (case["window"] - 64))
    if pattern == "window_sink":
        return causal & ((i - j < case["window"]) | (j < case["n_sink"]))
    G, off = case["group_num"], case["offset"]
    qb, kb = i // case["block"], j // case["block"]
    source = (qb + off) % G
    own = (kb == qb) & ((source == qb % G) | (off != 0))
    return causal & (((kb < qb) & (kb % G == source)) | own | (j < case["n_sink"]))


def exact(case, seed):
    """The outputs of `run` in float64: dense masked attention, a block of query rows at a time."""
    state = prepare(case, seed)
    q, k, v = (x.detach().transpose(1, 2) for x in state["qkv"])  # (B, heads, S, 128)
    B, H, S, D = q.shape
    train, ratio, scale = case["mode"] == "train", H // k.shape[1], D ** -0.5
    out = torch.empty(B, H, S, D, dtype=torch.float64, device=q.device)
    lse = torch.empty(B, H, S, dtype=torch.float64, device=q.device)
    dq = torch.empty_like(out)
    dk, dv = (torch.zeros(k.shape, dtype=torch.float64, device=q.device) for _ in range(2))
    step = max(64, (1 << 27) // S)
    for r0 in range(0, S, step):
        rows = slice(r0, min(S, r0 + step))
        hidden = ~_visible(case, torch.arange(S, device=q.device)[rows])
        for b in range(B):
            for h in range(H):
                g = h // ratio
                qr, kh, vh = q[b, h, rows].double(), k[b, g].double(), v[b, g].double()
                weights = (qr @ kh.T).mul_(scale).masked_fill_(hidden, -torch.inf)
                lse[b, h, rows] = torch.logsumexp(weights, 1)
                weights = weights.sub_(lse[b, h, rows, None]).exp_()
                out[b, h, rows] = weights @ vh
                if train:
                    do = state["dout"].transpose(1, 2)[b, h, rows].double()
                    dv[b, g] += weights.T @ do
                    ds = (do @ vh.T).sub_((do * out[b, h, rows]).sum(1, keepdim=True)).mul_(weights).mul_(scale)
                    dq[b, h, rows] = ds @ kh
                    dk[b, g] += ds.T @ qr
    if train:
        return tuple(x.transpose(1, 2) for x in (out, dq, dk, dv))
    return (out.transpose(1, 2), lse) if case["lse"] else out.transpose(1, 2)
