"""The work that a user of the Hy3 MoE FFN block has it do, as measurable cases.

A case is one or more resident layers (192 routed experts in Q4_K and the
shared expert in Q4_K or Q8_0, as a checkpoint holds them) and a batch of
tokens that runs through each of them once, by the public entry points of
hy3_amd.MoELayer: forward (the block), forward_residual (the attention's
output added first) or forward_static (the library's own scratch). Each layer
of a case gets a residual stream of its own, as the attention between two MoE
blocks gives it one; a pass starts by writing those streams, since the block
works in place.

Single tokens run over four layers and a few tokens over two: one layer's
touched experts fit the last-level cache, and a decode over a stack of layers
never finds its weights there.
"""
import torch

from hy3_amd import D_FF, D_MODEL, K_MAX, N_EXPERT, ROUTE_SCALE, SHARED, MoELayer

EXPERT_WEIGHTS = 3 * D_MODEL * D_FF
EXPERT_BYTES = EXPERT_WEIGHTS // 256 * 144  # Q4_K: 144 bytes per 256 weights
SHARED_Q8_BYTES = EXPERT_WEIGHTS // 32 * 36  # Q8_0: 36 bytes per 32 weights
STATIC_MAX_TOKENS = 64


def case(name, tokens, layers=1, k=K_MAX, shared="q4k", entry="forward", skewed=False):
    c = {"tokens": tokens, "layers": layers, "k": k, "shared": shared, "entry": entry,
         "skewed": skewed}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one token: the decode step of a chat, four layers of the stack
        case("decode_1", 1, layers=4),
        # the same on a real checkpoint's layer (Q8_0 shared expert), the
        # attention's output added by the block
        case("decode_1_q8_residual", 1, layers=4, shared="q8_0", entry="residual"),
        # three tokens: two or three sequences, or one with a short draft to verify
        case("decode_3_residual", 3, layers=2, entry="residual"),
        # eight sequences decoded together, by the entry that allocates nothing
        case("decode_8_static", 8, shared="q8_0", entry="static"),
        # the small decode batch of a server
        case("decode_32", 32),
        # a ragged decode batch, or a short prompt, with half the experts per token
        case("batch_75_top4", 75, k=4),
        # a prompt's last, short chunk
        case("prefill_201_q8", 201, shared="q8_0", entry="residual"),
        # an ordinary prefill chunk
        case("prefill_512", 512),
        # a ragged longer chunk of a real checkpoint
        case("prefill_1000_q8", 1000, shared="q8_0", entry="residual"),
        # long chunks, evenly routed
        case("prefill_2048", 2048),
        # the longest chunk, with a few experts that most tokens choose
        case("prefill_4096_skewed", 4096, skewed=True),
    ]


def draw(rng):
    tokens = max(1, min(4096, round(2.0 ** rng.uniform(0, 12.1))))
    if tokens > 16 and rng.random() < 0.5:
        tokens |= 1
    entry = rng.choice(["forward", "forward", "residual"])
    if tokens <= STATIC_MAX_TOKENS and rng.random() < 0.25:
        entry = "static"
    # the expert count is 8 in every published configuration, any up to it is accepted
    k = rng.choice([8, 8, 8, 8, 8, 7, 6, 5, 4, 3, 2])
    layers = rng.randint(4, 7) if tokens == 1 else rng.randint(2, 4) if tokens < 8 else 1
    return case(None, min(tokens, 4096), layers=layers, k=k, shared=rng.choice(["q4k", "q8_0"]),
                entry=entry, skewed=rng.random() < 0.3)


# ---- a layer's tensors, from the seed ---------------------------------------

def generator(seed, layer, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(1000003 * seed + layer)
    return g


def small_tensors(case, seed, layer):
    """norm_w, router and expert bias, on the host as a loader has them."""
    g = generator(seed, layer, "cpu")
    norm_w = 1.0 + 0.02 * torch.randn(D_MODEL, generator=g)
    router = 0.02 * torch.randn(N_EXPERT, D_MODEL, generator=g)
    if case["skewed"]:
        rank = torch.randperm(N_EXPERT, generator=g).float()
        bias = 0.5 * (1.0 / (rank + 1.0)) ** 0.8
    else:
        bias = 0.2 * torch.rand(N_EXPERT, generator=g) - 0.1
    return norm_w, router, bias


def quantize_q4k(w):
    """Q4_K blocks [n, 144] of w [n, 256]: eight sub-blocks of 32, each with a
    6-bit scale and minimum of the block's fp16 d and dmin."""
    s = w.view(-1, 8, 32)
    low = s.amin(2).clamp(max=0.0)
    scale = (s.amax(2) - low) / 15.0
    d = (scale.amax(1, keepdim=True) / 63.0).half()
    dmin = ((-low).amax(1, keepdim=True) / 63.0).half()
    sc = (scale / d.float()).round().clamp(0, 63)
    mn = (-low / dmin.float()).round().clamp(0, 63)
    step = (sc * d.float()).clamp(min=1e-12).unsqueeze(2)
    q = ((s + (mn * dmin.float()).unsqueeze(2)) / step).round_().clamp_(0, 15).to(torch.uint8)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    out = torch.empty(s.shape[0], 144, dtype=torch.uint8, device=w.device)
    out[:, 0:2] = d.view(torch.uint8)
    out[:, 2:4] = dmin.view(torch.uint8)
    out[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    out[:, 8:12] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    out[:, 12:16] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    out[:, 16:] = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)
    return out


def dequantize_q4k(blocks):
    """The weights of Q4_K blocks [n, 144], in 64 bits [n, 256]."""
    b = blocks.view(-1, 144)
    d = b[:, 0:2].contiguous().view(torch.float16).double()
    dmin = b[:, 2:4].contiguous().view(torch.float16).double()
    sc = torch.cat([b[:, 4:8] & 63, (b[:, 12:16] & 15) | ((b[:, 4:8] >> 6) << 4)], 1).double()
    mn = torch.cat([b[:, 8:12] & 63, (b[:, 12:16] >> 4) | ((b[:, 8:12] >> 6) << 4)], 1).double()
    qs = b[:, 16:].reshape(-1, 4, 32)
    q = torch.stack([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
    return (q * (d * sc).unsqueeze(2) - (dmin * mn).unsqueeze(2)).view(-1, 256)


def quantize_q8(w):
    """Q8_0 blocks [n, 36] of w [n, 32]: an fp32 scale and 32 signed bytes."""
    d = (w.abs().amax(1, keepdim=True) / 127.0).clamp(min=1e-12)
    return torch.cat([d.view(torch.uint8), (w / d).round().to(torch.int8).view(torch.uint8)], 1)


def dequantize_q8(blocks):
    b = blocks.view(-1, 36)
    return b[:, :4].contiguous().view(torch.float32).double() * b[:, 4:].view(torch.int8).double()


def expert_blocks(case, g, expert):
    """gate, up and down of the next expert that the generator gives."""
    w = 0.02 * torch.randn(EXPERT_WEIGHTS, generator=g, device="cuda")
    if expert == SHARED and case["shared"] == "q8_0":
        return quantize_q8(w.view(-1, 32)).view(3, -1)
    return quantize_q4k(w.view(-1, 256)).view(3, -1)


def streams(case, seed):
    """The residual stream of each layer, and the attention's output."""
    g = generator(seed, 9999)
    shape = (case["layers"], case["tokens"], D_MODEL)
    x = torch.randn(shape, generator=g, device="cuda")
    return x, 0.5 * torch.randn(shape, generator=g, device="cuda")


# ---- a pass ------------------------------------------------------------------

def prepare(case, seed):
    layers = []
    for i in range(case["layers"]):
        # one set of forward buffers for all layers, as an engine keeps it
        layer = MoELayer(case["tokens"], share_scratch_with=layers[0] if layers else None)
        layer.set_router(*(t.numpy() for t in small_tensors(case, seed, i)))
        g = generator(seed, i)
        for e in range(N_EXPERT + 1):
            blocks = expert_blocks(case, g, e)
            if e == SHARED and case["shared"] == "q8_0":
                layer.set_shared_q8_0(*blocks, on_device=True)
            else:
                layer.set_expert_q4k(e, *blocks, on_device=True)
        layers.append(layer)
    x0, attn = streams(case, seed)
    torch.cuda.synchronize()
    return {"case": case, "layers": layers, "x0": x0, "attn": attn, "x": torch.empty_like(x0)}


def run(state):
    c, x = state["case"], state["x"]
    t, k, entry = c["tokens"], c["k"], c["entry"]
    stream = torch.cuda.current_stream().cuda_stream
    x.copy_(state["x0"])
    for i, layer in enumerate(state["layers"]):
        if entry == "residual":
            layer.forward_residual(x[i].data_ptr(), state["attn"][i].data_ptr(), t, k,
                                   ROUTE_SCALE, stream)
        elif entry == "static":
            layer.forward_static(x[i].data_ptr(), t, k, ROUTE_SCALE, stream)
        else:
            layer.forward(x[i].data_ptr(), t, k, ROUTE_SCALE, stream)
    return x


def work(case):
    t, k = case["tokens"], case["k"]
    routed = N_EXPERT * (1.0 - (1.0 - k / N_EXPERT) ** t)  # experts that t even draws touch
    shared = SHARED_Q8_BYTES if case["shared"] == "q8_0" else EXPERT_BYTES
    small = 4 * (N_EXPERT * D_MODEL + D_MODEL + N_EXPERT)
    rows = (3 if case["entry"] == "residual" else 2) * 4 * D_MODEL * t
    flops = t * 2 * ((k + 1) * EXPERT_WEIGHTS + N_EXPERT * D_MODEL)
    return {"bytes": int(case["layers"] * (routed * EXPERT_BYTES + shared + small + rows)),
            "flops": case["layers"] * flops}


def tolerance(case):
    # fp16 activations against exact weights, sums in 32 bits: 2.6e-4 to 3.1e-4
    # from exact() at every size
    return {"rel": 1e-3, "max": 2e-2}


def exact(case, seed):
    """The block in 64 bits: RMSNorm, sigmoid scores, the k largest of score +
    bias, renormalised weights, SwiGLU experts, the weighted sum."""
    x, attn = streams(case, seed)
    k = case["k"]
    out = x.double()
    if case["entry"] == "residual":
        out = (x + attn).double()  # the add is the block's fp32 one
    for i in range(case["layers"]):
        norm_w, router, bias = (t.cuda().double() for t in small_tensors(case, seed, i))
        y = out[i]
        s = y * norm_w / torch.sqrt(y.pow(2).mean(1, keepdim=True) + 1e-5)
        sig = torch.sigmoid(s @ router.t())
        ids = torch.topk(sig + bias, k, dim=1).indices
        w = torch.gather(sig, 1, ids)
        w = ROUTE_SCALE * w / (w.sum(1, keepdim=True) + 1e-20)
        delta = torch.zeros_like(y)
        g = generator(seed, i)
        for e in range(N_EXPERT + 1):
            blocks = expert_blocks(case, g, e)
            t, place = (ids == e).nonzero(as_tuple=True)
            weight = w[t, place]
            if e == SHARED:
                t = torch.arange(case["tokens"], device="cuda")
                weight = torch.ones(t.numel(), dtype=torch.float64, device="cuda")
            if t.numel() == 0:
                continue
            read = dequantize_q8 if e == SHARED and case["shared"] == "q8_0" else dequantize_q4k
            gate, up, down = read(blocks).view(3, -1)
            h = s[t] @ gate.view(D_FF, D_MODEL).t()
            h = h * torch.sigmoid(h) * (s[t] @ up.view(D_FF, D_MODEL).t())
            delta.index_add_(0, t, weight.unsqueeze(1) * (h @ down.view(D_MODEL, D_FF).t()))
        out[i] = y + delta
    return out
