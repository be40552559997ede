"""The calls a user of this package makes, as measurable cases.

Shapes are the package's own workloads: the plumbing shape, the 512x512 and
1280x832 images (1280 and 4416 tokens, 30 heads of 128), the packed
mixed-resolution batch (1280 + 1216 + 4416 tokens), the k-tuple batch of four
padded 1024x1024 samples, and ragged sizes between them.  ``call`` says what
one pass does:

* ``fwd``       one forward op on q, k, v: ``sage_attn_masked`` (int8 QK, bf16
                P.V) for a tile mask in that variant, ``sage_attn_ext`` otherwise
* ``bwd``       one backward op on q, k, v, out, lse and dO
* ``train``     forward op and its autograd backward
* ``qkv``       ``sage_attn_qkv_masked`` on the QKV projection output
* ``qkv_train`` the same with its autograd backward (gradient of the projection)
* ``producer``  ``fused_qkv_postprocess`` with its autograd backward
"""

import math

import torch

import futudiffu_amd  # noqa: F401  (registers the ops)
import futudiffu_amd.fused_kernels  # noqa: F401
from futudiffu_amd import block_mask as BM

_LOG2E = math.log2(math.e)
_EPS = 1e-5


def _case(call, B, H, N, D, qk="int8", pv="bf16", gran="token", mask="none", segments="", text=0):
    return dict(call=call, B=B, H=H, N=N, D=D, qk=qk, pv=pv, gran=gran, mask=mask, segments=segments, text=text)


def listed():
    named = {
        # a unit-test sized call: nothing but launches and latency
        "plumbing_fwd": _case("fwd", 1, 4, 256, 64, gran="block64"),
        # a small fine-tuning step on a ragged two-segment pack, through autograd
        "small_train": _case("train", 2, 4, 333, 64, mask="tile", segments="200,133"),
        # one 512x512 image: less than one round of workgroups
        "dit512_fwd": _case("fwd", 1, 30, 1280, 128, pv="fp8"),
        # one 1280x832 image, the benchmark's headline call
        "dit1280_fwd": _case("fwd", 1, 30, 4416, 128, pv="fp8"),
        # the package's default variant (fp8 QK, bf16 P.V) on a ragged pair of samples
        "ragged_fp8_fwd": _case("fwd", 2, 30, 1337, 128, qk="fp8"),
        # the attention layer from the QKV projection output (producer inside the quantization)
        "dit1280_qkv_fwd": _case("qkv", 1, 30, 4416, 128, mask="tile", segments="4416"),
        # RMSNorm + RoPE + split and their gradient, as the model's layer runs them by themselves
        "dit1280_producer": _case("producer", 1, 30, 4416, 128),
        # packed mixed-resolution batch in the production variant with the reference tile mask
        "packed_tile_fwd": _case("fwd", 1, 30, 6912, 128, mask="tile", segments="1280,1216,4416"),
        # four 1024x1024 samples with padded text keys (the largest forward)
        "ktuple_fwd": _case("fwd", 4, 30, 4352, 128, pv="fp8", mask="keypad", text=256),
        # training backward of one 1280x832 image
        "dit1280_bwd": _case("bwd", 1, 30, 4416, 128),
        # training backward of the packed batch with exact document ids
        "packed_doc_bwd": _case("bwd", 1, 30, 6912, 128, mask="doc", segments="1280,1216,4416"),
        # a training step of the attention layer on a pack of odd segment lengths
        "packed_qkv_train": _case("qkv_train", 1, 30, 3071, 128, mask="tile", segments="1003,771,1297"),
    }
    out = []
    for name, c in named.items():
        c["name"] = name
        out.append(c)
    return out


def _segments(case):
    return [int(x) for x in case["segments"].split(",")] if case["segments"] else [case["N"]]


def draw(rng):
    """Calls of the same kinds over the range of sizes: 64 to 6912 tokens, odd ones among them."""
    while True:
        call = rng.choice(["fwd", "fwd", "fwd", "bwd", "bwd", "train", "qkv", "qkv_train", "producer"])
        n = int(round(math.exp(rng.uniform(math.log(64), math.log(6912)))))
        if rng.random() < 0.4:
            n = max(64, n // 64 * 64)
        b = rng.choice([1, 1, 2, 4])
        h = rng.choice([3, 4, 8, 12, 16, 24, 30, 30])
        d = rng.choice([64, 128, 128])
        c = _case(call, b, h, n, d)
        if call in ("fwd", "bwd", "train"):
            c["qk"] = rng.choice(["int8", "int8", "fp8"])
            c["mask"] = rng.choice(["none", "none", "tile", "doc", "keypad"])
        if call in ("qkv", "qkv_train"):
            c["mask"] = "tile"
        if call in ("fwd", "train"):
            c["pv"] = rng.choice(["fp8", "bf16"])
        if call == "fwd" and rng.random() < 0.15:
            c["gran"] = "block64"
        if c["mask"] in ("tile", "doc"):
            cuts = sorted(rng.sample(range(1, n), rng.choice([1, 2, 3]))) if n > 8 else []
            edges = [0] + cuts + [n]
            c["segments"] = ",".join(str(y - x) for x, y in zip(edges, edges[1:]))
        if c["mask"] == "keypad":
            c["text"] = min(n // 2, 256)
        # no dearer than the largest listed case of its direction
        if work(c)["flops"] <= (9e11 if call in ("fwd", "qkv") else 6e11) and b * h * n * d <= 4 * 30 * 4352 * 128:
            return c


def _valid_counts(case):
    """Valid text tokens of each sample of a key-padded batch."""
    text = case["text"]
    return [max(1, text - (37 + 61 * i) % max(text, 2)) for i in range(case["B"])]


def _tile_mask(case, device):
    return BM.build_block_mask(_segments(case), case["N"], device=device)


def _doc_ids(case, device):
    if case["mask"] == "doc":
        return BM.build_doc_ids(_segments(case), case["N"], device=device, batch=case["B"])
    valid = torch.ones(case["B"], case["N"], dtype=torch.bool)
    for i, x in enumerate(_valid_counts(case)):
        valid[i, x:case["text"]] = False
    return torch.where(valid, 0, -1).to(torch.int32).to(device)


def _visible(case, b, device):
    """Boolean [N, N] visibility (query, key) of sample b, or None for all."""
    n = case["N"]
    if case["mask"] == "none":
        return None
    if case["mask"] == "tile":
        m = _first_token_mask(case, device)
        return m.repeat_interleave(128, 0)[:n].repeat_interleave(64, 1)[:, :n]
    if case["mask"] == "doc":
        doc = torch.repeat_interleave(torch.arange(len(_segments(case)), device=device),
                                      torch.tensor(_segments(case), device=device))
        return doc[:, None] == doc[None, :]
    keys = torch.ones(n, dtype=torch.bool, device=device)
    keys[_valid_counts(case)[b]:case["text"]] = False
    return keys[None, :].expand(n, n)


def _first_token_mask(case, device):
    """The 128 x 64 tile rule in plain torch: a tile follows the documents of its first tokens."""
    n = case["N"]
    segs = torch.tensor(_segments(case), device=device)
    doc = torch.repeat_interleave(torch.arange(len(segs), device=device), segs)
    return doc[torch.arange(0, n, 128, device=device)][:, None] == doc[torch.arange(0, n, 64, device=device)][None, :]


def _pairs(case):
    """Visible (query, key) pairs of one head, summed over the samples."""
    n, b = case["N"], case["B"]
    if case["mask"] == "tile":
        m = _first_token_mask(case, "cpu").double()
        rows = torch.tensor([min(128, n - x) for x in range(0, n, 128)], dtype=torch.float64)
        cols = torch.tensor([min(64, n - x) for x in range(0, n, 64)], dtype=torch.float64)
        return b * float(rows @ m @ cols)
    if case["mask"] == "doc":
        return b * float(sum(s * s for s in _segments(case)))
    if case["mask"] == "keypad":
        return float(sum(n * (n - case["text"] + x) for x in _valid_counts(case)))
    return float(b * n * n)


def work(case):
    """Inputs read once and outputs written once; 4D operations per visible pair forward, 10D backward."""
    b, h, n, d, call = (case[x] for x in ("B", "H", "N", "D", "call"))
    rows = b * h * n * d * 2     # one bf16 [B, H, N, D]
    lse = b * h * n * 4
    rot = b * n * d // 2 * 16    # the fp32 rotation matrices
    pairs = _pairs(case) * h * d if call != "producer" else 0.0
    nbytes = {"fwd": 4 * rows + lse, "bwd": 8 * rows + lse, "train": 8 * rows + lse,
              "qkv": 4 * rows + lse + rot, "qkv_train": 8 * rows + lse + rot, "producer": 12 * rows + rot}[call]
    flops = {"fwd": 4, "qkv": 4, "bwd": 10, "train": 14, "qkv_train": 14, "producer": 0}[call] * pairs
    if call == "producer":
        flops = 30.0 * 3 * b * h * n * d
    return {"bytes": float(nbytes), "flops": float(flops)}


def _inputs(case, seed):
    """q, k, v ~ N(0, 1) with a per-channel offset in K, or the projection output with
    norm weights and rotations; the incoming gradients ~ N(0, 1)."""
    b, h, n, d, call = (case[x] for x in ("B", "H", "N", "D", "call"))
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(seed)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    st = {}
    if call in ("fwd", "bwd", "train"):
        st["q"] = rand(b, h, n, d).bfloat16()
        st["k"] = (rand(b, h, n, d) + 2.0 * rand(b, h, 1, d)).bfloat16()
        st["v"] = rand(b, h, n, d).bfloat16()
        if call != "fwd":
            st["dout"] = rand(b, h, n, d).bfloat16()
    else:
        st["qkv"] = rand(b, n, 3 * h * d).bfloat16()
        st["qw"] = 1.0 + 0.1 * rand(d)
        st["kw"] = 1.0 + 0.1 * rand(d)
        ang = torch.rand(b, n, 1, d // 2, generator=g, device=dev) * 6.283
        cs, sn = torch.cos(ang), torch.sin(ang)
        st["freqs"] = torch.stack([torch.stack([cs, -sn], -1), torch.stack([sn, cs], -1)], -2)
        if call == "qkv_train":
            st["dout"] = rand(b, n, h * d).bfloat16()
        if call == "producer":
            st["grads"] = [rand(b, h, n, d).bfloat16() for _ in range(3)]
    return st


def _forward(st):
    case, sm = st["case"], st["sm"]
    if case["mask"] == "tile" and (case["qk"], case["pv"], case["gran"]) == ("int8", "bf16", "token"):
        return torch.ops.futudiffu_ii.sage_attn_masked(st["q"], st["k"], st["v"], st["mask"], sm)
    return torch.ops.futudiffu_ii.sage_attn_ext(st["q"], st["k"], st["v"], st["mask"], st["doc"], sm, case["qk"],
                                                case["pv"], case["gran"], True)


def prepare(case, seed):
    st = _inputs(case, seed)
    dev = torch.device("cuda:0")
    st["case"], st["sm"] = dict(case), 1.0 / math.sqrt(case["D"])
    st["mask"] = _tile_mask(case, dev) if case["mask"] == "tile" else None
    st["doc"] = _doc_ids(case, dev) if case["mask"] in ("doc", "keypad") else None
    if case["call"] == "bwd":
        st["out"], st["lse"] = _forward(st)
    if case["call"] == "train":
        for x in ("q", "k", "v"):
            st[x].requires_grad_(True)
    if case["call"] in ("qkv_train", "producer"):
        st["qkv"].requires_grad_(True)
    return st


def run(state):
    st, call = state, state["case"]["call"]
    h, d = st["case"]["H"], st["case"]["D"]
    if call == "fwd":
        return _forward(st)
    if call == "bwd":
        return torch.ops.futudiffu_ii.sage_bwd_ext(st["q"], st["k"], st["v"], st["out"], st["lse"], st["dout"],
                                                   st["mask"], st["doc"], st["sm"], st["case"]["qk"], True)
    if call == "train":
        out, lse = _forward(st)
        return [out.detach(), lse.detach(), *torch.autograd.grad(out, (st["q"], st["k"], st["v"]), st["dout"])]
    if call == "producer":
        outs = torch.ops.futudiffu.fused_qkv_postprocess(st["qkv"], st["qw"], st["kw"], st["freqs"], h, d, _EPS)
        return [*(t.detach() for t in outs), *torch.autograd.grad(outs, (st["qkv"],), st["grads"])]
    out, lse = torch.ops.futudiffu_ii.sage_attn_qkv_masked(st["qkv"], st["qw"], st["kw"], st["freqs"], st["mask"], h, d,
                                                           _EPS, st["sm"])
    if call == "qkv":
        return [out, lse]
    return [out.detach(), lse.detach(), *torch.autograd.grad(out, (st["qkv"],), st["dout"])]


def tolerance(case):
    """Four times the largest relative difference seen when the 64-token blocks of keys and
    queries are summed in another order: 3.1e-3 where P is rounded to bf16 before P.V (out, and
    gradients that follow it: 1.9e-3), one bf16 rounding of a few results elsewhere."""
    if case["call"] == "producer" or (case["call"] == "fwd" and case["pv"] == "fp8"):
        return {"rel": 4e-3}
    return {"rel": 1.2e-2}


def _attention64(q, k, v, vis, sm, dout=None):
    """Attention of one head in 64 bits: out, base-2 LSE of the smoothed scores, gradients."""
    mu = k.mean(0).bfloat16().double()  # the key mean in the package's input precision
    s = (q @ (k - mu).T) * sm
    if vis is not None:
        s = s.masked_fill(~vis, float("-inf"))
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse[:, None])
    out = p @ v
    if dout is None:
        return out, lse * _LOG2E, None
    dp = dout @ v.T
    ds = p * (dp - (dout * out).sum(-1, keepdim=True)) * sm
    return out, lse * _LOG2E, (ds @ k, ds.T @ q, p.T @ dout)


def _producer64(st, case):
    """Split, RMSNorm and rotation in 64 bits: q, k, v [B, H, N, D]."""
    b, h, n, d = (case[x] for x in ("B", "H", "N", "D"))
    x = st["qkv"].detach().double().view(b, n, 3, h, d).requires_grad_(True)
    rot = st["freqs"].double()  # [B, N, 1, D/2, 2, 2]

    def one(y, w):
        y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + _EPS) * w.double()
        e, o = y[..., 0::2], y[..., 1::2]
        return torch.stack([rot[..., 0, 0] * e + rot[..., 0, 1] * o, rot[..., 1, 0] * e + rot[..., 1, 1] * o],
                           -1).flatten(-2)

    q, k, v = one(x[:, :, 0], st["qw"]), one(x[:, :, 1], st["kw"]), x[:, :, 2]
    return x, [t.transpose(1, 2) for t in (q, k, v)]


def exact(case, seed):
    b, h, n, d, call = (case[x] for x in ("B", "H", "N", "D", "call"))
    st = _inputs(case, seed)
    dev, sm = torch.device("cuda:0"), 1.0 / math.sqrt(d)
    x = None
    if call in ("qkv", "qkv_train", "producer"):
        x, (q, k, v) = _producer64(st, case)
        if call == "producer":
            grad, = torch.autograd.grad((q, k, v), (x,), [t.double() for t in st["grads"]])
            return [q.detach(), k.detach(), v.detach(), grad.reshape(b, n, 3 * h * d)]
    else:
        q, k, v = (st[t].double() for t in ("q", "k", "v"))
    dout = None
    if "dout" in st:
        dout = st["dout"].double()
        if call == "qkv_train":
            dout = dout.view(b, n, h, d).transpose(1, 2)
    out = torch.empty(b, h, n, d, dtype=torch.float64, device=dev)
    lse = torch.empty(b, h, n, dtype=torch.float64, device=dev)
    grads = [torch.empty_like(out) for _ in range(3)] if dout is not None else None
    with torch.no_grad():
        for i in range(b):
            vis = _visible(case, i, dev)
            for j in range(h):
                o, l, gr = _attention64(q[i, j].contiguous(), k[i, j].contiguous(), v[i, j].contiguous(), vis, sm,
                                        None if dout is None else dout[i, j].contiguous())
                out[i, j], lse[i, j] = o, l
                if gr is not None:
                    for t, y in zip(grads, gr):
                        t[i, j] = y
    lse = lse.view(b * h, n)
    if call == "fwd":
        return out, lse
    if call == "bwd":
        return tuple(grads)
    if call == "train":
        return [out, lse, *grads]
    merged = out.transpose(1, 2).reshape(b, n, h * d)
    if call == "qkv":
        return [merged, lse]
    dqkv, = torch.autograd.grad((q, k, v), (x,), grads)
    return [merged, lse, dqkv.reshape(b, n, 3 * h * d)]
