"""The workloads on which this framework's speed is measured: OAL grouped quadratic
attention called through its public entry points, as a model or a caller's
adapter calls it.

A case is a dict:
  path      the entry point
              "prepared"  prepare_grouped_hd_block_gemm once, then
                          run_prepared_grouped_hd_block_gemm per call (bf16 on the
                          matrix cores, the factor expanded per call, denominators
                          checked): what the model's layers do
              "grouped"   grouped_oal with ready coefficients (c0, lam, gam),
                          bf16 on the matrix cores, nothing checked
              "public"    oal_attention (fp32 kernels for every input type; all
                          outputs checked; float64 for execution="reference")
              "pair"      the logical per-pair Function with a bf16 plan
              "layer"     the OALAttention module: LoRA projections, rotary
                          embedding and the prepared attention, in bf16
  dtype     of q, k, v
  backward  whether the call is followed by its backward for an upstream
            gradient of `out`: a training step's share, all gradients requested
  batch, q_heads, kv_heads, seq, dim, groups
"""

import math

import torch
import torch.nn.functional as F

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32, "fp64": torch.float64}
_MODEL_SIZES = (2, 4, 6, 8, 10, 10, 12, 12)  # the model configuration's uneven groups
_KERNEL_EPS = 1e-6


def _case(name, path, batch, q_heads, kv_heads, seq, *, dim=64, groups=8, dtype="bf16", backward=True):
    return dict(name=name, path=path, batch=batch, q_heads=q_heads, kv_heads=kv_heads, seq=seq, dim=dim, groups=groups,
                dtype=dtype, backward=backward)


def listed():
    return [
        # a single head in fp32, four groups of 16, forward only: the smallest call there is
        _case("head_256_fp32", "public", 1, 1, 1, 256, groups=4, dtype="fp32", backward=False),
        # the model's heads at the length its quality sessions check a layer with
        _case("check_128", "prepared", 1, 14, 2, 128, backward=False),
        # fine-tuning on short texts: two sequences of ragged length
        _case("train_2x200", "prepared", 2, 14, 2, 200),
        # fine-tuning on ordinary texts, a length that fills no block
        _case("train_2x1000", "prepared", 2, 14, 2, 1000),
        # the operator by itself, one prompt at the headline length, forward
        _case("prefill_4096", "grouped", 1, 14, 2, 4096, backward=False),
        # the headline benchmark: forward and backward, batch 4
        _case("train_4x4096", "grouped", 4, 14, 2, 4096),
        # long context: one sequence of twice the headline batch's tokens
        _case("train_32768", "grouped", 1, 14, 2, 32768),
        # the default route of oal_attention in fp32, trained
        _case("train_2048_fp32", "public", 1, 14, 2, 2048, dtype="fp32"),
        # the default route on bf16 tensors, evaluation only, narrower heads with their own KV head each
        _case("eval_2x777_narrow", "public", 2, 8, 8, 777, dim=48, groups=5, backward=False),
        # per-pair coefficients (64 groups of one dimension), trained
        _case("pair_1024", "pair", 1, 14, 2, 1024, groups=64),
        # the double-precision reference execution that a validation compares with
        _case("reference_256_fp64", "public", 1, 14, 2, 256, dtype="fp64"),
        # a whole attention layer of the model in training
        _case("layer_2x2048", "layer", 2, 14, 2, 2048),
    ]


def draw(rng):
    """One more case of the same ranges: every path, lengths over their logarithm."""
    path, dtype, longest, most = rng.choice([
        # (path, dtype, longest sequence, most query-head tokens)
        ("prepared", "bf16", 8192, 14 * 8192),
        ("prepared", "bf16", 8192, 14 * 8192),
        ("grouped", "bf16", 32768, 14 * 16384),
        ("grouped", "bf16", 32768, 14 * 16384),
        ("public", "fp32", 2048, 14 * 2048),
        ("public", rng.choice(["bf16", "fp16"]), 2048, 14 * 2048),
        ("pair", "bf16", 2048, 14 * 2048),
        ("public", "fp64", 256, 14 * 256),
        ("layer", "bf16", 4096, 14 * 4096),
    ])
    q_heads, kv_heads = (14, 2) if path == "layer" else rng.choice([(14, 2), (14, 2), (14, 2), (8, 2), (4, 4), (8, 1), (1, 1)])
    seq = int(round(math.exp(rng.uniform(math.log(24), math.log(longest)))))
    batch = rng.choice([1, 1, 2, 3, 4, 8])
    while batch > 1 and batch * q_heads * seq > most:
        batch -= 1
    dim = 64 if path in ("grouped", "layer") else rng.choice([64, 64, 64, 48, 32])
    groups = dim if path == "pair" else 8 if path == "layer" else rng.choice([8, 8, 8, 4, 5, 2, 1])
    return dict(path=path, batch=batch, q_heads=q_heads, kv_heads=kv_heads, seq=seq, dim=dim, groups=groups, dtype=dtype,
                backward=path == "layer" or rng.random() < 0.6)


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _group_sizes(groups, dim):
    if groups == len(_MODEL_SIZES) and dim == sum(_MODEL_SIZES):
        return _MODEL_SIZES
    return tuple(dim // groups + (g < dim % groups) for g in range(groups))


def _labels(case, gen):
    """[Hq, D] group ids, the sizes over a permutation of each head's own."""
    sizes = _group_sizes(case["groups"], case["dim"])
    ids = torch.repeat_interleave(torch.arange(len(sizes)), torch.tensor(sizes)).to(torch.int32)
    return torch.stack([ids[torch.randperm(case["dim"], generator=gen)] for _ in range(case["q_heads"])])


def _factor(case, gen):
    """[Hq, P] packed lower-triangular factors of the model's initial distribution."""
    side = case["groups"] + 1
    r, c = torch.tril_indices(side, side)
    rows = []
    for _ in range(case["q_heads"]):
        low = torch.tril(torch.randn((side, side), generator=gen) * 0.15)
        low.diagonal().copy_(0.5 + 0.5 * torch.rand(side, generator=gen))
        rows.append(low[r, c])
    return torch.stack(rows)


def _pair_coefficients(case, gen):
    """(a, b, c) of a positive kernel [1, x] L L^T [1, x]^T + eps over x = scale q o k."""
    d = case["dim"]
    r, c = torch.tril_indices(d, d)
    out = ([], [], [])
    for _ in range(case["q_heads"]):
        low = torch.tril(torch.randn((d + 1, d + 1), generator=gen) * 0.08)
        low.diagonal().copy_(0.4 + 0.3 * torch.rand(d + 1, generator=gen))
        m = low @ low.T
        for part, value in zip(out, (m[0, 0] + 1e-3, 2 * m[0, 1:], m[1:, 1:][r, c])):
            part.append(value)
    return tuple(torch.stack(p) for p in out)


def _expanded(factor, heads):
    """(c0, lam, gam) of packed factors, in the factors' type (the operator's definition)."""
    side = (math.isqrt(1 + 8 * factor.shape[-1]) - 1) // 2
    r, c = torch.tril_indices(side, side, device=factor.device)
    low = torch.zeros((heads, side, side), dtype=factor.dtype, device=factor.device).index_put(
        (torch.arange(heads, device=factor.device)[:, None], r[None], c[None]), factor)
    m = (low.unsqueeze(2) * low.unsqueeze(1)).sum(-1)
    return m[:, 0, 0] + _KERNEL_EPS, 2 * m[:, 0, 1:], m[:, 1:, 1:].contiguous()


def _operands(case, seed):
    """q, k, v ~ N(0, 1) with two dimensions of each head eight times as large, as
    trained projections have them, and the upstream gradient; the small
    operands (labels, factor or coefficients) beside them."""
    dev, dtype = _device(), _DTYPES[case["dtype"]]
    big = torch.Generator(device=dev).manual_seed(seed)
    gen = torch.Generator().manual_seed(seed)
    b, hq, hkv, n, d = (case[x] for x in ("batch", "q_heads", "kv_heads", "seq", "dim"))
    got = {}
    for name, heads in (("q", hq), ("k", hkv), ("v", hkv)):
        t = torch.randn((b, heads, n, d), generator=big, device=dev)
        wide = torch.stack([torch.randperm(d, generator=gen)[:2] for _ in range(heads)])
        gain = torch.ones((heads, d)).scatter(1, wide, 8.0)
        got[name] = (t * gain.to(dev)[None, :, None, :]).to(dtype)
    got["dout"] = torch.randn((b, hq, n, d), generator=big, device=dev).to(dtype)
    if case["path"] == "pair":
        got["a"], got["b"], got["c"] = (t.to(dev) for t in _pair_coefficients(case, gen))
    else:
        got["labels"] = _labels(case, gen).to(dev)
        factor = _factor(case, gen)
        if case["path"] == "grouped":
            got["c0"], got["lam"], got["gam"] = (t.to(dev) for t in _expanded(factor, hq))
        else:
            got["factor"] = factor.to(dev, torch.float64 if case["dtype"] == "fp64" else torch.float32)
    return got


_DIFFERENTIABLE = {"prepared": ("q", "k", "v", "factor"), "public": ("q", "k", "v", "factor"),
                   "grouped": ("q", "k", "v", "c0", "lam", "gam"), "pair": ("q", "k", "v", "a", "b", "c")}


def _layer(case, seed):
    """The model's attention module, LoRA past its zero start, with its inputs."""
    from oal_amd.qwen_oal import OALAttention, QwenOALConfig, rotary_tables

    cfg, dev = QwenOALConfig(), _device()
    torch.manual_seed(seed)
    attn = OALAttention(cfg, 0, torch.Generator().manual_seed(seed))
    for name, p in attn.named_parameters():
        if name.endswith("base.weight") or name.endswith("lora_b"):
            torch.nn.init.normal_(p, std=0.02)
        elif name.endswith("base.bias"):
            torch.nn.init.zeros_(p)
    attn = attn.to(dev)
    for name, p in attn.named_parameters():
        if name != "factor":
            p.data = p.data.to(torch.bfloat16)
    gen = torch.Generator(device=dev).manual_seed(seed)
    shape = (case["batch"], case["seq"], cfg.hidden_size)
    x = torch.randn(shape, generator=gen, device=dev).to(torch.bfloat16).requires_grad_(case["backward"])
    dy = torch.randn(shape, generator=gen, device=dev).to(torch.bfloat16)
    cos, sin = rotary_tables(case["seq"], cfg.head_dim, cfg.rope_theta, dev, torch.bfloat16)
    return attn, x, dy, cos, sin


def prepare(case, seed):
    if case["path"] == "layer":
        attn, x, dy, cos, sin = _layer(case, seed)
        wrt = [x] + [p for p in attn.parameters() if p.requires_grad]
        return dict(case=case, attn=attn, x=x, dy=dy, cos=cos, sin=sin, wrt=wrt)
    state = dict(_operands(case, seed), case=case)
    state["wrt"] = [state[n] for n in _DIFFERENTIABLE[case["path"]]]
    if case["backward"]:
        for t in state["wrt"]:
            t.requires_grad_()
    if case["path"] == "prepared":
        from oal_amd.hd_block_gemm_adapters import prepare_grouped_hd_block_gemm

        state["prepared"] = prepare_grouped_hd_block_gemm(
            state["q"], state["k"], state["v"], state["labels"], state["factor"], kernel_eps=_KERNEL_EPS,
            precision="bf16_tensorcore")
    if case["path"] == "pair":
        from oal_amd.hd_block_gemm import build_hd_block_gemm_plan, canonical_pair_layout

        state["layout"] = canonical_pair_layout(case["dim"])
        state["plan"] = build_hd_block_gemm_plan(
            state["q"], state["k"], state["v"], precision="bf16_tensorcore",
            requested_gradient_mask=(case["backward"],) * 6)
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def _one_gradient(grads):
    """dq, dk, dv and the coefficients' gradients, as one vector per head where
    they come as three: the constant's alone is a near-cancelling sum over
    tokens, a single number per head, with no relative error worth stating."""
    if len(grads) == 4:
        return tuple(grads)
    return (*grads[:3], torch.cat([g.flatten(1) if g.ndim > 1 else g[:, None] for g in grads[3:]], 1))


def _forward(s):
    case = s["case"]
    path, scale = case["path"], case["dim"] ** -0.5
    q, k, v = s["q"], s["k"], s["v"]
    if path == "prepared":
        from oal_amd.hd_block_gemm_adapters import run_prepared_grouped_hd_block_gemm

        return run_prepared_grouped_hd_block_gemm(s["prepared"], q, k, v, s["factor"])
    if path == "grouped":
        from oal_amd.hd_block_gemm_autograd import grouped_oal

        return grouped_oal(q, k, v, s["labels"], s["c0"], s["lam"], s["gam"], scale=scale, floor=0.0, precision="bf16")
    if path == "pair":
        from oal_amd.hd_block_gemm_autograd import _hd_parallel_block_gemm, _hd_parallel_block_gemm_autograd

        call = _hd_parallel_block_gemm_autograd if case["backward"] else _hd_parallel_block_gemm
        return call(q, k, v, s["a"], s["b"], s["c"], scale=scale, eps=_KERNEL_EPS, layout=s["layout"], plan=s["plan"])
    from oal_amd import oal_attention

    return oal_attention(q, k, v, s["labels"], s["factor"], kernel_eps=_KERNEL_EPS, return_unnormalized=True,
                         execution="reference" if case["dtype"] == "fp64" else "auto")


def run(state):
    if state["case"]["path"] == "layer":
        if not state["case"]["backward"]:
            with torch.no_grad():
                return state["attn"](state["x"], state["cos"], state["sin"])
        y = state["attn"](state["x"], state["cos"], state["sin"])
        return (y.detach(), *torch.autograd.grad(y, state["wrt"], state["dy"]))
    if not state["case"]["backward"]:
        with torch.no_grad():
            return _forward(state)
    out, num, den = _forward(state)
    return (out.detach(), den.detach(), *_one_gradient(torch.autograd.grad(out, state["wrt"], state["dout"])))


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    """Each operand read once, each result written once; and the cheaper of the
    two exact evaluations: over token pairs (group sums, the kernel's quadratic
    form, the value product) or through the running state over the
    1 + D + D (D + 1) / 2 features, each with its backward's products."""
    b, hq, hkv, n, d, g = (case[x] for x in ("batch", "q_heads", "kv_heads", "seq", "dim", "groups"))
    size = {"bf16": 2, "fp16": 2, "fp32": 4, "fp64": 8}[case["dtype"]]
    wide = 8 if case["dtype"] == "fp64" else 4
    q, kv = b * hq * n * d, b * hkv * n * d
    features = 1 + d + d * (d + 1) // 2
    pairs = b * hq * n * (n + 1) / 2
    direct = pairs * (2 * d + 2 * g * (g + 1) + 2 * (d + 1))
    state = 2.0 * features * (d + 1) * b * n * (hq + hkv)
    if case["backward"]:
        # dkappa, dq, dk, dv and the coefficients' sums over pairs again; the state form's six contractions for two
        direct += pairs * (2 * (d + 1) + 3 * 2 * d + 3 * g * (g + 1))
        state *= 3
    flops = min(direct, state)
    if case["path"] == "layer":
        hidden, rank = 896, 16
        proj = 2.0 * b * n * hidden * (2 * hq + 2 * hkv) * d
        lora = 2.0 * b * n * rank * (4 * hidden + (2 * hq + 2 * hkv) * d)
        x = b * n * hidden * 2
        weights = (2 * hq + 2 * hkv) * d * hidden * 2
        if not case["backward"]:
            return {"bytes": 2 * x + weights, "flops": flops + proj + lora}
        return {"bytes": 4 * x + weights, "flops": flops + 2 * proj + 3 * lora}
    moved = (q + 2 * kv) * size
    if case["backward"]:
        # q, k, v, dout in; out, den, dq, dk, dv out
        return {"bytes": 2 * moved + 2 * q * size + b * hq * n * wide, "flops": flops}
    return {"bytes": moved + q * size + (q + b * hq * n) * wide, "flops": flops}


def tolerance(case):
    if case["dtype"] == "fp64":
        return {"rel": 1e-13}
    if case["path"] == "layer":
        return {"rel": 4e-2}
    if case["path"] == "public":
        # fp32 throughout; out and the gradients of 16-bit operands are rounded to 16 bits
        return {"rel": {"fp32": 1e-5, "fp16": 1e-3, "bf16": 6e-3}[case["dtype"]]}
    return {"rel": 2e-2}


# ---------------------------------------------------------------------------
# The same in 64 bits, over token pairs in plain torch
# ---------------------------------------------------------------------------


def _attend64(q, k, v, labels, c0, lam, gam, dout=None):
    """Outputs of the operator in float64 and, with `dout`, the gradients of
    sum(out * dout) with respect to (q, k, v, c0, lam, gam). q, k, v, dout
    [B, H, N, D] float64, coefficients per query head. One head and one block
    of queries at a time; every block's gradients by autograd."""
    b, hq, n, d = q.shape
    g = lam.shape[1]
    r = hq // k.shape[1]
    scale = d ** -0.5
    out, num, den = torch.empty_like(q), torch.empty_like(q), q.new_empty((b, hq, n, 1))
    grads = [torch.zeros_like(t) for t in (q, k, v, c0, lam, gam)] if dout is not None else None
    block = max(16, min(512, (1 << 25) // (g * n)))
    for h in range(hq):
        member = (labels[h][None, :] == torch.arange(g, device=q.device)[:, None]).double() * scale
        for bi in range(b):
            for i0 in range(0, n, block):
                i1 = min(n, i0 + block)
                leaves = [q[bi, h, i0:i1], k[bi, h // r, :i1], v[bi, h // r, :i1], c0[h], lam[h], gam[h]]
                leaves = [t.detach().clone().requires_grad_(dout is not None) for t in leaves]
                qb, kb, vb, cb, lb, gb = leaves
                with torch.set_grad_enabled(dout is not None):
                    rows = (member[:, None, :] * qb[None]).reshape(g * (i1 - i0), d)
                    s = (rows @ kb.T).view(g, -1)
                    kappa = (cb + ((lb[:, None] + gb @ s) * s).sum(0)).view(i1 - i0, i1)
                    seen = torch.arange(i1, device=q.device)[None, :] <= torch.arange(i0, i1, device=q.device)[:, None]
                    kappa = torch.where(seen, kappa, torch.zeros((), dtype=kappa.dtype, device=kappa.device))
                    nb, zb = kappa @ vb, kappa.sum(1, keepdim=True)
                    ob = nb / zb
                out[bi, h, i0:i1], num[bi, h, i0:i1], den[bi, h, i0:i1] = ob.detach(), nb.detach(), zb.detach()
                if dout is None:
                    continue
                dqb, dkb, dvb, dcb, dlb, dgb = torch.autograd.grad(ob, leaves, dout[bi, h, i0:i1])
                grads[0][bi, h, i0:i1] = dqb
                grads[1][bi, h // r, :i1] += dkb
                grads[2][bi, h // r, :i1] += dvb
                for into, part in zip(grads[3:], (dcb, dlb, dgb)):
                    into[h] += part
    return out, num, den, grads


def _too_long(case):
    """Pair-wise evaluation in float64 passes about 2e9 values of its group sums a second, backward included."""
    return case["batch"] * case["q_heads"] * case["seq"] ** 2 / 2 * case["groups"] > 3e10


def _through(outputs, inputs, upstream):
    """Gradients of `inputs` for the upstream gradients of `outputs`."""
    return torch.autograd.grad(outputs, inputs, upstream)


def exact(case, seed):
    if _too_long(case):
        return None
    if case["path"] == "layer":
        return _exact_layer(case, seed)
    s = {n: (t.double() if t.is_floating_point() else t) for n, t in _operands(case, seed).items()}
    d, hq, dev = case["dim"], case["q_heads"], s["q"].device
    wrt = [s[n].requires_grad_() for n in _DIFFERENTIABLE[case["path"]][3:]]
    with torch.enable_grad():
        if case["path"] == "pair":
            r, c = torch.tril_indices(d, d, device=dev)
            heads = torch.arange(hq, device=dev)[:, None]
            once = torch.zeros((hq, d, d), dtype=torch.float64, device=dev).index_put((heads, r[None], c[None]), s["c"])
            coef = (s["a"] * 1, s["b"] * 1, once + torch.tril(once, -1).transpose(1, 2))
            labels = torch.arange(d, device=dev)[None].expand(hq, -1)
        elif case["path"] == "grouped":
            coef, labels = (s["c0"], s["lam"], s["gam"]), s["labels"]
        else:
            coef, labels = _expanded(s["factor"], hq), s["labels"]
    values = [t.detach() for t in coef]
    out, num, den, grads = _attend64(s["q"], s["k"], s["v"], labels, *values, s["dout"] if case["backward"] else None)
    if not case["backward"]:
        return out, num, den
    if case["path"] == "grouped":
        return (out, den, *_one_gradient(grads))
    with torch.enable_grad():
        return (out, den, *_one_gradient((*grads[:3], *_through(coef, wrt, grads[3:]))))


def _exact_layer(case, seed):
    """The attention module in float64: the same weights, projections, rotary embedding and attention."""
    attn, x, dy, cos, sin = _layer(case, seed)
    b, n, _ = x.shape
    hq, hkv, d = case["q_heads"], case["kv_heads"], case["dim"]
    names = [m for m, p in attn.named_parameters() if p.requires_grad]
    w = {m: p.detach().double().requires_grad_(m in names) for m, p in attn.named_parameters()}
    x, dy, cos, sin = x.detach().double().requires_grad_(), dy.double(), cos.double(), sin.double()

    def linear(t, m):
        y = F.linear(t, w[m + ".base.weight"], w.get(m + ".base.bias"))
        return y + F.linear(F.linear(t, w[m + ".lora_a"]), w[m + ".lora_b"]) * attn.q_proj.scaling

    def rotated(t):
        return t * cos + torch.cat((-t[..., d // 2:], t[..., :d // 2]), -1) * sin

    with torch.enable_grad():
        q = rotated(linear(x, "q_proj").view(b, n, hq, d).transpose(1, 2))
        k = rotated(linear(x, "k_proj").view(b, n, hkv, d).transpose(1, 2))
        v = linear(x, "v_proj").view(b, n, hkv, d).transpose(1, 2)
        coef = _expanded(w["factor"], hq)
    inner = [t.detach() for t in (q, k, v, *coef)]
    out, _, _, _ = _attend64(*inner[:3], attn.dim_groups, *inner[3:])
    o = out.requires_grad_()
    with torch.enable_grad():
        y = linear(o.transpose(1, 2).reshape(b, n, hq * d), "o_proj")
    if not case["backward"]:
        return y.detach()
    after = [w["o_proj.lora_a"], w["o_proj.lora_b"]]
    do, *d_after = _through(y, [o, *after], dy)
    _, _, _, grads = _attend64(*inner[:3], attn.dim_groups, *inner[3:], do)
    before = [x] + [w[m] for m in names if not m.startswith("o_proj")]
    d_before = _through([q, k, v, *coef], before, grads)
    of = dict(zip(["o_proj.lora_a", "o_proj.lora_b"], d_after))
    of.update(zip([m for m in names if not m.startswith("o_proj")], d_before[1:]))
    return (y.detach(), d_before[0], *(of[m] for m in names))
