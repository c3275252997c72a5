"""The work this library does for its users, as cases that can be timed: single quantized linears, the two feed-forward
chains and the whole transformer blocks, through the public entry points and over the range of sizes, data types and quant
levels in use.

FLUX: width 3072, 24 heads of 128, 4096 image tokens at 1024 x 1024 and 6400 at 1280 x 1280 beside up to 512 text tokens;
SDXL: widths 640 (10 heads) and 1280 (20 heads), 4096 and 1024 tokens at 1024 x 1024, two images in a batch where classifier-free
guidance is on, 77 text tokens of width 2048.  Weights are random, ~ N(0, 0.02) or ~ N(0, 1/sqrt(K)) as the quantisers leave
them; activations ~ N(0, 1) with outlier channels where smoothing exists for them.
"""
import math

import torch

from lyradiff_amd import flux_ops, ops, sdxl_int8, weights

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
FLUX_DIM, FLUX_HEAD = 3072, 128
SDXL_TEXT, SDXL_TEXT_DIM, SDXL_HEAD = 77, 2048, 64
LEVELS = {"fp8": "FP8_W8A8", "fp8_full": "FP8_W8A8_FULL", "int4": "INT4_W4A4", "int4_full": "INT4_W4A4_FULL"}
RANK, GROUP = 32, 64

# (n, k) of the linears of the two models
FLUX_LINEARS = [(3 * FLUX_DIM, FLUX_DIM), (FLUX_DIM, FLUX_DIM), (4 * FLUX_DIM, FLUX_DIM), (FLUX_DIM, 4 * FLUX_DIM), (6 * FLUX_DIM, FLUX_DIM)]
SDXL_LINEARS = [(n * d, k * d) for d in (640, 1280) for n, k in ((1, 1), (3, 1), (8, 1), (1, 4))]


def listed():
    return [
        # attention projection of SDXL's 1280-wide stage, per-token scales: the smallest linear that runs in a loop
        {"name": "int8_linear_1024", "op": "int8_linear", "tokens": 1024, "n": 1280, "k": 1280, "dtype": "fp16", "dynamic": True},
        # SDXL's 640-wide GEGLU feed-forward with per-token scales at 1024 x 1024
        {"name": "int8_geglu_4096", "op": "int8_geglu", "tokens": 4096, "dim": 640, "dtype": "fp16"},
        # modulation linear of a FLUX block: one row, six chunks
        {"name": "fp8_modulation_1", "op": "fp8_linear", "tokens": 1, "n": 6 * FLUX_DIM, "k": FLUX_DIM, "dtype": "bf16", "dynamic": False},
        # QKV projection of a ragged number of text tokens, dynamic scale, the other 16-bit type
        {"name": "fp8_linear_333", "op": "fp8_linear", "tokens": 333, "n": 3 * FLUX_DIM, "k": FLUX_DIM, "dtype": "fp16", "dynamic": True},
        # FLUX feed-forward with dynamic scales at 1024 x 1024 (image and text tokens)
        {"name": "fp8_mlp_4608", "op": "fp8_mlp", "tokens": 4608, "dim": FLUX_DIM, "dtype": "bf16"},
        # FLUX attention projection, W4A4 with its low-rank branch
        {"name": "w4a4_linear_4608", "op": "w4a4_linear", "tokens": 4608, "n": FLUX_DIM, "k": FLUX_DIM, "dtype": "bf16"},
        # weight-only linear on the text states of two prompts
        {"name": "weight_only_154", "op": "weight_only", "tokens": 154, "n": 1280, "k": 2048, "dtype": "fp16", "kind": "int8", "group": 0, "zeros": False},
        # weight-only linear of FLUX's feed-forward, int4 with groups and zero points
        {"name": "weight_only_4608", "op": "weight_only", "tokens": 4608, "n": 4 * FLUX_DIM, "k": FLUX_DIM, "dtype": "bf16", "kind": "int4", "group": 128, "zeros": True},
        # whole FLUX double-stream block, FP8, 1024 x 1024
        {"name": "flux_double_fp8", "op": "flux_double", "level": "fp8_full", "image": 4096, "text": 512, "dtype": "bf16"},
        # whole FLUX single-stream block, FP8, 1280 x 1280
        {"name": "flux_single_fp8", "op": "flux_single", "level": "fp8", "image": 6400, "text": 512, "dtype": "bf16"},
        # whole FLUX single-stream block, INT4, 1024 x 1024
        {"name": "flux_single_int4", "op": "flux_single", "level": "int4_full", "image": 4096, "text": 512, "dtype": "bf16"},
        # SDXL transformer block at the highest INT8 level, batch of two
        {"name": "sdxl_block_int8", "op": "sdxl_block", "level": 3, "batch": 2, "tokens": 4096, "dim": 640, "dtype": "fp16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["int8_linear", "int8_geglu", "fp8_linear", "fp8_mlp", "w4a4_linear", "weight_only", "flux_double", "flux_single", "sdxl_block"])
    case = {"op": op, "dtype": rng.choice(["bf16", "fp16"])}
    if op == "int8_linear":
        n, k = rng.choice(SDXL_LINEARS)
        case.update(tokens=_log(rng, 64, 8192), n=n, k=k, dynamic=rng.random() < 0.5)
    elif op == "int8_geglu":
        case.update(tokens=_log(rng, 256, 8192), dim=rng.choice([640, 1280]))
    elif op == "fp8_linear":
        n, k = rng.choice(FLUX_LINEARS)
        case.update(tokens=_log(rng, 1, 6912), n=n, k=k, dynamic=rng.random() < 0.5)
    elif op == "fp8_mlp":
        case.update(tokens=_log(rng, 256, 6912), dim=FLUX_DIM)
    elif op == "w4a4_linear":
        n, k = rng.choice(FLUX_LINEARS[:4])
        case.update(tokens=_log(rng, 64, 4608), n=n, k=k)
    elif op == "weight_only":
        n, k = rng.choice(FLUX_LINEARS[:4] + [(1280, 2048), (1280, 1280)])
        group = rng.choice([0, 64, 128])
        case.update(tokens=_log(rng, 1, 4608), n=n, k=k, kind=rng.choice(["int8", "int4"]), group=group, zeros=group > 0 and rng.random() < 0.5)
    elif op in ("flux_double", "flux_single"):
        case.update(level=rng.choice(sorted(LEVELS)), image=rng.randint(16, 80) * rng.randint(16, 80), text=rng.randint(64, 512))
        if op == "flux_double" or case["level"].startswith("int4"):
            case["image"] = min(case["image"], 4608)
    else:
        dim = rng.choice([640, 1280])
        side = 32 if dim == 1280 else 64
        case.update(level=rng.choice([1, 2, 3]), batch=rng.choice([1, 2]), tokens=rng.randint(side // 2, side) * rng.randint(side // 2, side), dim=dim)
    return case


class _Maker:
    """Random tensors of one seed, made on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float32):
        return torch.empty(shape, device="cuda").normal_(mean, std, generator=self.g).to(dtype)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.empty(shape, device="cuda").uniform_(lo, hi, generator=self.g)

    def codes(self, *shape, hi=127):
        return torch.randint(-hi, hi + 1, shape, generator=self.g, device="cuda", dtype=torch.int8)

    def activation(self, rows, k, dtype, std=1.0, outlier=0.0):
        """~ N(0, std); with `outlier`, 1 % of the channels that many times larger, at places of this seed's own."""
        x = self.normal(rows, k, std=std)
        if outlier:
            cols = torch.randperm(k, generator=self.g, device="cuda")[: max(1, k // 100)]
            x[:, cols] *= outlier
        return x.to(dtype)


def _int8_entries(mk, name, n, k, input_amax):
    """A SmoothQuant linear as its export leaves it: codes whose weights are ~ N(0, 1/sqrt(K)) in size."""
    scale = k ** -0.5 / 73.0
    return {name + ".weight_int8": mk.codes(n, k), name + ".weight_quant_scale": mk.uniform(n, lo=0.5 * scale, hi=1.5 * scale),
            name + ".input_quant_scale": torch.full((1,), input_amax / 127.0, device="cuda"), name + ".pre_quant_scale": mk.uniform(k, lo=0.7, hi=1.3)}


def _fp8_entries(mk, name, n, k, dtype, input_amax):
    return {name + ".weight": mk.normal(n, k, std=0.02, dtype=dtype), name + ".bias": mk.normal(n, std=0.02, dtype=dtype),
            name + "_input_scale": torch.full((1,), input_amax / 448.0, device="cuda")}


def _w4a4_entries(mk, name, n, k, dtype, bias=True):
    words, scale = ops.w4a4_quant(mk.normal(n, k, std=0.02))
    sd = {name + "packed_weight": words.view(torch.int8), name + "weight_scale": scale, name + "smooth": mk.uniform(k, lo=0.7, hi=1.4),
          name + "lora_up": mk.normal(n, RANK, std=0.05, dtype=dtype), name + "lora_down": mk.normal(RANK, k, std=0.02, dtype=dtype)}
    if bias:
        sd[name + "bias"] = mk.normal(n, std=0.02, dtype=dtype)
    return sd


def _prepare_flux(case, mk, dtype):
    d, tokens = FLUX_DIM, case["image"] + case["text"]
    int4, double = case["level"].startswith("int4"), case["op"] == "flux_double"
    full = case["level"].endswith("full")
    sd = {}

    def fp8(name, n, k, amax):
        sd.update(_fp8_entries(mk, "b." + name, n, k, dtype, amax))

    def quantised(name, n, k, amax):  # an FP8 or a W4A4 linear, as the level has it
        if int4:
            sd.update(_w4a4_entries(mk, "b." + name + ".", n, k, dtype))
        else:
            fp8(name, n, k, amax)

    norms = ("norm_q", "norm_k", "norm_added_q", "norm_added_k") if double else ("norm_q", "norm_k")
    for n in norms:
        sd[f"b.attn.{n}.weight"] = mk.uniform(FLUX_HEAD, lo=1.0, hi=1.8).to(dtype)
    for n in ("norm1", "norm1_context") if double else ("norm",):
        fp8(n + ".linear", (6 if double else 3) * d, d, 4.0)
        if not full:
            del sd[f"b.{n}.linear_input_scale"]
    quantised("attn.to_qkv", 3 * d, d, 8.0)
    if double:
        quantised("attn.to_added_qkv", 3 * d, d, 8.0)
        quantised("attn.to_out.0", d, d, 4.0)
        quantised("attn.to_add_out", d, d, 4.0)
        for ff in ("ff.", "ff_context."):
            quantised(ff + "net.0.proj", 4 * d, d, 8.0)
            fp8(ff + "net.2", d, 4 * d, 6.0)
        op = flux_ops.FluxTransformerBlockOp
    else:
        quantised("proj_mlp", 4 * d, d, 8.0)
        if int4:
            sd.update(_w4a4_entries(mk, "b.proj_out.linears.0.", d, d, dtype))
            sd.update(_w4a4_entries(mk, "b.proj_out.linears.1.linear.", d, 4 * d, dtype, bias=False))
        else:
            fp8("proj_out", d, 5 * d, 6.0)
        op = flux_ops.FluxSingleTransformerBlockOp
    block = op(case["dtype"], d, d // FLUX_HEAD, FLUX_HEAD, 4, flux_ops.LyraQuantLevel[LEVELS[case["level"]]].value)
    block.initialize()
    block.reload_model_from_state_dict("b.", sd, "cuda")
    angle = mk.uniform(1, tokens, FLUX_HEAD // 2, hi=2 * math.pi)
    rope = torch.stack([angle.cos(), -angle.sin(), angle.sin(), angle.cos()], dim=-1).view(1, tokens, FLUX_HEAD // 2, 2, 2).to(dtype)
    temb = torch.nn.functional.silu(mk.normal(1, d)).to(dtype)
    # the residual stream is a few times what one block adds to it
    x = mk.activation(case["image"] if double else tokens, d, dtype, std=4.0)[None]
    return {"block": block, "args": (x, mk.activation(case["text"], d, dtype, std=4.0)[None], rope, temb) if double else (x, rope, temb)}


def _prepare_sdxl(case, mk, dtype):
    d, level, s = case["dim"], case["level"], case["tokens"]
    sd = {}
    t16 = lambda name, *shape, std: sd.update({"b." + name: mk.normal(*shape, std=std, dtype=dtype)})
    for n in ("norm1", "norm2", "norm3"):
        sd[f"b.{n}.weight"], sd[f"b.{n}.bias"] = mk.normal(d, std=0.1, mean=1.0, dtype=dtype), mk.normal(d, std=0.05, dtype=dtype)
    # what a calibration run sees in front of each linear: LayerNorm outputs, averages over the values, the gated hidden tensor
    int8 = [("ff.net.0.proj", 8 * d, d, 5.0), ("ff.net.2", d, 4 * d, 12.0)]
    if level >= 2:
        int8.append(("attn1.to_qkv", 3 * d, d, 5.0))
    else:
        for c in "qkv":
            t16(f"attn1.to_{c}.weight", d, d, std=d ** -0.5)
    for name, amax in (("attn1.to_out.0", 10.0 * (2.7 / s) ** 0.5), ("attn2.to_q", 5.0), ("attn2.to_out.0", 10.0 * (2.7 / SDXL_TEXT) ** 0.5)):
        if level == 3:
            int8.append((name, d, d, amax))
        else:
            t16(name + ".weight", d, d, std=d ** -0.5)
    for name, n, k, amax in int8:
        sd.update(_int8_entries(mk, "b." + name, n, k, amax))
    for name, n in (("attn1.to_out.0", d), ("attn2.to_out.0", d), ("ff.net.0.proj", 8 * d), ("ff.net.2", d)):
        t16(name + ".bias", n, std=0.02)
    for c in "kv":
        t16(f"attn2.to_{c}.weight", d, SDXL_TEXT_DIM, std=SDXL_TEXT_DIM ** -0.5)
    w = sdxl_int8.load_basic_transformer_int8(sd, "b.", d, SDXL_TEXT_DIM, level, dtype, "cuda")
    x = mk.activation(case["batch"] * s, d, dtype, std=2.0, outlier=4.0).view(case["batch"], s, d)
    return {"w": w, "x": x, "text": mk.normal(case["batch"], SDXL_TEXT, SDXL_TEXT_DIM, dtype=dtype), "heads": d // SDXL_HEAD}


def prepare(case, seed):
    op, dtype, mk = case["op"], DTYPES[case["dtype"]], _Maker(seed)
    if op in ("flux_double", "flux_single"):
        return {"op": op, **_prepare_flux(case, mk, dtype)}
    if op == "sdxl_block":
        return {"op": op, **_prepare_sdxl(case, mk, dtype)}
    m, st = case["tokens"], {"op": op, "dtype": dtype}
    if op == "int8_linear":
        sd = _int8_entries(mk, "l", case["n"], case["k"], 6.0)
        sd["l.bias"] = mk.normal(case["n"], std=0.02, dtype=dtype)
        st.update(lin=weights.load_int8_linear(sd, "", "l", case["n"], case["k"], bias_dtype=dtype), dynamic=case["dynamic"],
                  x=mk.activation(m, case["k"], dtype, outlier=15.0 if case["dynamic"] else 0.0))
    elif op == "int8_geglu":
        d = case["dim"]
        for name, n, k in (("up", 8 * d, d), ("down", d, 4 * d)):
            st[name] = weights.load_int8_linear({**_int8_entries(mk, "l", n, k, 6.0), "l.bias": mk.normal(n, std=0.02, dtype=dtype)}, "", "l", n, k,
                                                bias_dtype=dtype)
        st["x"] = mk.activation(m, d, dtype, outlier=15.0)
    elif op == "fp8_linear":
        lin = weights.load_fp8_linear(_fp8_entries(mk, "l", case["n"], case["k"], dtype, 6.0), "", "l", case["n"], case["k"], dtype)
        st.update(lin=lin, dynamic=case["dynamic"], x=mk.activation(m, case["k"], dtype))
    elif op == "fp8_mlp":
        d = case["dim"]
        for name, n, k in (("up", 4 * d, d), ("down", d, 4 * d)):
            st[name] = weights.load_fp8_linear(_fp8_entries(mk, "l", n, k, dtype, 6.0), "", "l", n, k, dtype)
        st.update(x=mk.activation(m, d, dtype), largest=[torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda")])
    elif op == "w4a4_linear":
        lin = weights.load_w4a4_linear(_w4a4_entries(mk, "", case["n"], case["k"], dtype), "", case["n"], case["k"], RANK, True, dtype)
        st.update(lin=lin, x=mk.activation(m, case["k"], dtype))
    elif op == "weight_only":
        n, k, kind, group = case["n"], case["k"], case["kind"], case["group"]
        half = 128.0 if kind == "int8" else 8.0
        std = k ** -0.5 / (half / 3.0)  # codes of a normal weight whose largest value is about three deviations
        code = mk.normal(k, n, std=half / 3.0).round_().clamp_(-half, half - 1).to(torch.int8)
        if kind == "int4":
            code = (code[:, 0::2] & 15) | (code[:, 1::2] << 4)
        rows = k // group if group else 1
        scale = mk.uniform(rows, n, lo=0.5 * std, hi=1.5 * std).to(dtype)
        st.update(w=ops.repack_weight_only(code.contiguous(), kind), scale=scale if group else scale.view(n), kind=kind, group=group,
                  zeros=mk.normal(rows, n, std=std, dtype=dtype) if case["zeros"] else None, bias=mk.normal(n, std=0.02, dtype=dtype),
                  x=mk.activation(m, k, dtype))
    else:
        raise ValueError(op)
    return st


def run(st):
    op = st["op"]
    if op in ("flux_double", "flux_single"):
        return st["block"].forward(*st["args"])
    if op == "sdxl_block":
        return sdxl_int8.basic_transformer_int8_block(st["x"], st["text"], st["w"], st["heads"])
    x = st["x"]
    if op in ("int8_linear", "fp8_linear"):
        return st["lin"].forward(x, dynamic=st["dynamic"])
    if op == "w4a4_linear":
        return st["lin"].forward(x)
    if op == "int8_geglu":
        up, down, dtype = st["up"], st["down"], st["dtype"]
        q, s = ops.sq_quant_dynamic(x, up.pre_quant_scale)
        h = ops.int8_linear(q, up.weight_rows32, up.weight_scale, s, None, dtype)
        q, s = ops.geglu_int8_dynamic(h, up.bias, down.pre_quant_scale)
        return ops.int8_linear(q, down.weight_rows32, down.weight_scale, s, down.bias, dtype)
    if op == "fp8_mlp":  # the quantiser of the hidden tensor clears the slot that the next pass's up projection joins its maximum into
        up, down, dtype = st["up"], st["down"], st["dtype"]
        now, later = st["largest"]
        st["largest"] = [later, now]
        q, s = ops.fp8_quant_panels(x)
        h = ops.fp8_linear_panels(q, up.weight_rows32, s, up.weight_scale, up.bias, now, dtype)
        q, s = ops.fp8_gelu_quant_panels(h, now, later)
        return ops.fp8_linear_panels(q, down.weight_rows32, s, down.weight_scale, down.bias, None, dtype)
    if st["group"]:
        return ops.weight_only_linear_grouped(x, st["w"], st["scale"], st["zeros"], st["bias"], st["kind"], st["group"])
    return ops.weight_only_linear(x, st["w"], st["scale"], st["bias"], st["kind"])


def work(case):
    """Operands read once, results written once; two operations for each multiply-add of the linears and of the attention."""
    op = case["op"]
    linear = lambda m, n, k, weight_bytes=1.0: (weight_bytes * n * k, 2.0 * m * n * k)
    parts = []
    if op in ("flux_double", "flux_single"):
        d, s = FLUX_DIM, case["image"] + case["text"]
        wb = 0.5 + 4.0 / GROUP if case["level"].startswith("int4") else 1.0
        ada = 1.0 if case["level"].endswith("full") else 2.0
        if op == "flux_double":
            for m in (case["image"], case["text"]):
                parts += [linear(1, 6 * d, d, ada), linear(m, 3 * d, d, wb), linear(m, d, d, wb), linear(m, 4 * d, d, wb), linear(m, d, 4 * d)]
        else:
            parts = [linear(1, 3 * d, d, ada), linear(s, 3 * d, d, wb), linear(s, 4 * d, d, wb), linear(s, d, 5 * d, wb)]
        parts += [(2 * 2.0 * s * d + 2.0 * s * FLUX_HEAD * 2, 4.0 * s * s * d)]
    elif op == "sdxl_block":
        d, b, s = case["dim"], case["batch"], case["tokens"]
        m, own = b * s, {1: 2.0, 2: 2.0, 3: 1.0}[case["level"]]
        parts = [linear(m, 3 * d, d, 2.0 if case["level"] == 1 else 1.0)] + 3 * [linear(m, d, d, own)]
        parts += 2 * [linear(b * SDXL_TEXT, d, SDXL_TEXT_DIM, 2.0)] + [linear(m, 8 * d, d), linear(m, d, 4 * d)]
        parts += [(2 * 2.0 * m * d + 2.0 * b * SDXL_TEXT * SDXL_TEXT_DIM, 4.0 * b * s * (s + SDXL_TEXT) * d)]
    elif op in ("int8_geglu", "fp8_mlp"):
        m, d = case["tokens"], case["dim"]
        parts = [linear(m, (8 if op == "int8_geglu" else 4) * d, d), linear(m, d, 4 * d), (2 * 2.0 * m * d, 0.0)]
    else:
        m, n, k = case["tokens"], case["n"], case["k"]
        wb = {"int8_linear": 1.0, "fp8_linear": 1.0, "w4a4_linear": 0.5 + 4.0 / GROUP}.get(op)
        if op == "weight_only":
            wb = (1.0 if case["kind"] == "int8" else 0.5) + ((4.0 if case["zeros"] else 2.0) / case["group"] if case["group"] else 0.0)
        parts = [linear(m, n, k, wb), (2.0 * m * k + 2.0 * m * n, 0.0)]
        if op == "w4a4_linear":
            parts += [linear(m, RANK, k, 2.0), linear(m, n, RANK, 2.0)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    """Blocks: about four times what they differ from themselves by with the attention in one pass of 32-bit floats instead of
    blocks of keys; they quantise what it returns, so a last bit there moves some codes by a whole step (4-bit ones most).
    Linears: a last bit of the result where 32-bit sums are taken in another order, more where e4m3 products are summed (the
    matrix instruction keeps 13 bits of a group's products) or a result is quantised again."""
    op, half = case["op"], case["dtype"] == "fp16"
    if op == "flux_double":
        return {"rel": 0.03, "max": 0.99 if case["level"].startswith("int4") else 0.6}
    if op == "flux_single":
        return {"rel": 0.01, "max": 0.15}
    if op == "sdxl_block":
        return {"rel": 0.03, "max": 0.3}
    if op in ("int8_linear", "w4a4_linear", "weight_only"):
        return {"rel": 1e-3 if half else 5e-3}
    return {"rel": 1e-2 if op == "fp8_mlp" else 5e-3}
