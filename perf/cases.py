"""Performance cases of the state codec and FP4 weight framework, at the geometry
of the 8B model it serves (128 heads of 64 channels, 8 B/C groups, 128 state
coordinates, 4096 hidden channels).

Each case is one piece of work that a decoding, prefilling, calibrating or
loading program gives to the package's public entry points:

* "step":    one token for several layers' packed states (decode), as one eager
             scan call or as a replayed HIP graph of one call per layer;
* "prefill": one multi-token scan call of one layer, of any of the codecs;
* "fp4":     fp4.decode_packet of one checkpoint matrix;
* "gemv":    fp4.gemv_g16 over several layers' projection matrices;
* "mixer":   whole mixer calls through an installed StateQuant controller.

`exact` restates each path in float64 torch, with the codecs' quantization
rules; values that are codes or stored scales have no 64-bit counterpart.
"""
import math
import sys
from pathlib import Path

import torch
from torch import nn

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "mamb2_8b_fp4_recall_sq3.25_amd"))
from mamba2_recall import fp4, ridge_codec, state_codec, state_codec_dense3, tier_codec  # noqa: E402
from mamba2_recall.state_quant import StateQuant  # noqa: E402

H, P, G, N, D_MODEL, D_INNER, CONV = 128, 64, 8, 128, 4096, 8192, 10240
IN_ROWS = 2 * D_INNER + 2 * G * N + H
LAYOUTS = ("36_24_68", "16_64_48", "32_32_64", "40_16_72", "24_48_56", "8_80_40", "44_8_76")
CODECS = ("ridge", "tier", "sq3p25", "dense3", "s16")
WARM_TOKENS = 4


def listed():
    return [
        # the smallest call: one layer's decode step called eagerly, where latency counts
        dict(name="step_layer_b1", kind="step", codec="ridge", batch=1, layers=1, graph=False, d32=False),
        # batched serving: a decode step over a layer of each published layout, replayed as a graph
        dict(name="step_graph_b64", kind="step", codec="ridge", batch=64, layers=7, graph=True, d32=False),
        # batch-1 prompt of one layer with the published codec (perplexity windows, prompts)
        dict(name="prefill_ridge_b1", kind="prefill", codec="ridge", layout="24_48_56", batch=1, tokens=512,
             table="permutation", stats=False, d32=False),
        # a batch of ragged-length prompts padded to one odd length
        dict(name="prefill_ridge_b12", kind="prefill", codec="ridge", layout="36_24_68", batch=12, tokens=201,
             table="permutation", stats=False, d32=True),
        # the stored-scale tier controller's prefill (state repair evaluation)
        dict(name="prefill_tier_b3", kind="prefill", codec="tier", layout="32_32_64", batch=3, tokens=300,
             table="permutation", stats=False, d32=False),
        # the dense 3-bit carry with its equalizer table
        dict(name="prefill_dense3_b1", kind="prefill", codec="dense3", layout="", batch=1, tokens=512,
             table="equalizer", stats=False, d32=False),
        # calibration: the FP16-carry control over a text window with its |carry| statistics
        dict(name="calibrate_s16_b1", kind="prefill", codec="s16", layout="", batch=1, tokens=512,
             table="", stats=True, d32=False),
        # checkpoint load: one in_proj matrix to resident FP16
        dict(name="fp4_in_proj", kind="fp4", format="fp4_g16_e4m3", rows=IN_ROWS, cols=D_MODEL),
        # a matrix whose columns are no multiple of the group (padded last group)
        dict(name="fp4_ragged", kind="fp4", format="fp4_g16_e4m3", rows=5003, cols=4100),
        # four sequences' projections with packed-resident weights, four layers
        dict(name="gemv_b4", kind="gemv", batch=4, layers=4),
        # one decode token through three mixers with packed projections, replayed as a graph
        dict(name="mixer_decode_b1", kind="mixer", codec="sq3p25", batch=1, tokens=1, layers=3),
        # a prompt through one whole mixer (projections, convolution, control carry, gated norm)
        dict(name="mixer_prefill_b1", kind="mixer", codec="s16", batch=1, tokens=1024, layers=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "prefill", "prefill", "prefill", "fp4", "gemv", "mixer"))
    if kind == "step":
        return dict(kind=kind, codec="ridge", batch=_log(rng, 1, 64), layers=rng.choice((3, 5, 7)), graph=True,
                    d32=rng.random() < 0.3)
    if kind == "prefill":
        codec = rng.choice(CODECS)
        batch = _log(rng, 1, 16)
        return dict(kind=kind, codec=codec, layout=rng.choice(LAYOUTS) if codec in ("ridge", "tier") else "",
                    batch=batch, tokens=_log(rng, 2, min(512, 2048 // batch)),
                    table=rng.choice(("permutation", "equalizer")) if codec == "dense3" else "",
                    stats=codec == "s16" and rng.random() < 0.5, d32=rng.random() < 0.3)
    if kind == "fp4":
        return dict(kind=kind, format=rng.choice(fp4.FORMATS), rows=_log(rng, 64, 18560),
                    cols=rng.choice((4096, 8192, _log(rng, 100, 8200))))
    if kind == "gemv":
        return dict(kind=kind, batch=rng.choice((1, 2, 4)), layers=rng.choice((2, 3, 4)))
    return dict(kind=kind, codec=rng.choice(("s16", "sq3p25")), batch=1, tokens=_log(rng, 8, 900), layers=1)


# ---------------------------------------------------------------- inputs
def _counts(codec, layout):
    """(INT8, INT4, zero-carry) coordinates of a packed row."""
    if codec == "sq3p25":
        return 16, 64, 48
    a, b, c = map(int, layout.split("_"))
    return (a, b - 4, c + 4) if codec == "ridge" else (a, b, c)


def _inputs(gen, dev, batch, tokens, d32):
    def normal(*shape):
        return torch.randn(shape, generator=gen, device=dev)
    pdt = torch.float32 if d32 else torch.float16
    return dict(x=normal(batch, tokens, H, P).half(), dt=normal(batch, tokens, H).half(),
                A=-torch.exp(torch.rand(H, generator=gen, device=dev) * math.log(16.0)),
                B=normal(batch, tokens, G, N).half(), C=normal(batch, tokens, G, N).half(), D=normal(H).to(pdt),
                dt_bias=(normal(H) * 0.5).to(pdt))


def _perms(gen, dev, rows):
    return torch.argsort(torch.rand(rows, N, generator=gen, device=dev), dim=-1).to(torch.uint8)


def _layer(codec, layout, batch, tokens, table, d32, gen, dev):
    """One layer's inputs, static tables and a carry in mid-sequence."""
    d = dict(codec=codec, layout=layout, **_inputs(gen, dev, batch, tokens, d32))

    def codes(t):
        t.copy_(torch.randint(0, 256, t.shape, generator=gen, device=dev, dtype=torch.uint8))

    def scales(t, mu):
        t.copy_(torch.exp(torch.randn(t.shape, generator=gen, device=dev) * 0.5 + mu))

    if codec == "s16":
        d["state"] = state_codec.allocate_state(batch, H, P, N, "s16", dev)
        t = d["state"].tensors["state"]
        t.copy_(torch.randn(t.shape, generator=gen, device=dev))
        return d
    if codec == "dense3":
        d["kind"] = table
        d["perm"] = (_perms(gen, dev, G) if table == "permutation" else
                     torch.randint(-4, 5, (G, N), generator=gen, device=dev).to(torch.int8))
        d["state"] = state_codec_dense3.allocate_state(batch, H, P, N, dev)
        bits = d["state"].tensors["codes"]
        codes(bits)
        # the codes are -3..3: clear the sign plane of a would-be -4
        bits[:, :, :, 2] &= bits[:, :, :, 0] | bits[:, :, :, 1]
        scales(d["state"].tensors["scales"], -1.0)
        return d
    d["perm"] = _perms(gen, dev, G)
    n8, n4, nz = _counts(codec, layout)
    if codec == "ridge":
        d["state"] = ridge_codec.allocate_state(batch, H, P, N, dev, layout=layout)
        d["basis"] = (torch.randn(G, nz, 2, generator=gen, device=dev) * 0.03).half()
        d["lscale"] = torch.full((G, 2), 0.001, device=dev, dtype=torch.float16)
        d["pred"] = (torch.randn(G, n8 + n4 + 2, nz, generator=gen, device=dev) * 0.05).half()
        lat = d["state"].tensors["latent"]
        lat.copy_((torch.randn(lat.shape, generator=gen, device=dev) * 40).clamp(-440, 440))
    elif codec == "tier":
        d["state"] = tier_codec.allocate_state(batch, H, P, N, dev, layout=layout)
    else:
        d["state"] = state_codec.allocate_state(batch, H, P, N, "sq3p25", dev)
    t = d["state"].tensors
    for k in ("lo", "hi", "q4"):
        codes(t[k])
    scales(t["s8"], -4.0)
    scales(t["s4"], -1.5)
    return d


def _scan(d, stats=False):
    a = (d["x"], d["dt"], d["A"], d["B"], d["C"], d["D"], d["dt_bias"], d["state"])
    if d["codec"] == "ridge":
        return ridge_codec.scan(*a, d["perm"], d["basis"], d["lscale"], d["pred"], layout=d["layout"], validate=False)
    if d["codec"] == "tier":
        return tier_codec.scan(*a, d["perm"], layout=d["layout"])
    if d["codec"] == "dense3":
        return state_codec_dense3.scan(*a, d["perm"], d["kind"]), None
    if d["codec"] == "sq3p25":
        return state_codec.scan(*a, permutation=d["perm"])
    return state_codec.scan(*a, collect_stats=stats)


def _carry(state):
    """The state's own buffers (E4M3 latents as their bytes)."""
    return {k: v.view(torch.uint8) if v.dtype == torch.float8_e4m3fn else v for k, v in state.tensors.items()}


def _packet(gen, dev, rows, cols, fmt="fp4_g16_e4m3"):
    """A canonical packet of weights of about unit fan-in scale."""
    group = 16 if fmt == "fp4_g16_e4m3" else 64
    groups = -(-cols // group)
    packed = torch.randint(0, 256, (rows, groups * group // 2), generator=gen, device=dev, dtype=torch.uint8)
    pad = groups * group - cols
    if pad:   # the padding of the last group holds zero codes
        packed[:, packed.shape[1] - pad // 2:] = 0
        if cols % 2:
            packed[:, cols // 2] &= 15
    if group == 16:
        scales = (torch.rand(rows, groups, generator=gen, device=dev) * 300 + 8).to(torch.float8_e4m3fn)
        glob = torch.full((), 1.0 / (200 * 3 * math.sqrt(cols)), dtype=torch.float32, device=dev)
    else:
        scales = (torch.rand(rows, groups, generator=gen, device=dev) / (2 * math.sqrt(cols)) + 1e-4).half()
        glob = None
    return dict(format=fmt, shape=[rows, cols], group_size=group, packed=packed, scales=scales, global_scale=glob)


def _captured(work, restore):
    """`work` as a HIP graph: one warm-up call on a side stream, its effects
    undone, then the capture.  Returns (graph, the captured outputs)."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        work()
    torch.cuda.current_stream().wait_stream(side)
    restore()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = work()
    return graph, out


# ---------------------------------------------------------------- a model of few mixers
class _GatedNorm(nn.Module):
    """norm(y * silu(z)) per group, as the model's own module defines it."""

    def __init__(self):
        super().__init__()
        self.eps, self.group_size = 1e-5, D_INNER // G
        self.weight = nn.Parameter(torch.ones(D_INNER))

    def forward(self, y, z):
        v = (y.float() * torch.nn.functional.silu(z.float())).unflatten(-1, (G, -1))
        v = v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + self.eps)
        return (v.flatten(-2) * self.weight.float()).to(y.dtype)


class _Mixer(nn.Module):
    def __init__(self):
        super().__init__()
        self.d_model, self.d_inner, self.d_ssm, self.nheads = D_MODEL, D_INNER, D_INNER, H
        self.headdim, self.d_state, self.ngroups, self.d_conv = P, N, G, 4
        self.use_mem_eff_path, self.rmsnorm, self.D_has_hdim = False, True, False
        self.activation, self.dt_limit, self.process_group = "silu", (0.0, float("inf")), None
        self.in_proj = nn.Linear(D_MODEL, IN_ROWS, bias=False)
        self.conv1d = nn.Conv1d(CONV, CONV, 4, groups=CONV, padding=3, bias=True)
        self.act = nn.SiLU()
        self.A_log, self.D, self.dt_bias = (nn.Parameter(torch.empty(H)) for _ in range(3))
        self.norm = _GatedNorm()
        self.out_proj = nn.Linear(D_INNER, D_MODEL, bias=False)


class _Block(nn.Module):
    def __init__(self):
        super().__init__()
        self.mixer = _Mixer()
        self.fused_add_norm, self.residual_in_fp32, self.mlp = False, False, None


class _Model(nn.Module):
    def __init__(self, layers):
        super().__init__()
        self.backbone = nn.Module()
        self.backbone.layers = nn.ModuleList(_Block() for _ in range(layers))
        self.backbone.fused_add_norm, self.backbone.residual_in_fp32 = False, False


def _mixers(layers, gen, dev):
    """A model of `layers` mixers with seeded FP16 weights, and the packets
    its projections were decoded from."""
    with torch.device("meta"):
        model = _Model(layers)
    model = model.to_empty(device=dev).half().requires_grad_(False).eval()
    packets = []
    for block in model.backbone.layers:
        mx = block.mixer
        mx.A_log.copy_(torch.rand(H, generator=gen, device=dev) * math.log(16.0))
        mx.D.copy_(torch.randn(H, generator=gen, device=dev))
        mx.dt_bias.copy_(torch.log(torch.expm1(torch.rand(H, generator=gen, device=dev) * 0.09 + 0.01)))
        mx.norm.weight.copy_(1 + 0.1 * torch.randn(D_INNER, generator=gen, device=dev))
        mx.conv1d.weight.copy_(torch.randn(CONV, 1, 4, generator=gen, device=dev) * 0.5)
        mx.conv1d.bias.copy_(torch.randn(CONV, generator=gen, device=dev) * 0.1)
        entry = {}
        for name, (rows, cols) in (("in_proj", (IN_ROWS, D_MODEL)), ("out_proj", (D_MODEL, D_INNER))):
            pk = _packet(gen, dev, rows, cols)
            getattr(mx, name).weight.copy_(fp4.decode_packet(pk))
            entry[name] = (pk["packed"], pk["scales"], pk["global_scale"])
        packets.append(entry)
    return model, packets


def _controller(model, layers, codec, perms):
    """A StateQuant over a model of `layers` layers instead of all 56."""
    params = list(model.parameters())
    cls = type("FewLayerStateQuant", (StateQuant,), dict(
        LAYERS=layers, TABLE_SHAPE=(layers, G, N), PARAMETER_TENSORS=len(params),
        PARAMETER_COUNT=sum(p.numel() for p in params)))
    return cls(model, mode=codec, permutations=perms).install()


def _through(mixers, h):
    for mx in mixers:
        h = mx(h)
    return h


# ---------------------------------------------------------------- the cases
@torch.no_grad()
def prepare(case, seed):
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(seed)
    kind = case["kind"]
    s = dict(case=case)
    if kind == "step":
        s["layers"] = [_layer("ridge", LAYOUTS[(i + 4) % 7], case["batch"], 1, "", case["d32"], gen, dev)
                       for i in range(case["layers"])]
        if case["graph"]:
            kept = [d["state"].clone() for d in s["layers"]]

            def restore():
                for d, k in zip(s["layers"], kept):
                    for name, t in d["state"].tensors.items():
                        t.copy_(k.tensors[name])
            s["graph"], s["y"] = _captured(lambda: [_scan(d)[0] for d in s["layers"]], restore)
    elif kind == "prefill":
        s["layer"] = _layer(case["codec"], case["layout"], case["batch"], case["tokens"], case["table"], case["d32"],
                            gen, dev)
    elif kind == "fp4":
        s["packet"] = _packet(gen, dev, case["rows"], case["cols"], case["format"])
    elif kind == "gemv":
        s["weights"] = [(_packet(gen, dev, IN_ROWS, D_MODEL), _packet(gen, dev, D_MODEL, D_INNER))
                        for _ in range(case["layers"])]
        s["u"] = [torch.randn(case["batch"], n, generator=gen, device=dev).half() for n in (D_MODEL, D_INNER)]
    else:
        layers, batch = case["layers"], case["batch"]
        s["model"], packets = _mixers(layers, gen, dev)
        s["mixers"] = [b.mixer for b in s["model"].backbone.layers]
        perms = _perms(gen, dev, layers * G).reshape(layers, G, N) if case["codec"] == "sq3p25" else None
        s["perms"] = perms
        s["control"] = c = _controller(s["model"], layers, case["codec"], perms)
        decode = case["tokens"] == 1
        s["u"] = torch.randn(batch, WARM_TOKENS + 1 if decode else case["tokens"], D_MODEL, generator=gen,
                             device=dev).half()
        if decode:   # a request in flight: its first tokens seen, then one-token steps as a graph
            c.use_packed_projections(packets)
            c.reset(batch)
            _through(s["mixers"], s["u"][:, :WARM_TOKENS])
            s["token"] = s["u"][:, WARM_TOKENS:].contiguous()
            kept = [(e.conv.clone(), e.state.clone()) for e in c._cache]

            def restore():
                for e, (conv, state) in zip(c._cache, kept):
                    e.conv.copy_(conv)
                    for name, t in e.state.tensors.items():
                        t.copy_(state.tensors[name])
            s["graph"], s["out"] = _captured(lambda: _through(s["mixers"], s["token"]), restore)
    return s


@torch.no_grad()
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "step":
        if case["graph"]:
            s["graph"].replay()
            y = s["y"]
        else:
            y = [_scan(d)[0] for d in s["layers"]]
        return dict(y=y, state=[_carry(d["state"]) for d in s["layers"]])
    if kind == "prefill":
        y, stats = _scan(s["layer"], case["stats"])
        return dict(y=y, stats=stats, state=_carry(s["layer"]["state"]))
    if kind == "fp4":
        return fp4.decode_packet(s["packet"])
    if kind == "gemv":
        return [fp4.gemv_g16(p["packed"], p["scales"], p["global_scale"], u)
                for pair in s["weights"] for p, u in zip(pair, s["u"])]
    c = s["control"]
    if "graph" in s:
        s["graph"].replay()
        out = s["out"]
    else:
        c.reset(case["batch"])
        out = _through(s["mixers"], s["u"])
    return dict(out=out, conv=[e.conv for e in c._cache], state=[_carry(e.state) for e in c._cache])


# ---------------------------------------------------------------- work and tolerance
def _state_row_bytes(codec):
    return 256 if codec == "s16" else 52


def work(case):
    kind = case["kind"]
    if kind in ("step", "prefill"):
        b, layers, L = case["batch"], case.get("layers", 1), case.get("tokens", 1)
        rows = b * H * P
        per = 2 * rows * _state_row_bytes(case["codec"]) + L * b * (4 * H * P + 4 * G * N + 2 * H)
        if case["codec"] == "ridge":
            per += sum(2 * G * nz * (n8 + n4 + 4) for n8, n4, nz in (_counts("ridge", "32_32_64"),))
        if case.get("stats"):
            per += b * H * 4 * N * 4
        # per carried coordinate and token: readout (2), input product (1) and update (2)
        return dict(bytes=layers * per, flops=5 * layers * L * rows * (128 if case["codec"] in ("dense3", "s16") else 70))
    if kind == "fp4":
        group = 16 if case["format"] == "fp4_g16_e4m3" else 64
        groups = -(-case["cols"] // group)
        scale = 1 if group == 16 else 2
        return dict(bytes=case["rows"] * (groups * (group // 2 + scale) + 2 * case["cols"]), flops=0)
    weights = IN_ROWS * D_MODEL + D_MODEL * D_INNER
    if kind == "gemv":
        return dict(bytes=case["layers"] * weights * 9 // 16, flops=2 * case["batch"] * case["layers"] * weights)
    tokens, layers = case["batch"] * case["tokens"], case["layers"]
    per_weight = 9 / 16 if case["tokens"] == 1 else 2
    carry = 2 * case["batch"] * H * P * _state_row_bytes(case["codec"])
    return dict(bytes=layers * int(weights * per_weight + carry + 4 * tokens * D_MODEL),
                flops=layers * tokens * (2 * weights + 5 * H * P * 128 + 8 * CONV))


def tolerance(case):
    kind = case["kind"]
    if kind == "fp4":
        return "exact"
    if kind in ("step", "prefill"):
        # codes and scales are exact; a readout rounded to FP16 is 2.1e-4 from float64
        return dict(rel=8e-4)
    if kind == "gemv":
        return dict(rel=8e-4)
    # FP16 activations between the projections, the convolution, the codec and the norm; a
    # packed carry's codes move with them where a value lies at a rounding boundary
    return dict(rel=4e-3, differ=0.0 if case["codec"] == "s16" else 0.01)


# ---------------------------------------------------------------- float64 restatements
def _half(v):
    return v.half().double()


def _away(v):
    """Round half away from zero."""
    return torch.sign(v) * torch.floor(v.abs() + 0.5)


def _nibbles(t):
    return torch.stack((t & 15, t >> 4), dim=-1).flatten(-2).long()


def _dequantized(d):
    """The carry in packed order, float64 [B, H, P, carried], and the latents."""
    codec, t = d["codec"], d["state"].tensors
    if codec == "s16":
        return t["state"].double(), None
    if codec == "dense3":
        bits = (t["codes"].unsqueeze(-1) >> torch.arange(8, device=t["codes"].device, dtype=torch.uint8)) & 1
        u = (bits.flatten(-2).long() * torch.tensor([1, 2, 4], device=bits.device)[:, None]).sum(-2)
        q = torch.where(u >= 4, u - 8, u).double()
        return q * t["scales"].double().repeat_interleave(64, dim=-1), None
    u8 = _nibbles(t["lo"]) | (_nibbles(t["hi"]) << 4)
    u4 = _nibbles(t["q4"])
    v8 = torch.where(u8 > 127, u8 - 256, u8).double() * t["s8"].double()[..., None]
    v4 = torch.where(u4 > 7, u4 - 16, u4).double() * t["s4"].double()[..., None]
    z = t["latent"].float().double() if codec == "ridge" else None
    return torch.cat((v8, v4), -1), z


def _requantized(codec, n8, u):
    if codec == "s16":
        return _half(u)
    if codec == "dense3":
        parts = ((u[..., :64], 3.0), (u[..., 64:], 3.0))
    else:
        parts = ((u[..., :n8], 127.0), (u[..., n8:], 7.0))
    out = []
    for v, lim in parts:
        den = (v.abs().amax(-1, keepdim=True) / lim).clamp_min(1e-8)
        s = _half(den)
        by = den if codec in ("dense3", "sq3p25") else s
        q = torch.where(by > 0, _away(v / torch.where(by > 0, by, 1.0)).clamp(-lim, lim), 0.0)
        out.append(q * s)
    return torch.cat(out, -1)


def _scan64(d, stats=False):
    """(readouts, statistics or None) of one layer's tokens from its carry."""
    codec, x = d["codec"], d["x"].double()
    batch, tokens = x.shape[:2]
    v = d["dt"].double() + d["dt_bias"].double()
    dt = torch.where(v <= 20, torch.log1p(torch.exp(v.clamp(max=20.0))), v)
    decay = torch.exp(d["A"].double() * dt)
    bm, cm = d["B"].double(), d["C"].double()
    carry, z = _dequantized(d)
    n8 = n = carry.shape[-1]
    if codec == "dense3" and d["kind"] == "equalizer":
        e = d["perm"].double()
        bm, cm = bm * torch.exp2(-e), cm * torch.exp2(e)
    elif codec != "s16":
        index = d["perm"].long()[None, None].expand(batch, tokens, G, N)
        bm, cm = bm.gather(3, index), cm.gather(3, index)
    if codec in ("ridge", "tier", "sq3p25"):
        n8 = _counts(codec, d["layout"])[0]
    dead = (bm[..., n:] * cm[..., n:]).sum(-1)
    if codec == "ridge":
        corr = torch.einsum("btgd,gfd->btgf", cm[..., n:], d["pred"].double())
        e = d["basis"].double()
        dots_c = torch.einsum("btgd,gdk->btgk", cm[..., n:], e)
        dots_b = torch.einsum("btgd,gdk->btgk", bm[..., n:], e)
        ls = d["lscale"].double().repeat_interleave(H // G, 0)[None, :, None, :]
        z = z * ls
    total = torch.zeros_like(carry) if stats else None

    def heads(w):   # a [B, G, ...] value for each head
        return w.repeat_interleave(H // G, 1)

    y = torch.empty_like(x)
    for t in range(tokens):
        xt, dtt, dec = x[:, t, ..., None], dt[:, t, :, None, None], decay[:, t, :, None, None]
        u = carry * dec + heads(bm[:, t, :, :n])[:, :, None, :] * dtt * xt
        out = (u * heads(cm[:, t, :, :n])[:, :, None, :]).sum(-1)
        out = out + xt[..., 0] * (dtt[..., 0] * heads(dead[:, t])[..., None] + d["D"].double()[None, :, None])
        if codec == "ridge":
            c = heads(corr[:, t])[:, :, None, :]
            latent = (z * (heads(dots_c[:, t])[:, :, None, :] + c[..., n:])).sum(-1)
            out = out + dec[..., 0] * ((carry * c[..., :n]).sum(-1) + latent)
            z = z * dec + xt * dtt * heads(dots_b[:, t])[:, :, None, :]
            z = (z / ls).clamp(-448, 448).float().to(torch.float8_e4m3fn).float().double() * ls
        y[:, t] = out
        carry = _requantized(codec, n8, u)
        if stats:
            total += carry.abs()
    return y, total.unflatten(2, (P // 16, 16)).sum(3) if stats else None


def _blank(state):
    return {k: None for k in state.tensors}


def _weights64(p):
    levels = torch.tensor(fp4.E2M1_MAGNITUDES, device=p["packed"].device)
    q = _nibbles(p["packed"])[:, :p["shape"][1]]
    w = levels[q & 7] * (1 - 2 * (q >> 3)).float()
    w = w * p["scales"].float().repeat_interleave(p["group_size"], -1)[:, :w.shape[1]]
    return w.half() if p["global_scale"] is None else (w * p["global_scale"]).half()


def _mixer64(s):
    """The mixers' outputs with every value between the modules in float64."""
    case, h = s["case"], s["u"].double()
    for i, mx in enumerate(s["mixers"]):
        z, xbc, dt = torch.split(h @ mx.in_proj.weight.double().T, (D_INNER, CONV, H), dim=-1)
        w = mx.conv1d.weight.double()[:, 0]
        padded = torch.cat((torch.zeros_like(xbc[:, :1]).expand(-1, 3, -1), xbc), 1)
        L = xbc.shape[1]
        conv = sum(padded[:, k:k + L] * w[:, k] for k in range(4)) + mx.conv1d.bias.double()
        x, bm, cm = torch.split(conv * torch.sigmoid(conv), (D_INNER, G * N, G * N), dim=-1)
        shape = h.shape[:2]
        state = state_codec.allocate_state(shape[0], H, P, N, case["codec"], h.device)
        d = dict(codec=case["codec"], layout="", x=x.reshape(*shape, H, P), dt=dt, A=-torch.exp(mx.A_log.double()),
                 B=bm.reshape(*shape, G, N), C=cm.reshape(*shape, G, N), D=mx.D, dt_bias=mx.dt_bias, state=state,
                 perm=None if s["perms"] is None else s["perms"][i])
        y = _scan64(d)[0].flatten(-2)
        v = (y * z * torch.sigmoid(z)).unflatten(-1, (G, -1))
        v = (v / torch.sqrt(v.pow(2).mean(-1, keepdim=True) + mx.norm.eps)).flatten(-2) * mx.norm.weight.double()
        h = v @ mx.out_proj.weight.double().T
    return h


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    # the inputs alone: nothing of the package has stepped the carries yet
    s = prepare(dict(case, graph=False) if kind == "step" else case, seed)
    if kind == "step":
        return dict(y=[_scan64(d)[0] for d in s["layers"]], state=[_blank(d["state"]) for d in s["layers"]])
    if kind == "prefill":
        y, stats = _scan64(s["layer"], case["stats"])
        return dict(y=y, stats=stats, state=_blank(s["layer"]["state"]))
    if kind == "fp4":
        return _weights64(s["packet"])
    if kind == "gemv":
        return [u.double() @ _weights64(p).double().T for pair in s["weights"] for p, u in zip(pair, s["u"])]
    out = _mixer64(s)
    if case["tokens"] == 1:
        out = out[:, WARM_TOKENS:]
    entries = s["control"]._cache or [None] * case["layers"]
    return dict(out=out, conv=[None for _ in entries], state=[{} for _ in entries])
