"""The work that a user of this framework has it do, as measurable cases.

Every case goes through luisaml_amd.capi, the binding of the C ABI, with
synthetic seeded data of the sizes that the benchmark, the tests and ordinary
networks of these kinds have.  A case is a dict of plain values; its "kind"
names the program:

  block    the four linears of a transformer block (QKV, output projection,
           up + GELU, down), activations quantised dynamically, E4M3 weights
  gemm     one GEMM on activations that are already E4M3
  mlp      a three-layer perceptron on fp32 activations
  w8a32    one weight-only linear: fp32 activations, E4M3 weights
  conv     NCHW fp32 -> dynamic E4M3 in NHWC -> FP8 convolution -> NCHW
  load     a weight's way into the engine: per-channel QuantizeLinear, packing
  codec    QuantizeLinear / DequantizeLinear of an activation tensor
  fp32     the layers that the FP8 path does not take: an fp32 convolution
           (input channels not a multiple of 16) and an fp32 Gemm
"""
import math

import torch
import torch.nn.functional as F

from luisaml_amd import capi

DEV = "cuda:0"
KERNELS = {"auto": capi.KERNEL_AUTO, "auto_fp8": capi.KERNEL_AUTO_FP8}
ACTS = {"none": capi.ACT_NONE, "relu": capi.ACT_RELU, "gelu": capi.ACT_GELU_ERF}
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # one decode step of one sequence, and of a batch of 16: the smallest
        # GEMMs, bound by reading the weights and by launches, so a serving
        # loop captures the step in a HIP graph
        {"name": "decode_m1", "kind": "block", "m": 1, "hidden": 4096, "ffn": 11008, "kernel": "auto", "graph": True},
        {"name": "decode_m16", "kind": "block", "m": 16, "hidden": 4096, "ffn": 11008, "kernel": "auto", "graph": True},
        # a batch of 100 sequences, or a short prompt: between the decode
        # sizes and the ones that fill the matrix cores, and a ragged M
        {"name": "batch_m100", "kind": "block", "m": 100, "hidden": 4096, "ffn": 11008, "kernel": "auto", "graph": False},
        # prefill: batch 8 x 512 tokens, the benchmark's transformer linears
        {"name": "prefill_m4096", "kind": "block", "m": 4096, "hidden": 4096, "ffn": 11008, "kernel": "auto",
         "graph": False},
        # the benchmark's large GEMM on the native FP8 matrix cores (the
        # opt-in for callers that accept their precision)
        {"name": "gemm_8192_fp8", "kind": "gemm", "m": 8192, "n": 8192, "k": 8192, "kernel": "auto_fp8", "act": "none",
         "bias": False, "out": "bf16"},
        # the perceptron 784-256-128-10 at batch 64, DequantizeLinear weights
        {"name": "mlp_b64", "kind": "mlp", "m": 64, "d0": 784, "d1": 256, "d2": 128, "d3": 10, "weights": "e4m3",
         "graph": True},
        # a weight-only up-projection with GELU over a batch of 128 rows
        {"name": "w8a32_m128", "kind": "w8a32", "m": 128, "n": 11008, "k": 4096, "act": "gelu", "out": "fp32"},
        # the ResNet 3x3 convolution of the benchmark, batch 32
        {"name": "conv3x3_56", "kind": "conv", "n": 32, "c": 256, "h": 56, "w": 56, "cout": 256, "ks": 3, "stride": 1,
         "pad": 1, "group": 1, "kernel": "auto", "act": "relu", "out": "fp32"},
        # a down-sampling convolution at a small batch: odd planes, grouped,
        # native FP8 and bf16 out
        {"name": "conv3x3_s2_ragged", "kind": "conv", "n": 5, "c": 192, "h": 57, "w": 57, "cout": 320, "ks": 3,
         "stride": 2, "pad": 1, "group": 2, "kernel": "auto_fp8", "act": "relu", "out": "bf16"},
        # one weight of the model at load time: [K, N] with a scale per
        # output channel
        {"name": "load_4096x11008", "kind": "load", "n": 11008, "k": 4096, "nk": False},
        # QDQ of an activation tensor between nodes that are not fused
        {"name": "codec_2050x11008", "kind": "codec", "rows": 2050, "cols": 11008, "how": "dynamic"},
        # the stem and the classifier of a ResNet, batch 16
        {"name": "fp32_stem_head", "kind": "fp32", "n": 16, "c": 3, "h": 224, "w": 224, "cout": 64, "ks": 7, "stride": 2,
         "pad": 3, "group": 1, "gm": 16, "gn": 1000, "gk": 2048, "tb": True},
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["block", "block", "gemm", "mlp", "w8a32", "conv", "load", "codec", "fp32"])
    if kind == "block":
        m = _log(rng, 1, 4096)
        return {"kind": kind, "m": m, "hidden": 16 * _log(rng, 64, 256), "ffn": 16 * _log(rng, 160, 688),
                "kernel": rng.choice(["auto", "auto", "auto_fp8"]), "graph": m <= 32}
    if kind == "gemm":
        return {"kind": kind, "m": _log(rng, 1, 8192), "n": _log(rng, 64, 8192), "k": 16 * _log(rng, 8, 512),
                "kernel": rng.choice(["auto", "auto_fp8"]), "act": rng.choice(["none", "none", "gelu"]),
                "bias": rng.random() < 0.5, "out": rng.choice(["bf16", "fp32"])}
    if kind == "mlp":
        return {"kind": kind, "m": _log(rng, 1, 512), "d0": _log(rng, 100, 1024), "d1": _log(rng, 64, 512),
                "d2": _log(rng, 64, 512), "d3": _log(rng, 10, 100), "weights": rng.choice(["e4m3", "e4m3", "fp32"]),
                "graph": True}
    if kind == "w8a32":
        return {"kind": kind, "m": _log(rng, 1, 512), "n": _log(rng, 64, 11008), "k": _log(rng, 100, 4096),
                "act": rng.choice(["none", "relu", "gelu"]), "out": rng.choice(["bf16", "fp32"])}
    if kind == "conv":
        group = rng.choice([1, 1, 1, 2])
        ks = rng.choice([1, 3, 3, 5])
        return {"kind": kind, "n": _log(rng, 1, 32), "c": 16 * group * _log(rng, 2, 16 // group), "h": rng.randint(7, 57),
                "w": rng.randint(7, 57), "cout": 8 * group * _log(rng, 4, 32 // group), "ks": ks,
                "stride": rng.choice([1, 1, 2]), "pad": ks // 2, "group": group,
                "kernel": rng.choice(["auto", "auto_fp8"]), "act": rng.choice(["none", "relu"]),
                "out": rng.choice(["bf16", "fp32"])}
    if kind == "load":
        return {"kind": kind, "n": _log(rng, 64, 11008), "k": _log(rng, 128, 4096), "nk": rng.random() < 0.5}
    if kind == "codec":
        return {"kind": kind, "rows": _log(rng, 1, 4096), "cols": _log(rng, 100, 11008),
                "how": rng.choice(["dynamic", "dynamic", "axis0", "axis1", "e5m2"])}
    return {"kind": kind, "n": _log(rng, 1, 16), "c": rng.choice([1, 3, 3, 8, 20]), "h": rng.randint(28, 224),
            "w": rng.randint(28, 224), "cout": _log(rng, 8, 64), "ks": rng.choice([3, 5, 7]), "stride": rng.choice([1, 2, 2]),
            "pad": 1, "group": 1, "gm": _log(rng, 1, 512), "gn": _log(rng, 10, 2048), "gk": _log(rng, 64, 2048),
            "tb": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs --

def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, device=DEV, generator=g).mul_(std)


def _amax_scale(a):
    s = a / torch.full_like(a, 448.0)  # a division by a number would be a product with its reciprocal
    return torch.where(s > 0, s, torch.ones_like(s))


def _e4m3(v):
    """fp32 values to the E4M3 values nearest to them, as torch float8."""
    return v.clamp(-448.0, 448.0).to(torch.float8_e4m3fn)


def _weight(g, k, n, per_channel=True, nk=False):
    """E4M3 codes [K, N] (or [N, K]) of N(0, 1/sqrt(K)) weights, and their scales."""
    w = _randn(g, n, k, std=k ** -0.5) if nk else _randn(g, k, n, std=k ** -0.5)
    dim = 1 if nk else 0
    a = w.abs().amax(dim=dim, keepdim=True) if per_channel else w.abs().amax().reshape(1, 1)
    s = _amax_scale(a)
    return _e4m3(w / s), s.reshape(-1).contiguous()


def _block_shapes(case):
    h, f = case["hidden"], case["ffn"]
    return [("qkv", h, 3 * h), ("o", h, h), ("up", h, f), ("down", f, h)]


def _raw(case, seed):
    """Everything that is made from the seed, before this package sees it."""
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 11)
    kind = case["kind"]
    r = {}
    if kind == "block":
        r["x"] = _randn(g, case["m"], case["hidden"])
        for name, k, n in _block_shapes(case):
            q, s = _weight(g, k, n)
            r[name] = (q, s, _randn(g, n, std=0.01))
    elif kind == "gemm":
        x = _randn(g, case["m"], case["k"])
        r["sa"] = _amax_scale(x.abs().amax()).reshape(1)
        r["a"] = _e4m3(x / r["sa"])
        r["q"], r["s"] = _weight(g, case["k"], case["n"])
        r["b"] = _randn(g, case["n"], std=0.01) if case["bias"] else None
    elif kind == "mlp":
        r["x"] = torch.rand(case["m"], case["d0"], device=DEV, generator=g)
        dims = [case["d%d" % i] for i in range(4)]
        r["layers"] = []
        for k, n in zip(dims, dims[1:]):
            if case["weights"] == "e4m3":
                q, s = _weight(g, k, n, per_channel=False, nk=True)
            else:
                q, s = _randn(g, n, k, std=k ** -0.5), None
            r["layers"].append((q, s, _randn(g, n, std=0.01)))
    elif kind == "w8a32":
        r["x"] = _randn(g, case["m"], case["k"])
        r["q"], r["s"] = _weight(g, case["k"], case["n"])
        r["b"] = _randn(g, case["n"], std=0.01)
    elif kind == "conv":
        cg = case["c"] // case["group"]
        r["x"] = _randn(g, case["n"], case["c"], case["h"], case["w"])
        q, r["s"] = _weight(g, cg * case["ks"] ** 2, case["cout"], nk=True)
        r["q"] = q.reshape(case["cout"], cg, case["ks"], case["ks"])
        r["b"] = _randn(g, case["cout"], std=0.01)
    elif kind == "load":
        shape = (case["n"], case["k"]) if case["nk"] else (case["k"], case["n"])
        r["w"] = _randn(g, *shape, std=0.02)
        r["s"] = _amax_scale(r["w"].abs().amax(dim=1 if case["nk"] else 0))
    elif kind == "codec":
        r["x"] = _randn(g, case["rows"], case["cols"])
        dim = {"axis0": 1, "axis1": 0}.get(case["how"])
        r["s"] = _amax_scale(r["x"].abs().amax(dim=dim) if dim is not None else r["x"].abs().amax().reshape(1))
    else:
        cg = case["c"] // case["group"]
        r["x"] = _randn(g, case["n"], case["c"], case["h"], case["w"])
        r["w"] = _randn(g, case["cout"], cg, case["ks"], case["ks"], std=(cg * case["ks"] ** 2) ** -0.5)
        r["b"] = _randn(g, case["cout"], std=0.01)
        r["ga"] = _randn(g, case["gm"], case["gk"])
        shape = (case["gn"], case["gk"]) if case["tb"] else (case["gk"], case["gn"])
        r["gb"] = _randn(g, *shape, std=case["gk"] ** -0.5)
        r["gc"] = _randn(g, case["gn"], std=0.01)
    return r


def _out_hw(case):
    return tuple((case[d] + 2 * case["pad"] - case["ks"]) // case["stride"] + 1 for d in ("h", "w"))


def _u8(q):
    return q.view(torch.uint8)


# ----------------------------------------------------------------- programs --

def prepare(case, seed):
    """Packed weights, inputs, outputs and workspaces, as an engine keeps them."""
    r = _raw(case, seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "block":
        m, dt = case["m"], {"up": torch.float32}
        st["x"] = r["x"]
        st["w"] = {}
        st["y"] = {}
        for name, k, n in _block_shapes(case):
            q, s, b = r[name]
            st["w"][name] = (capi.pack_weight(_u8(q), w_is_nk=False), s, b, k, n)
            st["y"][name] = torch.empty((m, n), dtype=dt.get(name, torch.bfloat16), device=DEV)
        kk = max(case["hidden"], case["ffn"])
        st["ws"] = torch.empty(capi.lib().lcml_fp8_gemm_dynamic_workspace_bytes(m, kk, capi.KERNEL_MFMA),
                               dtype=torch.uint8, device=DEV)
        st["parts"] = capi.amax_parts_buffer(m, case["ffn"], DEV)
    elif kind == "gemm":
        st.update(a=_u8(r["a"]), sa=r["sa"], w=capi.pack_weight(_u8(r["q"]), w_is_nk=False), s=r["s"], b=r["b"],
                  y=torch.empty((case["m"], case["n"]), dtype=DTYPES[case["out"]], device=DEV))
    elif kind == "mlp":
        st["x"] = r["x"]
        st["layers"] = []
        for q, s, b in r["layers"]:
            n, k = q.shape
            w = capi.pack_weight(_u8(q), w_is_nk=True) if s is not None else q
            st["layers"].append((w, s, b, k, n, torch.empty((case["m"], n), dtype=torch.float32, device=DEV)))
    elif kind == "w8a32":
        st.update(x=r["x"], w=capi.pack_weight(_u8(r["q"]), w_is_nk=False), s=r["s"], b=r["b"],
                  y=torch.empty((case["m"], case["n"]), dtype=DTYPES[case["out"]], device=DEV))
    elif kind == "conv":
        n, c, h, w = r["x"].shape
        st.update(x=r["x"], w=capi.pack_conv_weight(_u8(r["q"]), group=case["group"]), s=r["s"], b=r["b"],
                  q=torch.empty((n, h, w, c), dtype=torch.uint8, device=DEV),
                  sx=torch.empty(1, dtype=torch.float32, device=DEV),
                  ws=torch.empty(capi.DYNAMIC_WORKSPACE_BYTES, dtype=torch.uint8, device=DEV),
                  y=torch.empty((n, case["cout"], *_out_hw(case)), dtype=DTYPES[case["out"]], device=DEV))
    elif kind == "load":
        st.update(w=r["w"], s=r["s"], q=torch.empty(r["w"].shape, dtype=torch.uint8, device=DEV))
    elif kind == "codec":
        st.update(x=r["x"], s=r["s"], q=torch.empty(r["x"].shape, dtype=torch.uint8, device=DEV),
                  y=torch.empty_like(r["x"]), sx=torch.empty(1, dtype=torch.float32, device=DEV),
                  ws=torch.empty(capi.DYNAMIC_WORKSPACE_BYTES, dtype=torch.uint8, device=DEV))
    else:
        st.update(r)
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):  # once eagerly, so that the capture loads nothing
            _pass(st)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        st["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(st["graph"]):
            st["out"] = _pass(st)
        torch.cuda.synchronize()
    return st


def _pass(st):
    """The calls of one pass."""
    case = st["case"]
    kind = case["kind"]
    if kind == "block":
        kern, m, y = KERNELS[case["kernel"]], case["m"], st["y"]

        def linear(x, name, act=capi.ACT_NONE, **kw):
            w, s, b, k, n = st["w"][name]
            if m <= 16:
                return capi.gemm_dynamic(x, w, s, n, k, c=b, act=act, out=y[name], kernel=kern, workspace=st["ws"])
            return capi.gemm_dynamic_ex(x, w, s, n, k, c=b, act=act, out=y[name], kernel=kern, workspace=st["ws"], **kw)

        linear(st["x"], "qkv")
        linear(st["x"], "o")
        if m <= 16:
            linear(st["x"], "up", capi.ACT_GELU_ERF)
            linear(y["up"], "down")
        else:  # the down-projection takes its scale from the up-projection's partial maxima
            parts = linear(st["x"], "up", capi.ACT_GELU_ERF, y_amax_part=st["parts"])[1]
            linear(y["up"], "down", x_amax=(st["parts"], parts))
        return dict(y)
    if kind == "gemm":
        return capi.gemm(st["a"], st["sa"], st["w"], st["s"], case["n"], case["k"], c=st["b"], act=ACTS[case["act"]],
                         out=st["y"], kernel=KERNELS[case["kernel"]])
    if kind == "mlp":
        h, outs = st["x"], []
        for i, (w, s, b, k, n, y) in enumerate(st["layers"]):
            act = capi.ACT_RELU if i < 2 else capi.ACT_NONE
            if s is not None:
                h = capi.gemm_w8a32(h, w, s, n, k, c=b, act=act, out=y)
            else:
                h = capi.sgemm(h, w, c=b, trans_b=True, act=act)
            outs.append(h)
        return outs
    if kind == "w8a32":
        return capi.gemm_w8a32(st["x"], st["w"], st["s"], case["n"], case["k"], c=st["b"], act=ACTS[case["act"]],
                               out=st["y"])
    if kind == "conv":
        q, sx = capi.quantize_nhwc(st["x"], out=st["q"], scale_out=st["sx"], workspace=st["ws"])
        y = capi.conv2d(q, sx, st["w"], st["s"], case["cout"], (case["ks"], case["ks"]),
                        strides=(case["stride"],) * 2, pads=(case["pad"],) * 2, bias=st["b"], act=ACTS[case["act"]],
                        out=st["y"], kernel=KERNELS[case["kernel"]], group=case["group"])
        return y, q, sx
    if kind == "load":
        q = capi.quantize(st["w"], st["s"], axis=0 if case["nk"] else 1, out=st["q"])
        return q, capi.pack_weight(q, w_is_nk=case["nk"])
    if kind == "codec":
        how = case["how"]
        if how == "dynamic":
            q, s = capi.quantize_dynamic(st["x"], out=st["q"], scale_out=st["sx"], workspace=st["ws"])
            return q, s, capi.dequantize(q, s, out=st["y"])
        if how == "e5m2":
            q = capi.quantize_e5m2(st["x"], st["s"], out=st["q"])
            return q, capi.dequantize_e5m2(q, st["s"], out=st["y"])
        axis = int(how[-1])
        q = capi.quantize(st["x"], st["s"], axis=axis, out=st["q"])
        return q, capi.dequantize(q, st["s"], axis=axis, out=st["y"])
    y = capi.conv2d_f32(st["x"], st["w"], st["b"], (case["stride"],) * 2, (case["pad"],) * 2, group=case["group"],
                        act=capi.ACT_RELU)
    return y, capi.sgemm(st["ga"], st["gb"], c=st["gc"], trans_b=case["tb"])


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _pass(state)


# ------------------------------------------------------- 64-bit expectation --

def _act(v, act):
    if act == "relu":
        return v.clamp_min(0.0)
    if act == "gelu":
        return 0.5 * v * (1.0 + torch.erf(v * (0.5 ** 0.5)))
    return v


def _qdq_dynamic(x):
    """fp32 x through a dynamic E4M3 quantisation, as 64-bit values and the scale."""
    s = _amax_scale(x.abs().amax())
    return _e4m3(x / s).double(), s


def _conv64(x, w, case):
    """Convolution in 64 bits, an image and a group at a time."""
    oh, ow = _out_hw(case)
    grp = case["group"]
    cg, mg = case["c"] // grp, case["cout"] // grp
    y = torch.empty((x.shape[0], case["cout"], oh * ow), dtype=torch.float64, device=x.device)
    for i in range(x.shape[0]):
        for j in range(grp):
            cols = F.unfold(x[i:i + 1, j * cg:(j + 1) * cg].double(), case["ks"], padding=case["pad"],
                            stride=case["stride"])[0]
            y[i, j * mg:(j + 1) * mg] = w[j * mg:(j + 1) * mg].reshape(mg, -1).double() @ cols
    return y.reshape(x.shape[0], case["cout"], oh, ow)


def exact(case, seed):
    r = _raw(case, seed)
    kind = case["kind"]
    if kind == "block":
        y = {}

        def linear(x, name, act="none"):
            q, s, b = r[name]
            xq, sx = _qdq_dynamic(x)
            y[name] = _act(xq @ q.double() * (sx.double() * s.double()) + b.double(), act)
            return y[name]

        linear(r["x"], "qkv")
        linear(r["x"], "o")
        linear(linear(r["x"], "up", "gelu").float(), "down")
        return y
    if kind == "gemm":
        v = r["a"].double() @ r["q"].double() * (r["sa"].double() * r["s"].double())
        return _act(v if r["b"] is None else v + r["b"].double(), case["act"])
    if kind == "mlp":
        h, outs = r["x"].double(), []
        for i, (q, s, b) in enumerate(r["layers"]):
            v = h @ q.double().t()
            h = _act((v if s is None else v * s.double()) + b.double(), "relu" if i < 2 else "none")
            outs.append(h)
        return outs
    if kind == "w8a32":
        return _act(r["x"].double() @ r["q"].double() * r["s"].double() + r["b"].double(), case["act"])
    if kind == "conv":
        xq, sx = _qdq_dynamic(r["x"])
        v = _conv64(xq, r["q"].double(), case) * (sx.double() * r["s"].double()).reshape(1, -1, 1, 1)
        return _act(v + r["b"].double().reshape(1, -1, 1, 1), case["act"]), None, sx.double().reshape(1)
    if kind == "load":
        return None
    if kind == "codec":
        s = r["s"].reshape(-1, 1) if case["how"] == "axis0" else r["s"]
        v = r["x"] / s
        q = v.clamp(-57344.0, 57344.0).to(torch.float8_e5m2) if case["how"] == "e5m2" else _e4m3(v)
        y = q.double() * s.double()
        return (None, r["s"].double(), y) if case["how"] == "dynamic" else (None, y)
    v = _conv64(r["x"], r["w"], case) + r["b"].double().reshape(1, -1, 1, 1)
    gb = r["gb"].double()
    return _act(v, "relu"), r["ga"].double() @ (gb.t() if case["tb"] else gb) + r["gc"].double()


# ---------------------------------------------------------- work, tolerance --

def work(case):
    """Bytes read once and written once, and multiply-adds as two operations."""
    kind = case["kind"]
    if kind == "block":
        m, sh = case["m"], _block_shapes(case)
        b = sum(k * n + 8 * n + m * n * (4 if name == "up" else 2) for name, k, n in sh)
        return {"bytes": b + 4 * m * case["hidden"], "flops": 2 * m * sum(k * n for _, k, n in sh)}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k + k * n + 4 * n * (1 + case["bias"]) + m * n * (2 if case["out"] == "bf16" else 4),
                "flops": 2 * m * n * k}
    if kind == "mlp":
        m, d = case["m"], [case["d%d" % i] for i in range(4)]
        wb = 1 if case["weights"] == "e4m3" else 4
        kn = [(k, n) for k, n in zip(d, d[1:])]
        return {"bytes": 4 * m * sum(d) + sum(wb * k * n + 4 * n for k, n in kn), "flops": 2 * m * sum(k * n for k, n in kn)}
    if kind == "w8a32":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4 * m * k + k * n + 8 * n + m * n * (2 if case["out"] == "bf16" else 4), "flops": 2 * m * n * k}
    if kind == "conv":
        oh, ow = _out_hw(case)
        x, y = case["n"] * case["c"] * case["h"] * case["w"], case["n"] * case["cout"] * oh * ow
        kk = case["c"] // case["group"] * case["ks"] ** 2
        return {"bytes": 5 * x + kk * case["cout"] + 8 * case["cout"] + y * (2 if case["out"] == "bf16" else 4),
                "flops": 2 * y * kk}
    if kind == "load":
        kn = case["k"] * case["n"]
        return {"bytes": 6 * kn + 4 * case["n"], "flops": 2 * kn}
    if kind == "codec":
        n = case["rows"] * case["cols"]
        return {"bytes": 9 * n, "flops": 3 * n}
    oh, ow = _out_hw(case)
    y, kk = case["n"] * case["cout"] * oh * ow, case["c"] // case["group"] * case["ks"] ** 2
    gm, gn, gk = case["gm"], case["gn"], case["gk"]
    return {"bytes": 4 * (case["n"] * case["c"] * case["h"] * case["w"] + case["cout"] * (kk + 1) + y
                          + gm * gk + gk * gn + gn + gm * gn),
            "flops": 2 * y * kk + 2 * gm * gn * gk}


def tolerance(case):
    """About four times what the summation orders of the present kernels differ by."""
    kind = case["kind"]
    if kind in ("load", "codec"):  # codes, and one rounded product each
        return "exact"
    if kind == "block" or case.get("out") == "bf16":
        # bf16 roundings that fall on the other side (one of a small output's
        # values alone is up to 1e-3 of its norm), and, in the block, codes
        # of the GELU output that do
        return {"rel": 1e-3, "max": 2e-2}
    if case.get("kernel") == "auto_fp8":  # the FP8 matrix instructions drop low product bits: 1.5e-5
        return {"rel": 6e-5, "max": 2e-3}
    return {"rel": 4e-6, "max": 1.6e-4}  # 32-bit sums: 1e-7 to 8e-7 seen
