"""The measured work of the library: what a detector built on it calls, per frame and per batch.

Cases go through the C ABI as `thintnpu_amd.capi` binds it, on torch device
tensors, and one through the `npu` device with `CapturedForward`.  Sequences
that a serving program replays unchanged are recorded once into a HIP graph
(`"graph"` below: the graph is the plan such a program keeps); the others are
called one by one.  Sizes are those of 640-pixel and 1280-pixel inputs of the
YOLOv8s / YOLO11s / YOLO26s layers, at batch 1 and 32; `draw` takes sizes in
between, odd ones included.
"""
import math

import torch

KINDS = ("c2f", "affine", "neck", "sppf", "decode", "tail", "attention", "chain", "bmm", "npu_tail")


def listed():
    return [
        # One frame's C2f block between two convolutions, called op by op: the smallest
        # calls, where the host's share of a call and the launch are most of the time.
        {"name": "c2f_frame", "kind": "c2f", "n": 1, "c": 128, "h": 80, "w": 80},
        # Batch norm folded to a per-channel affine + SiLU after the three neck
        # convolutions of a batch, each on the whole tensor and on its C2f half: the
        # bandwidth-bound elementwise path.
        {"name": "affine_batch", "kind": "affine", "n": 32, "s": 80},
        # The neck's data movement for a batch: the C2f concat, the 2x upsample and the
        # upsample feeding a concat.  The largest tensors of the path.
        {"name": "neck_batch", "kind": "neck", "n": 32, "s": 80},
        # The SPPF block of a batch of 1280-pixel inputs: three chained max pools and
        # their concat.
        {"name": "sppf_batch", "kind": "sppf", "n": 32, "c": 256, "h": 40, "w": 40},
        # The anchor-free head (YOLOv8 / YOLO11: 16 bins a side) of a batch, decoded for
        # a non-maximum suppression that runs elsewhere.
        {"name": "decode_batch", "kind": "decode", "n": 32, "px_h": 640, "px_w": 640, "nc": 80},
        # The end of a YOLO26 forward: decode of the direct-distance head, then the
        # NMS-free top-300 selection.  One frame (latency), a batch, and 1280-pixel frames.
        {"name": "tail_frame", "kind": "tail", "n": 1, "px_h": 640, "px_w": 640, "nc": 80},
        {"name": "tail_batch", "kind": "tail", "n": 32, "px_h": 640, "px_w": 640, "nc": 80},
        {"name": "tail_1280", "kind": "tail", "n": 4, "px_h": 1280, "px_w": 1280, "nc": 80},
        # The C2PSA attention of eight frames in the blocked layout (the fused entry
        # takes one image a call) with the positional branch's channel select.
        {"name": "attention_frames", "kind": "attention", "images": 8, "heads": 4, "t": 400},
        # The same attention at 1280 pixels (40 x 40 tokens), beyond the fused entry's
        # tokens: channel select, scale, q^T k, row softmax, v p^T.
        {"name": "attention_1280", "kind": "chain", "heads": 4, "t": 1600},
        # The attention of a batch as the unpatched PyTorch module computes it: rank-3
        # products over strided views of the NCHW qkv tensor.
        {"name": "attention_batch", "kind": "bmm", "n": 32, "heads": 4, "t": 400},
        # The frame's tail on the npu device: a captured forward called on each new head
        # output, and the detections read back to the host.
        {"name": "npu_frame_tail", "kind": "npu_tail", "n": 1, "px_h": 640, "px_w": 640, "nc": 80},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _pixels(rng, low, high):
    return 32 * rng.randint(low // 32, high // 32)


def draw(rng):
    kind = rng.choice(KINDS)
    if kind == "c2f":
        while True:
            c = {"kind": kind, "n": rng.randint(1, 4), "c": 32 * rng.randint(1, 16), "h": _log(rng, 7, 160), "w": _log(rng, 7, 160)}
            if c["n"] * c["c"] * c["h"] * c["w"] <= 4 * 128 * 80 * 80:
                return c
    if kind in ("affine", "neck"):
        while True:
            c = {"kind": kind, "n": _log(rng, 1, 32), "s": _log(rng, 20, 160)}
            if c["n"] * c["s"] ** 2 <= 32 * 80 * 80:
                return c
    if kind == "sppf":
        while True:
            c = {"kind": kind, "n": _log(rng, 1, 32), "c": 16 * rng.randint(4, 32), "h": rng.randint(10, 44), "w": rng.randint(10, 44)}
            if c["n"] * c["c"] * c["h"] * c["w"] <= 32 * 256 * 40 * 40:
                return c
    if kind in ("decode", "tail", "npu_tail"):
        while True:
            c = {"kind": kind, "n": 1 if kind == "npu_tail" else _log(rng, 1, 32), "px_h": _pixels(rng, 320, 1280), "px_w": _pixels(rng, 320, 1280),
                 "nc": rng.choice([80, 80, 80, rng.randint(1, 200)])}
            if c["n"] * c["px_h"] * c["px_w"] * (c["nc"] + 64) <= 32 * 640 * 640 * 144:
                return c
    if kind == "attention":
        return {"kind": kind, "images": rng.randint(1, 8), "heads": rng.randint(2, 4), "t": 8 * rng.randint(17, 55)}
    if kind == "chain":
        return {"kind": kind, "heads": rng.randint(2, 4), "t": rng.randint(520, 1600)}
    while True:
        c = {"kind": kind, "n": _log(rng, 1, 32), "heads": rng.randint(2, 8), "t": rng.randint(100, 900)}
        if c["n"] * c["heads"] * c["t"] ** 2 <= 32 * 4 * 400 * 400:
            return c


# ------------------------------------------------------------------ sizes

KEY, DIM = 32, 64          # key and value channels of a head
MAX_DET = 300


def _affine_shapes(case):
    s = case["s"]
    return [(128, s, s), (256, (s + 1) // 2, (s + 1) // 2), (512, (s + 3) // 4, (s + 3) // 4)]


def _levels(case):
    return [(case["px_h"] // s, case["px_w"] // s) for s in (8, 16, 32)], [8.0, 16.0, 32.0]


def _anchors(case):
    return sum(h * w for h, w in _levels(case)[0])


# ------------------------------------------------------------------ inputs

def _rand(seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, mean=0.0, std=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * std + mean).half()

    def uniform(*shape, low=0.0, high=1.0):
        return (torch.rand(shape, generator=g, device="cuda") * (high - low) + low).half()

    return normal, uniform


def _inputs(case, seed):
    normal, uniform = _rand(seed)
    kind = case["kind"]
    if kind == "c2f":  # a convolution's NCHW output and its folded batch norm
        c1 = case["c"] // 16
        return {"x": normal(case["n"], case["c"], case["h"], case["w"]), "s": uniform(1, c1, 1, 1, 16, low=0.5, high=1.5),
                "b": normal(1, c1, 1, 1, 16, std=0.1)}
    if kind == "affine":
        sets = []
        for c, h, w in _affine_shapes(case):
            x = normal(case["n"], c // 16, h, w, 16)
            s, b = uniform(1, c // 16, 1, 1, 16, low=0.5, high=1.5), normal(1, c // 16, 1, 1, 16, std=0.1)
            half = c // 32
            sets += [(x, s, b), (x[:, half:], s[:, half:], b[:, half:])]
        return {"sets": sets}
    if kind == "neck":
        n, s = case["n"], case["s"]
        low = (s + 1) // 2
        return {"chunks": [normal(n, 4, s, s, 16) for _ in range(4)], "up": normal(n, 16, low, low, 16), "skip": normal(n, 8, 2 * low, 2 * low, 16)}
    if kind == "sppf":
        return {"x": normal(case["n"], case["c"] // 16, case["h"], case["w"], 16)}
    if kind == "decode":
        a = _anchors(case)
        return {"boxes": normal(case["n"], 64, a, std=3.0), "scores": normal(case["n"], case["nc"], a, mean=-4.0, std=2.0)}
    if kind in ("tail", "npu_tail"):  # one head tensor, as the concatenated convolution outputs leave it
        a = _anchors(case)
        return {"head": torch.cat([uniform(case["n"], 4, a, high=20.0), normal(case["n"], case["nc"], a, mean=-4.0, std=2.0)], 1)}
    if kind == "attention":
        c1 = case["heads"] * (2 * KEY + DIM) // 16
        return {"qkv": [normal(1, c1, case["t"], 16) for _ in range(case["images"])]}
    if kind == "chain":
        return {"qkv": normal(1, case["heads"] * (2 * KEY + DIM) // 16, case["t"], 16)}
    return {"qkv": normal(case["n"] * case["heads"], 2 * KEY + DIM, case["t"])}


def _scale():
    return float(torch.tensor(KEY ** -0.5, dtype=torch.float64).half())


# ------------------------------------------------------------------ the calls

def _c2f(capi, st):
    x = capi.pack_nc1hwc0(st["x"])
    x = capi.affine_silu(x, st["s"], st["b"])
    half = x.shape[1] // 2
    a, b = x[:, :half], x[:, half:]
    z = capi.silu_add(b, a)
    y = capi.cat([a, b, z], 1)
    return [y, capi.unpack_nc1hwc0(y)]


def _affine(capi, st):
    return [capi.affine_silu(*operands) for operands in st["sets"]]


def _neck(capi, st):
    return [capi.cat(st["chunks"], 1), capi.upsample2x_nc1hwc0(st["up"]), capi.upsample_cat_nc1hwc0([st["up"], st["skip"]], [True, False])]


def _sppf(capi, st):
    return [capi.sppf_nc1hwc0(st["x"], 5, 3)]


def _decode(capi, st):
    return [capi.detect_decode(st["boxes"], st["scores"], st["shapes"], st["strides"])]


def _tail(capi, st):
    head = st["head"]
    decoded = capi.detect_decode(head[:, :4], head[:, 4:], st["shapes"], st["strides"])
    return [decoded, capi.detection_select(decoded.transpose(1, 2), MAX_DET)]


def _attention(capi, st):
    heads, out = st["heads"], []
    for qkv in st["qkv"]:
        out.append(capi.attention(qkv, heads, KEY, DIM, _scale()))
        out.append(capi.channel_select(qkv, heads, 2 * KEY, DIM))
    return out


def _chain(capi, st):
    qkv, heads = st["qkv"], st["heads"]
    query = capi.binary_scalar(capi.MUL, capi.channel_select(qkv, heads, 0, KEY), _scale())
    scores = capi.layout_bmm(query, qkv, True, False, False, heads, 0, KEY, KEY, KEY)
    probability = capi.softmax(scores, 2)
    return [scores, probability, capi.layout_bmm(qkv, probability, False, True, True, heads, 2 * KEY, DIM)]


def _bmm(capi, st):
    q, k, v = st["qkv"].split((KEY, KEY, DIM), 1)
    scores = capi.binary_scalar(capi.MUL, capi.bmm(q.transpose(1, 2), k), _scale())
    probability = capi.softmax(scores, 2)
    return [scores, probability, capi.bmm(v, probability.transpose(1, 2))]


CALLS = {"c2f": _c2f, "affine": _affine, "neck": _neck, "sppf": _sppf, "decode": _decode, "tail": _tail, "attention": _attention,
         "chain": _chain, "bmm": _bmm}
GRAPHS = {"affine", "decode", "tail", "attention", "chain", "bmm"}


def prepare(case, seed):
    if case["kind"] == "npu_tail":
        return _prepare_npu(case, seed)
    from thintnpu_amd import capi
    capi.lib()
    st = _inputs(case, seed)
    if case["kind"] in ("decode", "tail"):
        st["shapes"], st["strides"] = _levels(case)
    if "heads" in case:
        st["heads"] = case["heads"]
    call = CALLS[case["kind"]]
    if case["kind"] in GRAPHS:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            st["outputs"] = call(capi, st)
        st["graph"] = graph
    st["call"] = lambda: call(capi, st)
    return st


def _prepare_npu(case, seed):
    import thin_backend
    from thin_backend.graph import CapturedForward
    thin_backend.load_flow_libraries()
    shapes, strides = _levels(case)
    flat = [v for hw in shapes for v in hw]
    head = _inputs(case, seed)["head"].cpu().to("npu")

    def forward(x):
        boxes, scores = x.split((4, x.shape[1] - 4), 1)
        decoded = torch.ops.thin_fused.detect_decode(boxes, scores, flat, strides)
        return torch.ops.thin_native_flow.detection_select(decoded.transpose(1, 2), MAX_DET)

    return {"head": head, "forward": CapturedForward(forward, head)}


def run(state):
    if "forward" in state:
        with torch.inference_mode():
            return state["forward"](state["head"]).cpu()
    if "graph" in state:
        state["graph"].replay()
        return state["outputs"]
    return state["call"]()


# ------------------------------------------------------------------ what a pass cannot do without

def work(case):
    """fp16 elements read and written once each by every call of the pass, and the operations of
    its arithmetic (a multiply-add counts two, an exponential one)."""
    kind = case["kind"]
    if kind == "c2f":
        e = case["n"] * case["c"] * case["h"] * case["w"]
        # pack, affine: 2 each; silu_add: 3 halves; cat: 3 halves in and out; unpack: 3 halves in and out
        return {"bytes": 2 * e * (2 + 2 + 1.5 + 3 + 3), "flops": 10 * e}
    if kind == "affine":
        e = sum(case["n"] * c * h * w for c, h, w in _affine_shapes(case)) * 1.5
        return {"bytes": 4 * e, "flops": 6 * e}
    if kind == "neck":
        n, s, low = case["n"], case["s"], (case["s"] + 1) // 2
        up, skip = n * 256 * low * low, n * 128 * 4 * low * low
        return {"bytes": 2 * (2 * n * 256 * s * s + 5 * up + 5 * up + 2 * skip), "flops": 0}
    if kind == "sppf":
        e = case["n"] * case["c"] * case["h"] * case["w"]
        return {"bytes": 2 * 5 * e, "flops": 3 * 8 * e}
    if kind == "decode":
        e = case["n"] * _anchors(case)
        return {"bytes": 2 * e * (64 + 4 + 2 * case["nc"]), "flops": e * (64 * 4 + 4 * case["nc"])}
    if kind in ("tail", "npu_tail"):
        e = case["n"] * _anchors(case)
        return {"bytes": 2 * e * 3 * (4 + case["nc"]) + case["n"] * MAX_DET * 24, "flops": e * 5 * case["nc"]}
    t, heads = case["t"], case["heads"]
    if kind == "attention":
        e = case["images"] * heads * t
        return {"bytes": 2 * e * (2 * KEY + 4 * DIM), "flops": e * t * (2 * KEY + 2 * DIM + 4)}
    e = heads * t * case.get("n", 1)
    small = 2 * e * (2 * KEY + 2 * DIM)
    if kind == "chain":  # select and scale q, then scores and probabilities written and read back
        return {"bytes": small + 2 * e * 4 * KEY + 2 * e * 4 * t, "flops": e * t * (2 * KEY + 2 * DIM + 4)}
    return {"bytes": small + 2 * e * 6 * t, "flops": e * t * (2 * KEY + 2 * DIM + 5)}


def tolerance(case):
    """Moved values and selected rows keep their bits (the decode feeding a selection too: its steps are
    single correctly rounded operations, and an ulp would reorder rows).  Elsewhere the figures are about
    four times the measured distance of the fp16 results from the same sums in 64 bits."""
    kind = case["kind"]
    if kind in ("neck", "sppf", "tail", "npu_tail"):
        return "exact"
    if kind in ("c2f", "affine"):
        return {"rel": 1.5e-3, "max": 0.02}
    if kind == "decode":
        return {"rel": 1e-3, "max": 0.02}
    return {"rel": 2.5e-3, "max": 0.02}


# ------------------------------------------------------------------ the same in 64 bits

def _silu(x):
    return x * torch.sigmoid(x)


def _blocked(x):
    """[1, C1, T, 16] as [channels, T]."""
    return x.permute(0, 1, 3, 2).reshape(-1, x.shape[2])


def _attend(q, k, v):
    scores = torch.bmm(q.transpose(1, 2).contiguous(), k.contiguous()) * KEY ** -0.5
    probability = torch.softmax(scores, 2)
    return scores, probability, torch.bmm(v.contiguous(), probability.transpose(1, 2).contiguous())


def _decoded(case, distances, scores):
    """[N, 4, A] distances in grid cells and class logits to boxes in pixels and scores."""
    shapes, strides = _levels(case)
    centre, stride = [], []
    for (h, w), s in zip(shapes, strides):
        y, x = torch.meshgrid(torch.arange(h, device="cuda").double() + 0.5, torch.arange(w, device="cuda").double() + 0.5, indexing="ij")
        centre.append(torch.stack([x.reshape(-1), y.reshape(-1)]))
        stride.append(torch.full((h * w,), s, dtype=torch.float64, device="cuda"))
    centre, stride = torch.cat(centre, 1), torch.cat(stride)
    boxes = torch.cat([centre - distances[:, :2], centre + distances[:, 2:]], 1) * stride
    return torch.cat([boxes, torch.sigmoid(scores)], 1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "npu_tail":
        return None
    st = _inputs(case, seed)
    if kind == "c2f":
        n, c, h, w = st["x"].shape
        s, b = (st[k].double().reshape(1, c, 1, 1) for k in ("s", "b"))
        x = _silu(st["x"].double() * s + b)
        a, b = x.split(c // 2, 1)
        y = torch.cat([a, b, a + _silu(b)], 1)
        return [y.reshape(n, -1, 16, h, w).permute(0, 1, 3, 4, 2), y]
    if kind == "affine":
        return [_silu(x.double() * s.double() + b.double()) for x, s, b in st["sets"]]
    if kind == "neck":
        up = st["up"].repeat_interleave(2, 2).repeat_interleave(2, 3)
        return [torch.cat(st["chunks"], 1).double(), up.double(), torch.cat([up, st["skip"]], 1).double()]
    if kind == "sppf":
        x = st["x"].double()
        n, c1, h, w, _ = x.shape
        slots = [x.permute(0, 1, 4, 2, 3).reshape(n, c1 * 16, h, w)]
        for _ in range(3):
            slots.append(torch.nn.functional.max_pool2d(slots[-1], 5, 1, 2))
        return [torch.cat([y.reshape(n, c1, 16, h, w).permute(0, 1, 3, 4, 2) for y in slots], 1)]
    if kind == "decode":
        n, _, a = st["boxes"].shape
        bins = torch.arange(16, device="cuda", dtype=torch.float64).reshape(1, 1, 16, 1)
        distances = (torch.softmax(st["boxes"].double().reshape(n, 4, 16, a), 2) * bins).sum(2)
        return [_decoded(case, distances, st["scores"].double())]
    if kind == "tail":
        head = st["head"].double()
        return [_decoded(case, head[:, :4], head[:, 4:]), None]
    heads, t = case["heads"], case["t"]
    if kind == "bmm":
        return list(_attend(*st["qkv"].double().split((KEY, KEY, DIM), 1)))
    out = []
    for qkv in st["qkv"] if kind == "attention" else [st["qkv"]]:
        q, k, v = _blocked(qkv.double()).reshape(heads, 2 * KEY + DIM, t).split((KEY, KEY, DIM), 1)
        scores, probability, mixed = _attend(q, k, v)

        def block(x):
            return x.reshape(1, -1, 16, t).permute(0, 1, 3, 2)

        out += [block(mixed), block(v.contiguous())] if kind == "attention" else [scores, probability, block(mixed)]
    return out
