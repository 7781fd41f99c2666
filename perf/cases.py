"""Workloads of the convolution library, from the smallest call to a whole network trunk.

A layer case is one forward pass of one fp32 NCHW convolution through the public entry points, the way
the layer classes and the benchmark call them: the library's own untuned choice of algorithm, pipeline and
tile shape; filter re-layout of the implicit GEMM done once beforehand; the Winograd filter transform inside
the pass ("online", the default of the drivers) or done once beforehand (`offline`).  A trunk case is the
13-layer VGG-16 convolution stack with its ReLUs and 2x2 max pools, each layer reading what the one before wrote.

Fields of a layer case: algo ("auto": the rule behind `-a auto`; "winograd"; "im2col"), n, c, h, w (input),
k (output channels), ks, stride, pad, bias_relu (bias and ReLU in the epilogue), offline.
Fields of a trunk case: algo "trunk", n, h.
"""
import ctypes
import math

import torch

import fastconv_amd as F

# (C, K) of the VGG-16 convolutions between its 2x2 max pools
TRUNK = (((3, 64), (64, 64)), ((64, 128), (128, 128)), ((128, 256), (256, 256), (256, 256)),
         ((256, 512), (512, 512), (512, 512)), ((512, 512), (512, 512), (512, 512)))


def _layer(name, algo, n, c, k, h, ks=3, stride=1, pad=None, w=None, bias_relu=False, offline=False):
    case = {"algo": algo, "n": n, "c": c, "h": h, "w": h if w is None else w, "k": k, "ks": ks, "stride": stride,
            "pad": ks // 2 if pad is None else pad, "bias_relu": bias_relu, "offline": offline}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # One image, latency: a strided 3x3 layer, the stride-2 entry of a ResNet-50 stage.
        _layer("3x3s2 128-256@56 n1", "im2col", 1, 128, 256, 56, stride=2),
        # One image, an ordinary 3x3 layer of VGG-16, algorithm left to the library.
        _layer("3x3 256-256@56 n1", "auto", 1, 256, 256, 56),
        # One image, the deep VGG-16 layers: few pixels, a filter much larger than the image, filter transform online.
        _layer("wino 512-512@14 n1", "winograd", 1, 512, 512, 14),
        # One image in serving: filter transformed beforehand, bias and ReLU in the epilogue.
        _layer("wino 512-512@28 n1 off", "winograd", 1, 512, 512, 28, bias_relu=True, offline=True),
        # First layer of a network on a batch: three input channels, bound by writing the output.
        _layer("wino 3-64@224 n32", "winograd", 32, 3, 64, 224),
        # Large images, few channels, on a batch: the most expensive single layer of VGG-16.
        _layer("3x3 64-64@224 n32", "auto", 32, 64, 64, 224, bias_relu=True),
        # A size off every grid: channels, image and batch that no tile divides.
        _layer("wino 96-192@35 n8", "winograd", 8, 96, 192, 35, bias_relu=True),
        # Deep 3x3 layer on a batch.
        _layer("3x3 512-512@14 n32", "auto", 32, 512, 512, 14),
        # 1x1 bottleneck layer of ResNet-50 on a batch.
        _layer("1x1 256-64@56 n32", "im2col", 32, 256, 64, 56, ks=1),
        # Strided 3x3 layer of ResNet-50 on a batch.
        _layer("3x3s2 256-256@28 n32", "auto", 32, 256, 256, 28, stride=2),
        # 7x7 stem of ResNet-50 on a batch: the reduction has no whole channels to share a tap.
        _layer("7x7s2 3-64@224 n32", "im2col", 32, 3, 64, 224, ks=7, stride=2),
        # A whole trunk on a batch: what a user of the library runs in the end.
        {"name": "vgg16 trunk n32", "algo": "trunk", "n": 32, "h": 224},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(("3x3", "3x3", "3x3", "1x1", "1x1", "strided", "first", "stem", "trunk"))
    if family == "trunk":
        h = rng.randrange(64, 225)
        return {"algo": "trunk", "n": _log_int(rng, 1, min(32, 32 * 224 * 224 / (h * h))), "h": h}
    while True:
        n, h = _log_int(rng, 1, 64), _log_int(rng, 7, 224)
        w = h if rng.random() < 0.7 else _log_int(rng, 7, 224)
        c, k = _log_int(rng, 16, 1024), _log_int(rng, 16, 1024)
        if rng.random() < 0.6:
            c, k = 16 * max(1, c // 16), 16 * max(1, k // 16)
        ks, stride, algo = 3, 1, rng.choice(("auto", "auto", "winograd", "im2col"))
        if family == "1x1":
            ks, stride, algo = 1, rng.choice((1, 1, 1, 2)), "im2col"
        elif family == "strided":
            ks, stride, algo = rng.choice((3, 3, 5)), 2, "im2col"
        elif family == "first":
            c, algo = rng.randrange(1, 5), rng.choice(("auto", "winograd"))
            h, w = _log_int(rng, 32, 224), _log_int(rng, 32, 224)
        elif family == "stem":
            c, ks, stride, algo = rng.randrange(1, 5), 7, 2, "im2col"
            k, h, w = _log_int(rng, 16, 128), _log_int(rng, 32, 224), _log_int(rng, 32, 224)
        case = _layer(None, algo, n, c, k, h, ks, stride, ks // 2 if rng.random() < 0.9 else 0, w,
                      rng.random() < 0.5, algo == "winograd" and rng.random() < 0.4)
        cost = work(case)
        # between a few microseconds of work and the largest listed layer's
        direct = _shape(case).flops()
        if 1e8 < direct < 1.2e11 and cost["bytes"] < 1e9:
            return case


def _shape(case):
    p, s = case["pad"], case["stride"]
    return F.ConvShape(case["n"], case["c"], case["h"], case["w"], case["k"], case["ks"], case["ks"], s, s, p, p, p, p)


_handle = None


def _library():
    """One handle per process, as a program keeps it; buffers are the caller's own."""
    global _handle
    if _handle is None:
        _handle = F.load(torch.cuda.current_device(), 1 << 20)
    return _handle


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _buffer(nbytes):
    return torch.empty((nbytes + 3) // 4, dtype=torch.float32, device="cuda") if nbytes else None


class _Conv:
    """One layer with its plan, its weights and the buffers that are its own."""

    def __init__(self, L, algo, shape, w, bias, relu, offline):
        self.L, self.shape, self.w, self.bias, self.relu, self.offline = L, shape, w, bias, relu, offline
        self.y_shape = (shape.N, shape.K) + shape.out_hw()
        if algo == "auto":
            algo = "winograd" if L.prefer_winograd(shape) else "im2col"
        self.V_bytes = self.M_bytes = 0
        if algo == "im2col":
            self.pipe = "im2col"
            self.plan = L.igemm_plan(shape, L.igemm_default_config(shape))
            self.U, self.table = _buffer(self.plan.Wp_bytes), _buffer(self.plan.table_bytes)
            self.ws = _buffer(self.plan.ws_bytes)
            L.igemm_pack_filter(self.plan, _ptr(w), _ptr(self.U), _ptr(self.table))
            return
        if L.wino_prefer_onepass(shape):
            self.pipe, self.plan = "onepass", L.wino_onepass_plan(shape)
        else:
            self.pipe = "fused" if L.wino_prefer_fused(shape) else "staged"
            self.plan = L.wino_plan(shape, L.wino_default_config(shape))
            self.V_bytes = self.plan.V_bytes
            self.M_bytes = self.plan.M_bytes if self.pipe == "staged" else 0
        self.U = _buffer(self.plan.U_bytes)
        if offline:
            transform = L.wino_onepass_filter_transform if self.pipe == "onepass" else L.wino_filter_transform
            transform(self.plan, _ptr(w), _ptr(self.U))

    def forward(self, x, V, M, y):
        L, b, r = self.L, _ptr(self.bias), self.relu
        if self.pipe == "im2col":
            L.conv_implicit_gemm(self.plan, _ptr(x), _ptr(self.U), _ptr(self.table), _ptr(y), b, r, _ptr(self.ws))
        elif self.pipe == "onepass":
            L.wino_forward_onepass(self.plan, _ptr(x), _ptr(self.w), _ptr(self.U), _ptr(y), b, r, self.offline)
        elif self.pipe == "fused":
            L.wino_forward_fused(self.plan, _ptr(x), _ptr(self.w), _ptr(self.U), _ptr(V), _ptr(y), b, r, self.offline)
        else:
            L.wino_forward(self.plan, _ptr(x), _ptr(self.w), _ptr(self.U), _ptr(V), _ptr(M), _ptr(y), b, r, self.offline)


def _inputs(gen, n, c, h, w):
    return torch.rand((n, c, h, w), generator=gen, device="cuda") * 2 - 1


def _weights(gen, k, c, ks):
    return torch.randn((k, c, ks, ks), generator=gen, device="cuda") * math.sqrt(2.0 / (ks * ks * c))


def _bias(gen, k):
    return torch.rand((k,), generator=gen, device="cuda") * 0.2 - 0.1


def prepare(case, seed):
    """Images uniform in [-1, 1), He-normal weights; plan, packed filter and workspaces as a program keeps them."""
    L = _library()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["algo"] != "trunk":
        shape = _shape(case)
        x = _inputs(gen, case["n"], case["c"], case["h"], case["w"])
        w = _weights(gen, case["k"], case["c"], case["ks"])
        bias = _bias(gen, case["k"]) if case["bias_relu"] else None
        torch.cuda.synchronize()
        conv = _Conv(L, case["algo"], shape, w, bias, case["bias_relu"], case["offline"])
        L.sync()
        return {"conv": conv, "x": x, "V": _buffer(conv.V_bytes), "M": _buffer(conv.M_bytes),
                "y": torch.empty(conv.y_shape, device="cuda")}
    n, h = case["n"], case["h"]
    x = _inputs(gen, n, 3, h, h)
    steps = []
    for block in TRUNK:
        for c, k in block:
            w, bias = _weights(gen, k, c, 3), _bias(gen, k)
            torch.cuda.synchronize()
            conv = _Conv(L, "auto", F.ConvShape(n, c, h, h, k, 3, 3, 1, 1, 1, 1, 1, 1), w, bias, True, False)
            steps.append((conv, torch.empty(conv.y_shape, device="cuda"), None))
        steps.append((None, torch.empty((n, k, h // 2, h // 2), device="cuda"), (n, k, h, h)))
        h //= 2
    L.sync()
    return {"steps": steps, "x": x, "V": _buffer(max(s[0].V_bytes for s in steps if s[0])),
            "M": _buffer(max(s[0].M_bytes for s in steps if s[0]))}


def run(state):
    if "conv" in state:
        state["conv"].forward(state["x"], state["V"], state["M"], state["y"])
        return state["y"]
    L, x = _library(), state["x"]
    for conv, y, pool in state["steps"]:
        if conv is None:
            L.maxpool2x2(_ptr(x), _ptr(y), *pool)
        else:
            conv.forward(x, state["V"], state["M"], y)
        x = y
    return x


def _layer_work(n, c, h, w, k, ks, stride, pad, winograd):
    oh, ow = (h + 2 * pad - ks) // stride + 1, (w + 2 * pad - ks) // stride + 1
    nbytes = 4.0 * (n * c * h * w + k * c * ks * ks + n * k * oh * ow)
    if winograd:      # the products of F(6x6,3x3)
        return nbytes, 2.0 * 64 * k * c * n * ((oh + 5) // 6) * ((ow + 5) // 6)
    return nbytes, 2.0 * n * k * c * oh * ow * ks * ks


def work(case):
    if case["algo"] != "trunk":
        winograd = case["algo"] != "im2col" and case["ks"] == 3 and case["stride"] == 1
        nbytes, flops = _layer_work(case["n"], case["c"], case["h"], case["w"], case["k"], case["ks"], case["stride"],
                                    case["pad"], winograd)
        return {"bytes": nbytes, "flops": flops}
    # x, the weights and the last pool's output once; the products of every layer
    n, h, nbytes, flops = case["n"], case["h"], 4.0 * case["n"] * 3 * case["h"] ** 2, 0.0
    for block in TRUNK:
        for c, k in block:
            flops += _layer_work(n, c, h, h, k, 3, 1, 1, True)[1]
            nbytes += 36.0 * c * k
        h //= 2
    return {"bytes": nbytes + 4.0 * n * TRUNK[-1][-1][1] * h * h, "flops": flops}


def tolerance(case):
    """Four times the largest difference of each path from the same convolution in 64 bits, over these cases and
    drawn ones: 2-norm 1.7e-6, 8.4e-6 and 3.7e-6, largest single value 1.1e-5, 1.7e-4 and 2.1e-5 (the trunk's last
    layers have few pixels; a smaller batch shows more)."""
    if case["algo"] == "im2col":
        return {"rel": 6e-6, "max": 5e-5}
    if case["algo"] == "trunk":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 3.5e-5, "max": 7e-4}


def _conv64(x, w, bias, relu, stride, pad):
    """The convolution as one product per window tap, summed in 64 bits."""
    x = torch.nn.functional.pad(x, (pad, pad, pad, pad))
    ks = w.shape[2]
    oh, ow = (x.shape[2] - ks) // stride + 1, (x.shape[3] - ks) // stride + 1
    y = torch.zeros((x.shape[0], w.shape[0], oh * ow), dtype=torch.float64, device=x.device)
    for image in range(x.shape[0]):
        for r in range(ks):
            for s in range(ks):
                tap = x[image, :, r:r + (oh - 1) * stride + 1:stride, s:s + (ow - 1) * stride + 1:stride]
                y[image].addmm_(w[:, :, r, s].contiguous(), tap.reshape(tap.shape[0], oh * ow))
    if bias is not None:
        y += bias[:, None]
    return (y.clamp_(min=0) if relu else y).view(x.shape[0], w.shape[0], oh, ow)


def exact(case, seed):
    """The outputs of run() in 64 bits, from the same draws of the generator as prepare()."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["algo"] != "trunk":
        x = _inputs(gen, case["n"], case["c"], case["h"], case["w"]).double()
        w = _weights(gen, case["k"], case["c"], case["ks"]).double()
        bias = _bias(gen, case["k"]).double() if case["bias_relu"] else None
        return _conv64(x, w, bias, case["bias_relu"], case["stride"], case["pad"])
    x = _inputs(gen, case["n"], 3, case["h"], case["h"]).double()
    for block in TRUNK:
        for c, k in block:
            w, bias = _weights(gen, k, c, 3).double(), _bias(gen, k).double()
            x = _conv64(x, w, bias, True, 1, 1)
        x = torch.nn.functional.max_pool2d(x, 2)
    return x
