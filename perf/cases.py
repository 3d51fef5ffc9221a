"""The work that a user of this package has it do, as cases that can be timed.

Two kinds of work, both through the package's public entry points:

  * training steps: an executor (``TrainExecute`` / ``TrainExecuteAdam``) is built once
    for one of the networks of ``tinyflow_amd.models`` and then called with one batch
    of host data per step, which is what the package exists for;
  * single operators through ``gpu_op`` on device arrays, for callers who bring their own
    graph: a convolution or a matrix product, each with its forward pass and both of
    its gradients.

A case is a dict of plain values; ``prepare`` makes what the program holds before the
call, ``run`` is one pass.
"""
import math
import random

import numpy as np
import torch

from tinyflow_amd import TrainExecute, TrainExecuteAdam, gpu_op, models, ndarray

# ------------------------------------------------------------------------------ the cases


def _step(name, net, batch, image=0, optimizer="sgd", head="softmax_xent", bn_mode="pre_activation", fused=False):
    return {"name": name, "kind": "step", "net": net, "batch": batch, "image": image, "optimizer": optimizer,
            "head": head, "bn_mode": bn_mode, "fused": fused}


def _conv(name, n, c, h, w, k, r, padding, stride):
    return {"name": name, "kind": "conv", "n": n, "c": c, "h": h, "w": w, "k": k, "r": r, "padding": padding,
            "stride": stride}


def _matmul(name, m, k, n):
    return {"name": name, "kind": "matmul", "m": m, "k": k, "n": n}


def listed():
    return [
        # the smallest training step of the benchmark's configurations: a few hundred microseconds in
        # which launches and host work are everything
        _step("mlp b128", "mlp", 128),
        # the small convolutional network at its benchmark batch ...
        _step("lenet5 b64", "lenet5", 64),
        # ... and as a user runs it who wants throughput from it: a large ragged batch, Adam, the
        # batch-norm / softmax / cross-entropy head of the model scripts
        _step("lenet5 b1000 adam", "lenet5", 1000, optimizer="adam", head="cross"),
        # the plain deep network at its benchmark batch: large maps, large fully connected layers
        _step("vgg16 b32", "vgg16", 32, 224),
        # the model script's form of it (dropout, cross head, Adam) at a small batch and image, where
        # the 138 M-parameter classifier shrinks and the deep maps are 3 x 3 and 6 x 6
        _step("vgg16 script b6 96px", "vgg16", 6, 96, optimizer="adam", head="cross"),
        # the headline workload
        _step("resnet50 b64", "resnet50", 64, 224),
        # the executor's fusion option at half that batch
        _step("resnet50 b32 fused", "resnet50", 32, 224, fused=True),
        # spatial batch norm, a small batch and an image whose maps are odd (5 x 5 ... 40 x 40)
        _step("resnet50 b8 160px spatial", "resnet50", 8, 160, bn_mode="spatial"),
        # single layers: a padded 3 x 3 on the odd 55 x 55 maps, a strided unpadded 5 x 5 with ragged
        # channel counts, a matrix product with no round extent and a fully connected layer
        _conv("conv 3x3 55px", 32, 64, 55, 55, 64, 3, "SAME", 1),
        _conv("conv 5x5 stride 2 ragged", 20, 50, 61, 59, 70, 5, "VALID", 2),
        _matmul("matmul 1000x1537x777", 1000, 1537, 777),
        _matmul("matmul 32x25088x4096", 32, 25088, 4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: batches from one sample to the listed sizes and beyond for the
    small networks, images of any multiple of 32 up to 224 pixels (what the networks' five halvings ask
    for), layers and matrices of any extent."""
    kind = rng.choice(["mlp", "lenet5", "vgg16", "resnet50", "resnet50", "conv", "conv", "matmul"])
    if kind == "mlp":
        case = _step("", "mlp", _log_int(rng, 1, 8192), optimizer=rng.choice(["sgd", "adam"]))
    elif kind == "lenet5":
        head = rng.choice(["softmax_xent", "cross"])
        case = _step("", "lenet5", _log_int(rng, 4, 4096), optimizer=rng.choice(["sgd", "adam"]), head=head)
    elif kind == "vgg16":
        image = 32 * rng.randint(1, 7)
        most = min(256, 32 * 224 * 224 // image ** 2)
        head = rng.choice(["softmax_xent", "cross"])
        case = _step("", "vgg16", _log_int(rng, 2, most), image, optimizer="adam" if head == "cross" else "sgd", head=head)
    elif kind == "resnet50":
        bn_mode = rng.choice(["pre_activation", "spatial"])
        # a per-activation statistic is taken over the batch alone: nobody trains that on a few samples,
        # and on the 2 x 2 maps of small images it is as good as random
        image = 32 * rng.randint(2 if bn_mode == "spatial" else 4, 7)
        most = min(128, 64 * 224 * 224 // image ** 2)
        batch = _log_int(rng, 4 if bn_mode == "spatial" else 32, most)
        case = _step("", "resnet50", batch, image, bn_mode=bn_mode,
                     fused=bn_mode == "pre_activation" and rng.random() < 0.5)
    elif kind == "conv":
        r = rng.choice([1, 1, 3, 3, 3, 5, 7])
        c, k = _log_int(rng, 3, 512), _log_int(rng, 8, 512)
        h = _log_int(rng, max(7, r), 112)
        w = h if rng.random() < 0.7 else _log_int(rng, max(7, r), 112)
        stride = rng.choice([1, 1, 2])
        # up to about 200 GFLOP and 100 MB a tensor
        most = min(128, 1e11 / (2.0 * c * k * r * r * h * w), 25e6 / (max(c, k) * h * w))
        n = _log_int(rng, 1, max(1, int(most)))
        case = _conv("", n, c, h, w, k, r, rng.choice(["SAME", "VALID"]) if r > 1 else "VALID", stride)
    else:
        case = _matmul("", _log_int(rng, 1, 4096), _log_int(rng, 16, 8192), _log_int(rng, 8, 4096))
    del case["name"]
    return case


# ------------------------------------------------------------------------------- preparing

class _DeviceView(object):
    """A device array of the library as torch sees foreign device memory."""

    def __init__(self, arr):
        self.__cuda_array_interface__ = {"shape": arr.shape, "typestr": "<f4", "version": 2,
                                         "data": (arr.handle.contents.data, False)}


def _as_tensor(arr):
    return torch.as_tensor(_DeviceView(arr), device="cuda")


def _network(case, rng):
    net, batch = case["net"], case["batch"]
    if net == "mlp":
        return models.mlp(rng, batch=batch, head=case["head"])
    if net == "lenet5":
        return models.lenet5(rng, batch=batch, head=case["head"])
    if net == "vgg16":  # the script's head comes with its dropout
        return models.vgg16(rng, batch=batch, image=case["image"], head=case["head"],
                            dropout=0.5 if case["head"] == "cross" else None)
    return models.resnet50(rng, batch=batch, image=case["image"], bn_mode=case["bn_mode"])


def _learning_rate(case):
    """Small enough that thousands of steps on one batch stay finite and that the third step of two correct
    implementations is still the same step (the gradient is a sum over the batch, and the deep networks
    multiply a difference between two parameter sets by about ten per step at rates ten times these)."""
    if case["optimizer"] == "adam":
        return {"mlp": 1e-4, "lenet5": 1e-4, "vgg16": 1e-6}[case["net"]]
    return {"mlp": 1e-4, "lenet5": 1e-4, "vgg16": 1e-7, "resnet50": 3e-7}[case["net"]]


def _prepare_step(case, seed):
    rng = np.random.default_rng(seed)
    random.seed(seed)  # dropout draws its seeds from Python's generator
    model = _network(case, rng)
    shape = model.input_shape
    if case["net"] in ("mlp", "lenet5"):
        X = rng.random(shape, dtype=np.float32)
    else:
        X = rng.standard_normal(shape, dtype=np.float32)
    y = np.zeros((shape[0], model.n_class), np.float32)
    y[np.arange(shape[0]), rng.integers(0, model.n_class, shape[0])] = 1.0
    lr = _learning_rate(case)
    if case["optimizer"] == "adam":
        executor = TrainExecuteAdam.TrainExecutor(model.loss, lr, fuse_bn_relu=case["fused"])
    else:
        executor = TrainExecute.TrainExecutor(model.loss, lr, fuse_bn_relu=case["fused"])
    executor.init_Variable(dict(model.variables))
    feed = {model.X: X, model.y_: y}
    # the first step plans and allocates; a training program is past it
    result = executor.run(feed)
    gradients = {v.name: executor.value_of(g)
                 for v, g in zip(executor.Variable_node_list, executor.Variable_node_grad_list)}
    parameters = {v.name: executor.value_of(v) for v in executor.Variable_node_list}
    if case["head"] == "cross":
        # the bias under the head's batch norm has no gradient: what is computed for it, and what
        # Adam makes of that, is rounding
        last = {"mlp": "fc3_b", "lenet5": "fc5_b", "vgg16": "fc8_b"}[case["net"]]
        del gradients[last], parameters[last]
    outputs = {"loss": result[0], "logits": executor.value_of(model.logits)}
    outputs.update(("updated " + name, a) for name, a in parameters.items())
    if case["net"] == "resnet50":  # 55 parameters; of the gradients those above its batch norms, see tolerance()
        gradients = {name: gradients[name] for name in ("fc_W", "fc_b")}
    outputs.update(("gradient " + name, a) for name, a in gradients.items())
    outputs = {name: _as_tensor(a) for name, a in outputs.items()}
    return {"kind": "step", "executor": executor, "feed": feed, "outputs": outputs}


_stream = None


def _op_stream():
    """The one stream and handle pair of a program that calls operators itself."""
    global _stream
    if _stream is None:
        stream = gpu_op.create_cudaStream()
        _stream = (stream, gpu_op.create_cudnnHandle(stream), gpu_op.create_cublasHandle(stream))
    return _stream


def _device_array(values):
    return ndarray.array(values, ctx=ndarray.gpu(0))


def _prepare_conv(case, seed):
    rng = np.random.default_rng(seed)
    x_shape = (case["n"], case["c"], case["h"], case["w"])
    w_shape = (case["k"], case["c"], case["r"], case["r"])
    y_shape, desc = gpu_op.convolution_2d_forward_get_out_shape(x_shape, w_shape, "NCHW", case["padding"],
                                                                case["stride"], case["stride"])
    # what a layer meets: activations behind a ReLU, He-scaled filters, gradients of either sign
    x = np.maximum(rng.standard_normal(x_shape, dtype=np.float32), 0)
    w = rng.standard_normal(w_shape, dtype=np.float32) * np.float32(math.sqrt(2.0 / (case["c"] * case["r"] ** 2)))
    dy = rng.standard_normal(y_shape, dtype=np.float32)
    x, w, dy = _device_array(x), _device_array(w), _device_array(dy)
    y, dx, dw = (ndarray.empty(s, ctx=ndarray.gpu(0)) for s in (y_shape, x_shape, w_shape))
    return {"kind": "conv", "desc": desc, "arrays": (x, w, dy, y, dx, dw), "stream": _op_stream(),
            "outputs": [_as_tensor(a) for a in (y, dx, dw)]}


def _prepare_matmul(case, seed):
    rng = np.random.default_rng(seed)
    m, k, n = case["m"], case["k"], case["n"]
    a = np.maximum(rng.standard_normal((m, k), dtype=np.float32), 0)
    b = rng.standard_normal((k, n), dtype=np.float32) * np.float32(math.sqrt(2.0 / k))
    dc = rng.standard_normal((m, n), dtype=np.float32)
    a, b, dc = _device_array(a), _device_array(b), _device_array(dc)
    c, da, db = (ndarray.empty(s, ctx=ndarray.gpu(0)) for s in ((m, n), (m, k), (k, n)))
    return {"kind": "matmul", "arrays": (a, b, dc, c, da, db), "stream": _op_stream(),
            "outputs": [_as_tensor(t) for t in (c, da, db)]}


def prepare(case, seed):
    return {"step": _prepare_step, "conv": _prepare_conv, "matmul": _prepare_matmul}[case["kind"]](case, seed)


# --------------------------------------------------------------------------------- running

def run(state):
    if state["kind"] == "step":
        state["executor"].run(state["feed"])
        return state["outputs"]
    stream, cudnn, cublas = state["stream"]
    if state["kind"] == "conv":
        x, w, dy, y, dx, dw = state["arrays"]
        desc = state["desc"]
        wanted = gpu_op.convolution_2d_forward(x, w, y, desc, cudnn, stream)
        wanted += gpu_op.convolution_backward_data(x, dy, w, dx, desc, cudnn, stream)
        wanted += gpu_op.convolution_backward_filter(x, dy, w, dw, desc, cudnn, stream)
        if wanted:
            raise MemoryError("%d bytes of device scratch could not be had" % wanted)
    else:
        a, b, dc, c, da, db = state["arrays"]
        gpu_op.matrix_multiply(a, False, b, False, c, cublas, stream)
        gpu_op.matrix_multiply(dc, False, b, True, da, cublas, stream)
        gpu_op.matrix_multiply(a, True, dc, False, db, cublas, stream)
    return state["outputs"]


# ---------------------------------------------------------------------- what it has to cost

def _resnet50_layers(image):
    """(C, H, K, R, stride) of every convolution, and the classifier's width."""
    layers = [(3, image, 64, 7, 2)]
    size, in_ch = image // 4, 64
    for stage, count in enumerate([3, 4, 6, 3]):
        f = 64 * 2 ** stage
        for i in range(count):
            stride = 2 if i == 0 and stage > 0 else 1
            if i == 0:
                layers.append((in_ch, size, 4 * f, 1, stride))
            layers.append((in_ch, size, f, 1, stride))
            size //= stride
            layers.append((f, size, f, 3, 1))
            layers.append((f, size, 4 * f, 1, 1))
            in_ch = 4 * f
    return layers, [(2048, 1000)]


def _layers(case):
    """Convolutions as (C, H, K, R, stride) and dense layers as (inputs, outputs) of a network."""
    if case["net"] == "mlp":
        return [], [(784, 256), (256, 100), (100, 10)]
    if case["net"] == "lenet5":
        return [(1, 28, 6, 5, 1), (6, 10, 16, 5, 1)], [(400, 120), (120, 84), (84, 10)]
    if case["net"] == "resnet50":
        return _resnet50_layers(case["image"])
    convs, size, in_ch = [], case["image"], 3
    for widths in models.VGG16_CHANNELS:
        for k in widths:
            convs.append((in_ch, size, k, 3, 1))
            in_ch = k
        size //= 2
    return convs, [(in_ch * size * size, 4096), (4096, 4096), (4096, 1000)]


def work(case):
    """Every product's multiply-adds, in each direction; parameters (and moments) read and written once,
    the batch read once, every layer's output written in the forward pass and read in the backward
    pass, its gradient likewise."""
    if case["kind"] == "conv":
        pad = case["r"] // 2 if case["padding"] == "SAME" else 0
        p = (case["h"] + 2 * pad - case["r"]) // case["stride"] + 1
        q = (case["w"] + 2 * pad - case["r"]) // case["stride"] + 1
        macs = case["n"] * case["k"] * p * q * case["c"] * case["r"] ** 2
        x = case["n"] * case["c"] * case["h"] * case["w"]
        w = case["k"] * case["c"] * case["r"] ** 2
        y = case["n"] * case["k"] * p * q
        return {"bytes": 8 * (x + w + y), "flops": 6 * macs}
    if case["kind"] == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": 8 * (m * k + k * n + m * n), "flops": 6 * m * k * n}
    convs, dense = _layers(case)
    batch = case["batch"]
    flops = params = values = 0
    for i, (c, h, k, r, stride) in enumerate(convs):
        p = h // stride
        macs = batch * k * p * p * c * r * r
        flops += (4 if i == 0 else 6) * macs  # nobody asks for the gradient of the images
        params += k * c * r * r
        values += batch * k * p * p
    for i, (rows, cols) in enumerate(dense):
        flops += (4 if i == 0 and not convs else 6) * batch * rows * cols
        params += rows * cols + cols
        values += batch * cols
    side = {"mlp": 784, "lenet5": 784}.get(case["net"], 3 * case["image"] ** 2)
    state = 6 if case["optimizer"] == "adam" else 2
    return {"bytes": 4 * (batch * side + state * params + 4 * values), "flops": flops}


def tolerance(case):
    """Measured by running the same tree with its sums in other orders (direct and transformed-domain
    convolutions, with and without k-splits), the small networks against float64 on the CPU.

    Single operators differ by 1.5e-6 at most.  In a network a ReLU or a max-pool whose input lies within
    rounding of its threshold decides one way or the other, and one such decision moves the gradients below
    it by up to 4e-3 (MLP, LeNet-5) or 7e-3 (VGG-16, where several do); logits and parameters alone stay
    within 1e-6.  The ResNets' gradients below a batch norm differ by 3e-2 to 1e-1 between any two fp32
    evaluations at random weights, so they are seen through the updated parameters and through the logits
    that the next step computes from those: 2.3e-3 after three steps."""
    if case["kind"] != "step":
        return {"rel": 1e-5, "max": 1e-3}
    return {"mlp": {"rel": 0.02, "max": 0.5}, "lenet5": {"rel": 0.02, "max": 0.5},
            "vgg16": {"rel": 0.03, "max": 0.99}, "resnet50": {"rel": 0.01, "max": 0.1}}[case["net"]]
