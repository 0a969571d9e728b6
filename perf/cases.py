"""The work that users of butterfly_amd have it do, as measurable cases.

A case is one pass through the public entry points: a layer's forward call (inference), or its
forward call followed by autograd's backward for every parameter and the input (a training step
without the optimiser).  Five kinds:

* ``layer``: ``Butterfly`` as the drop-in for ``nn.Linear``, real or complex;
* ``base4``: ``ButterflyBase4``, the same layer with its stages stored in pairs;
* ``multiply``: the operators ``butterfly_multiply`` / ``butterfly_multiply_base4`` called directly;
* ``fft``: ``special.fft``, the Fourier transform as a (learnable) complex butterfly behind a bit reversal;
* ``circulant``: ``special.circulant``, a real circulant matrix as FFT, diagonal and inverse FFT.

Sizes: features 32 to 4096, rows 1 to 32768, with no more elements in a call than the widest
configuration of the benchmark (32768 rows of 4096).
"""
import math

import torch

import butterfly_amd
from butterfly_amd import special

DEVICE = "cuda"
MAX_ELEMENTS = 32768 * 4096


def listed():
    return [
        # one token or request through the widest layer (4096 -> 4096, B B^T): pure latency
        _layer("layer_4096_one_row", 4096, 4096, 1, nblocks=2, train=False),
        # a small training step on flattened images; neither size is a power of two
        _layer("layer_784_300_step", 784, 300, 50, nblocks=1),
        # the operator's forward call alone (benchmark configuration 1)
        _multiply("multiply_1024_forward", 10, 2048, increasing=True, train=False),
        # the headline workload (benchmark configuration 2)
        _multiply("multiply_1024_step", 10, 16384, nblocks=2, increasing=False),
        # a learnable Fourier transform at length 4096 (benchmark configuration 3)
        _fft("fft_4096_step", 4096, 8192),
        # base-4 factors, four independent stacks (benchmark configuration 4)
        _multiply("multiply_base4_256_step", 8, 16384, stacks=4, base=4),
        # the widest layer at its training batch (benchmark configuration 5): the largest case
        _layer("layer_4096_step", 4096, 4096, 32768, nblocks=2),
        # inputs narrower than the transform, zero padded by the layer, at the batch of the padding benchmark
        _layer("layer_400_512_step", 400, 512, 2048, nblocks=1, increasing=False),
        # more outputs than inputs: four stacks that share the input; ragged row count
        _layer("layer_256_1000_step", 256, 1000, 3001, nblocks=2),
        # spectra of a small batch of short signals
        _fft("fft_256_forward", 256, 100, train=False),
        # a learnable circular convolution of real signals, length not a power of two
        _circulant("circulant_1000_step", 1000, 512),
        # base-4 layer beyond one workgroup's row length, odd number of stages, B B^T
        _layer("base4_2000_2048_step", 2000, 2048, 1500, nblocks=2, kind="base4"),
    ]


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def rows(elements_per_row, nblocks=1, slow=False):
        # long schedules, complex and base-4 ones take more passes than the largest listed case
        weight = elements_per_row * max(2, nblocks) * (3 if slow else 2) // 4
        return spread(1, max(1, min(32768, MAX_ELEMENTS // weight)))

    def ceil2(v):
        return 1 << (v - 1).bit_length()

    kind = rng.choice(("layer",) * 5 + ("multiply",) * 3 + ("fft",) * 2 + ("base4",) * 2 + ("circulant",))
    train = rng.random() < 0.7
    if kind in ("layer", "base4"):
        in_size = spread(32, 4096)
        out_size = spread(16, 4096)
        if rng.random() < 0.4:   # the sizes that layers are most often given
            in_size, out_size = ceil2(in_size), ceil2(out_size)
        complex_ = kind == "layer" and rng.random() < 0.2
        n = ceil2(in_size)
        width = -(-out_size // n) * n * (2 if complex_ else 1)
        nblocks = rng.choice((1, 1, 2, 2, 2, 3))
        case = _layer(None, in_size, out_size, rows(width, nblocks, complex_ or kind == "base4"), nblocks=nblocks,
                      increasing=rng.random() < 0.5, complex_=complex_, bias=rng.random() < 0.75, train=train, kind=kind)
    elif kind == "multiply":
        log_n, stacks = rng.randint(5, 12), rng.choice((1, 1, 1, 2, 4))
        base = rng.choice((2, 2, 4))
        complex_ = base == 2 and rng.random() < 0.3
        width = stacks * (1 << log_n) * (2 if complex_ else 1)
        nblocks = rng.choice((1, 1, 2, 2, 2, 3))
        case = _multiply(None, log_n, rows(width, nblocks, complex_ or base == 4), stacks=stacks, nblocks=nblocks, base=base,
                         increasing=rng.random() < 0.5, complex_=complex_, train=train)
    elif kind == "fft":
        n = 1 << rng.randint(5, 12)
        case = _fft(None, n, rows(2 * n, slow=True), train=train)
    else:
        n = spread(32, 2048)
        # (sizes that are no power of two run embedded in twice the next one, as complex numbers,
        # through several modules)
        case = _circulant(None, n, rows(16 * ceil2(n)), train=train)
    del case["name"]
    return case


def _layer(name, in_size, out_size, batch, nblocks, increasing=True, complex_=False, bias=True, train=True, kind="layer"):
    return dict(name=name, kind=kind, in_size=in_size, out_size=out_size, batch=batch, nblocks=nblocks,
                increasing=increasing, complex=complex_, bias=bias, train=train)


def _multiply(name, log_n, batch, stacks=1, nblocks=1, base=2, increasing=True, complex_=False, train=True):
    return dict(name=name, kind="multiply", log_n=log_n, batch=batch, stacks=stacks, nblocks=nblocks, base=base,
                increasing=increasing, complex=complex_, train=train)


def _fft(name, n, batch, train=True):
    return dict(name=name, kind="fft", n=n, batch=batch, train=train)


def _circulant(name, n, batch, train=True):
    return dict(name=name, kind="circulant", n=n, batch=batch, train=train)


def _is_complex(case):
    return case["kind"] == "fft" or bool(case.get("complex"))


def prepare(case, seed):
    """The layer (or factors) and the rows, as a training or serving program holds them on the GPU."""
    torch.manual_seed(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = torch.complex64 if _is_complex(case) else torch.float32
    kind, train, batch = case["kind"], case["train"], case["batch"]

    def randn(*shape, scale=1.0):
        return torch.randn(*shape, dtype=dtype, device=DEVICE, generator=gen) * scale

    if kind == "multiply":
        L, S, nb = case["log_n"], case["stacks"], case["nblocks"]
        n = 1 << L
        # entries of variance 1/2 (1/4 for 4x4 factors): the outputs are as large as the inputs
        if case["base"] == 4:
            params = [randn(S, nb, L // 2, n // 4, 4, 4, scale=0.5), randn(S, nb, L % 2, n // 2, 2, 2, scale=0.5 ** 0.5)]
        else:
            params = [randn(S, nb, L, n // 2, 2, 2, scale=0.5 ** 0.5)]
        params = [p.requires_grad_(train) for p in params]
        op = butterfly_amd.butterfly_multiply_base4 if case["base"] == 4 else butterfly_amd.butterfly_multiply

        def call(x):
            return op(*params, x, case["increasing"])

        x, out_shape = randn(batch, S, n), (batch, S, n)
    else:
        if kind == "fft":
            n = case["n"]
            layer, sizes = special.fft(n, normalized=True), (n, n)
        elif kind == "circulant":
            n = case["n"]
            layer, sizes = special.circulant(torch.randn(n) / n ** 0.5), (n, n)
        else:
            make = butterfly_amd.Butterfly if kind == "layer" else butterfly_amd.ButterflyBase4
            sizes = (case["in_size"], case["out_size"])
            layer = make(*sizes, bias=case["bias"], complex=case["complex"], increasing_stride=case["increasing"],
                         init="ortho", nblocks=case["nblocks"])
        call = layer.to(DEVICE)
        params = list(layer.parameters())
        x, out_shape = randn(batch, sizes[0]), (batch, sizes[1])
    state = {"call": call, "x": x}
    if train:
        state["x"] = x.requires_grad_()
        # (base-4 factors of an even number of stages come with an empty tensor of 2x2 ones)
        state["wanted"] = [state["x"]] + [p for p in params if p.numel() > 0]
        state["grad"] = randn(*out_shape)
    return state


def run(state):
    if "grad" not in state:
        with torch.no_grad():
            return state["call"](state["x"])
    y = state["call"](state["x"])
    return [y.detach(), *torch.autograd.grad(y, state["wanted"], state["grad"])]


def work(case):
    """Bytes: each call's operands once -- forward: rows in, rows out, factors; backward: rows,
    output gradient, factors in, input gradient and factor gradients out.  Flops: a 2x2 stage is
    two multiply-adds an element (a 4x4 stage, which stands for two, four), in the forward sweep,
    the replay, the input gradient and the factor gradient."""
    kind, batch = case["kind"], case["batch"]
    if kind == "multiply":
        L, S, nb = case["log_n"], case["stacks"], case["nblocks"]
        layers, row_in, row_out = [(L, S, nb, case["base"])], S << L, S << L
    elif kind == "fft":
        L = case["n"].bit_length() - 1
        layers, row_in, row_out = [(L, 1, 1, 2)], case["n"], case["n"]
    elif kind == "circulant":
        n = case["n"]
        up = (n - 1).bit_length()
        L = up if n == 1 << up else up + 1
        layers, row_in, row_out = [(L, 1, 1, 2)] * 2, n, n
    else:
        L = (case["in_size"] - 1).bit_length()
        S = -(-case["out_size"] >> L)
        layers = [(L, S, case["nblocks"], 4 if kind == "base4" else 2)]
        row_in, row_out = case["in_size"], case["out_size"]
    elem = 8 if _is_complex(case) else 4
    factor_elem = 8 if kind == "circulant" else elem
    factors = sum(S * nb * ((L // 2) * 4 + (L % 2) * 2 if base == 4 else L * 2) << L for L, S, nb, base in layers) * factor_elem
    sweep = sum((S * nb * L << L) * 4 for L, S, nb, base in layers) * batch * (4 if factor_elem == 8 else 1)
    if not case["train"]:
        return {"bytes": batch * (row_in + row_out) * elem + factors, "flops": sweep}
    return {"bytes": batch * (3 * row_in + 2 * row_out) * elem + 3 * factors, "flops": 4 * sweep}


def tolerance(case):
    # float32 throughout: some 24 stages of multiply-adds, and sums over up to 32768 rows
    return {"rel": 1e-5}
