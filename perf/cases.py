"""The work this framework is used for, as measurable cases.

Every case is one call (or, for attention training, a forward and its backward)
of the tensor front end `jules_amd.ops`, at sizes of this repository's own
benchmark and tests or at generic ones: fused GEMMs in fp32 and bf16, attention
forward and backward, the quantised GEMMs of decoding and prefill, the row
kernels, and the two-layer training step.  `listed` gives a fixed dozen, `draw`
any number of others from the same ranges, odd and ragged sizes included.
"""
import math

import torch

from jules_amd import ops

DEV = "cuda:0"
ACTS = ("none", "relu", "sigmoid", "tanh", "gelu", "silu")


def listed():
    return [
        # fp32 layer with its tanh-approximated GELU, the smallest of the
        # benchmark's configurations: launch and latency count
        dict(name="gemm_f32_512", kind="gemm", dtype="f32", M=512, N=512, K=512, act="gelu",
             bias=True),
        # an fp32 layer over a batch that is no multiple of a tile
        dict(name="gemm_f32_batch", kind="gemm", dtype="f32", M=2000, N=3072, K=1024, act="relu",
             bias=True),
        # the compute-bound bf16 layer of the benchmark
        dict(name="gemm_bf16_4096", kind="gemm", dtype="bf16", M=4096, N=4096, K=4096, act="gelu",
             bias=True),
        # the same layer over one prompt: few, ragged rows
        dict(name="gemm_bf16_prompt", kind="gemm", dtype="bf16", M=328, N=4096, K=4096, act="silu",
             bias=True),
        # fp32 attention of the benchmark
        dict(name="flash_f32_1024", kind="flash", dtype="f32", B=4, H=8, S=1024, D=64, causal=True),
        # bf16 attention of the benchmark: a batch of long sequences
        dict(name="flash_bf16_4096", kind="flash", dtype="bf16", B=8, H=32, S=4096, D=128,
             causal=True),
        # an encoder's attention: short ragged sequence, a head size between
        # the two the kernels are built for
        dict(name="flash_bf16_333", kind="flash", dtype="bf16", B=2, H=16, S=333, D=80,
             causal=False),
        # attention of a training step, forward and backward
        dict(name="flash_train_2048", kind="flash_train", B=4, H=16, S=2048, D=128, causal=True),
        # one decoding step of a weight-quantised layer (row-major weights)
        dict(name="w8a16_decode", kind="w8a16", packed=False, M=8, N=8192, K=8192, act="silu",
             bias=True),
        # the same quantisation at prefill, int8 activations, ragged rows
        dict(name="w8a8_prefill", kind="int8", per_token=True, M=500, N=4096, K=4096, bias=True),
        # the training step of a small classifier: all its launches, little work
        dict(name="mlp_train_64", kind="mlp", backward=True, M=64, K1=784, N1=256, N2=10, dX=False),
        # a language model's loss and logit gradient
        dict(name="xent_50257", kind="xent", M=2048, N=50257),
    ]


def _log(rng, lo, hi, multiple=1):
    """A size in [lo, hi], spread over its logarithm, a multiple of `multiple`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))
    return max(multiple, min(hi, int(v)) // multiple * multiple)


def draw(rng):
    kind = rng.choice(("gemm_f32", "gemm_bf16", "flash", "flash_train", "w8a16", "int8", "rows",
                       "mlp", "activation"))
    if kind == "gemm_f32":
        while True:
            M, N, K = _log(rng, 8, 4096), _log(rng, 8, 4096), _log(rng, 16, 4096)
            if M * N * K <= 2 ** 33:
                break
        return dict(kind="gemm", dtype="f32", M=M, N=N, K=K, act=rng.choice(ACTS),
                    bias=rng.random() < 0.75)
    if kind == "gemm_bf16":
        return dict(kind="gemm", dtype="bf16", M=_log(rng, 24, 4096, 8),
                    N=_log(rng, 256, 8192, rng.choice((8, 8, 64, 256))),
                    K=_log(rng, 256, 8192, rng.choice((8, 8, 64, 256))), act=rng.choice(ACTS),
                    bias=rng.random() < 0.75)
    if kind in ("flash", "flash_train"):
        bf16 = kind == "flash_train" or rng.random() < 0.7
        D = rng.choice((64, 64, 128, 128, 128, 32, 80, 96))
        while True:
            B, H, S = _log(rng, 1, 8), _log(rng, 1, 32), _log(rng, 16, 4096)
            if B * H * S * S * D <= (2 ** 38 if bf16 else 2 ** 34):
                break
        c = dict(kind=kind, B=B, H=H, S=S, D=D, causal=rng.random() < 0.6)
        if kind == "flash":
            c["dtype"] = "bf16" if bf16 else "f32"
        return c
    if kind == "w8a16":
        return dict(kind="w8a16", packed=rng.random() < 0.5, M=rng.randint(1, 16),
                    N=_log(rng, 512, 16384, 16), K=_log(rng, 512, 8192, 8), act=rng.choice(ACTS),
                    bias=rng.random() < 0.75)
    if kind == "int8":
        # mostly rows of whole 16-byte pieces, now and then any size
        m = 1 if rng.random() < 0.2 else 16
        hi = 1024 if m == 1 else 8192
        return dict(kind="int8", per_token=rng.random() < 0.5, M=_log(rng, 1, 4096 if m > 1 else 512),
                    N=_log(rng, 256, hi, m), K=_log(rng, 256, hi, m), bias=rng.random() < 0.5)
    if kind == "rows":
        kind = rng.choice(("softmax", "layernorm", "xent", "xent"))
        while True:
            M, N = _log(rng, 1, 16384), _log(rng, 16, 131072)
            if M * N <= 2 ** 27:
                break
        return dict(kind=kind, M=M, N=N)
    if kind == "mlp":
        while True:
            M, K1, N1 = _log(rng, 16, 8192), _log(rng, 32, 4096), _log(rng, 32, 4096)
            N2 = _log(rng, 4, 1024)
            if M * N1 * (K1 + N2) <= 2 ** 33:
                break
        return dict(kind="mlp", backward=rng.random() < 0.7, M=M, K1=K1, N1=N1, N2=N2,
                    dX=rng.random() < 0.5)
    return dict(kind="activation", act=rng.choice(ACTS[1:]), n=_log(rng, 1000, 2 ** 24))


# --- inputs -----------------------------------------------------------------

def _inputs(case, seed):
    """The case's tensors, from the seed alone, in the order the call takes them.

    fp32 GEMM operands are uniform in [-1, 1]; bf16 ones normal with deviation
    1/sqrt(K); attention's normal; int8 weights uniform in [-127, 127] with
    per-channel scales in [1e-3, 1e-2]; logits and row inputs normal; the
    training step's uniform, weights divided by about sqrt(fan in)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)

    def uni(shape, lo=-1.0, hi=1.0):
        return torch.rand(shape, generator=g, device=DEV).mul_(hi - lo).add_(lo)

    def nrm(shape, std=1.0):
        return torch.randn(shape, generator=g, device=DEV).mul_(std)

    def i8(shape):
        return torch.randint(-127, 128, shape, generator=g, device=DEV, dtype=torch.int8)

    k = case["kind"]
    if k == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        if case["dtype"] == "f32":
            A, B, b = uni((M, K)), uni((K, N)), uni((N,))
        else:
            std = 1.0 / math.sqrt(K)
            A, B = nrm((M, K), std).bfloat16(), nrm((K, N), std).bfloat16()
            b = uni((N,), -0.1, 0.1)
        return dict(A=A, B=B, bias=b if case["bias"] else None)
    if k in ("flash", "flash_train"):
        dt = torch.float32 if case.get("dtype") == "f32" else torch.bfloat16
        shape = (case["B"], case["H"], case["S"], case["D"])
        t = {n: nrm(shape).to(dt) for n in ("Q", "K", "V")}
        if k == "flash_train":
            t["dO"] = nrm(shape).to(dt)
        return t
    if k == "w8a16":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(x=nrm((M, K)).bfloat16(), W=i8((K, N)), scale=uni((N,), 1e-3, 1e-2),
                    bias=uni((N,), -0.1, 0.1) if case["bias"] else None)
    if k == "int8":
        M, N, K = case["M"], case["N"], case["K"]
        return dict(A=i8((M, K)), B=i8((K, N)), sa=uni((M,), 1e-3, 1e-2), sb=uni((N,), 1e-3, 1e-2),
                    bias=uni((N,)) if case["bias"] else None)
    if k == "mlp":
        M, K1, N1, N2 = case["M"], case["K1"], case["N1"], case["N2"]
        # X, W1 and b1 lie on a grid (like pixels and weights stored in fixed
        # point) on which the hidden layer's sums are exact: a hidden value
        # within rounding of 0 would otherwise pass the ReLU in one order of
        # summation and not in another, and move dW1 by 1e-4 and more
        fan = 2.0 ** round(math.log2(K1) / 2)
        t = dict(X=uni((M, K1)).mul_(64).round_().div_(64),
                 W1=uni((K1, N1)).mul_(512).round_().div_(512 * fan),
                 b1=uni((N1,)).mul_(64).round_().div_(64),
                 W2=uni((N1, N2)).div_(math.sqrt(N1)), b2=uni((N2,)))
        t["targets"] = torch.randint(0, N2, (M,), generator=g, device=DEV, dtype=torch.int32)
        return t
    if k == "activation":
        return dict(x=nrm((case["n"],)))
    M, N = case["M"], case["N"]
    t = dict(x=nrm((M, N)))
    if k == "layernorm":
        t.update(gamma=uni((N,), 0.5, 1.5), beta=uni((N,)))
    if k == "xent":
        t["targets"] = torch.randint(0, N, (M,), generator=g, device=DEV, dtype=torch.int32)
    return t


def prepare(case, seed):
    """The tensors, and what a program keeps between its calls: repacked
    weights, workspaces, the training step's output buffers."""
    s = dict(case=case, **_inputs(case, seed))
    k = case["kind"]
    if k == "w8a16" and case["packed"]:
        s["packed"] = ops.w8a16_pack(s.pop("W"))
    elif k == "w8a16":
        s["workspace"] = ops.w8a16_workspace(case["M"], case["N"], case["K"], DEV)
    elif k == "xent":
        s["workspace"] = ops.cross_entropy_workspace(case["M"], DEV)
    elif k == "mlp" and case["backward"]:
        M, K1, N1, N2 = case["M"], case["K1"], case["N1"], case["N2"]
        s["workspace"] = ops.mlp_workspace(M, K1, N1, N2, DEV)

        def buf(*shape):
            return torch.empty(shape, dtype=torch.float32, device=DEV)

        s["out"] = dict(output=buf(M, N2), loss=buf(1), dW1=buf(K1, N1), db1=buf(N1),
                        dW2=buf(N1, N2), db2=buf(N2), dX=buf(M, K1) if case["dX"] else None)
    return s


def run(state):
    c = state["case"]
    k = c["kind"]
    if k == "gemm":
        return ops.gemm_bias_act(state["A"], state["B"], state["bias"], c["act"])
    if k == "flash":
        return ops.flash_attention(state["Q"], state["K"], state["V"], causal=c["causal"])
    if k == "flash_train":
        Q, K, V = state["Q"], state["K"], state["V"]
        lse = torch.empty(Q.shape[:3], dtype=torch.float32, device=Q.device)
        O = ops.flash_attention(Q, K, V, causal=c["causal"], lse=lse)
        dQ, dK, dV = ops.flash_attention_bwd(Q, K, V, O, state["dO"], lse, causal=c["causal"])
        return dict(O=O, lse=lse, dQ=dQ, dK=dK, dV=dV)
    if k == "w8a16" and c["packed"]:
        return ops.w8a16_gemm_packed(state["x"], state["packed"], state["scale"], state["bias"],
                                     c["act"])
    if k == "w8a16":
        return ops.w8a16_gemm(state["x"], state["W"], state["scale"], state["bias"], c["act"],
                              workspace=state["workspace"])
    if k == "int8":
        if c["per_token"]:
            return ops.matmul_w8a8(state["A"], state["B"], state["sa"], state["sb"], state["bias"])
        return ops.matmul_int8(state["A"], state["B"], 0.013, 0.021, state["bias"])
    if k == "softmax":
        return ops.softmax(state["x"])
    if k == "layernorm":
        return ops.layernorm(state["x"], state["gamma"], state["beta"])
    if k == "xent":
        loss, grad = ops.cross_entropy(state["x"], state["targets"], workspace=state["workspace"])
        return dict(loss=loss, grad=grad)
    if k == "mlp":
        args = [state[n] for n in ("X", "W1", "b1", "W2", "b2")]
        if not c["backward"]:
            return ops.mlp_forward(*args)
        out = ops.mlp_forward_backward(*args, state["targets"], with_dX=c["dX"],
                                       workspace=state["workspace"], out=state["out"])
        return {n: t for n, t in out.items() if t is not None}
    return ops.activation(state["x"], c["act"])


def work(case):
    """Bytes of every input once and every output once, and the algorithm's
    operations (attention's causal half only; its backward 2.5 times its
    forward)."""
    k = case["kind"]
    if k == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        es = 4 if case["dtype"] == "f32" else 2
        return {"bytes": es * (M * K + K * N + M * N) + (4 * N if case["bias"] else 0),
                "flops": 2 * M * N * K}
    if k in ("flash", "flash_train"):
        B, H, S, D = case["B"], case["H"], case["S"], case["D"]
        n = B * H * S * D
        pairs = S * (S + 1) // 2 if case["causal"] else S * S
        f = 4 * B * H * D * pairs
        if k == "flash_train":
            # Q, K, V, dO in; O, dQ, dK, dV and the log-sum-exp out
            return {"bytes": 16 * n + 4 * B * H * S, "flops": f * 7 // 2}
        return {"bytes": 4 * n * (4 if case["dtype"] == "f32" else 2), "flops": f}
    if k == "w8a16":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": K * N + (8 if case["bias"] else 4) * N + 2 * M * K + 2 * M * N,
                "flops": 2 * M * N * K}
    if k == "int8":
        M, N, K = case["M"], case["N"], case["K"]
        extra = (4 * N if case["bias"] else 0) + (4 * (M + N) if case["per_token"] else 0)
        return {"bytes": M * K + K * N + 4 * M * N + extra, "flops": 2 * M * N * K}
    if k == "mlp":
        M, K1, N1, N2 = case["M"], case["K1"], case["N1"], case["N2"]
        weights = K1 * N1 + N1 + N1 * N2 + N2
        fwd = 2 * M * N1 * (K1 + N2)
        if not case["backward"]:
            return {"bytes": 4 * (M * K1 + weights + M * N2), "flops": fwd}
        # dW2, dA, dW1 and, when asked for, dX
        bwd = 2 * M * N1 * (2 * N2 + K1 + (K1 if case["dX"] else 0))
        return {"bytes": 4 * (M * K1 * (2 if case["dX"] else 1) + 2 * weights + M * N2 + M + 1),
                "flops": fwd + bwd}
    if k == "activation":
        return {"bytes": 8 * case["n"], "flops": 20 * case["n"]}
    M, N = case["M"], case["N"]
    extra = {"softmax": 0, "layernorm": 8 * N, "xent": 4 * M + 4}[k]
    return {"bytes": 8 * M * N + extra, "flops": 10 * M * N}


def tolerance(case):
    """Relative 2-norm differences, four times what the kernels show against
    64-bit results, rounded up."""
    k = case["kind"]
    if k in ("gemm", "flash") and case["dtype"] == "f32":
        # sums of K products each rounded to fp32; tanh and sigmoid on the
        # reference's degree-6 exponential
        return {"rel": 7e-6 if k == "gemm" else 2e-6}
    if k in ("gemm", "w8a16"):
        return {"rel": 7e-3}
    if k in ("flash", "flash_train"):
        # bf16 probabilities as well as bf16 results
        return {"rel": 1e-2}
    return {"rel": {"int8": 2.5e-7, "softmax": 1.5e-5, "layernorm": 5e-7, "xent": 3e-6,
                    "mlp": 1.5e-5, "activation": 1.2e-5}[k]}


# --- 64-bit results ---------------------------------------------------------

def _act64(v, act):
    if act == "relu":
        return v.clamp_min(0.0)
    if act == "sigmoid":
        return torch.sigmoid(v)
    if act == "tanh":
        return torch.tanh(v)
    if act == "gelu":
        return torch.nn.functional.gelu(v, approximate="tanh")
    if act == "silu":
        return torch.nn.functional.silu(v)
    return v


def _attention64(t, case):
    """Attention (and its gradients when `dO` is there), one head at a time."""
    B, H, S, D = case["B"], case["H"], case["S"], case["D"]
    scale = 1.0 / math.sqrt(D)
    train = "dO" in t
    names = ("O", "dQ", "dK", "dV") if train else ("O",)
    out = {n: torch.empty((B * H, S, D), dtype=torch.float64, device=DEV) for n in names}
    lse = torch.empty((B * H, S), dtype=torch.float64, device=DEV)
    hidden = None
    if case["causal"]:
        hidden = torch.ones((S, S), dtype=torch.bool, device=DEV).triu_(1)
    flat = {n: v.reshape(B * H, S, D) for n, v in t.items()}
    for h in range(B * H):
        q, k, v = (flat[n][h].double() for n in ("Q", "K", "V"))
        s = (q @ k.t().contiguous()).mul_(scale)
        if hidden is not None:
            s.masked_fill_(hidden, -math.inf)
        lse[h] = torch.logsumexp(s, 1)
        p = s.sub_(lse[h][:, None]).exp_()
        o = p @ v
        out["O"][h] = o
        if train:
            do = flat["dO"][h].double()
            out["dV"][h] = p.t().contiguous() @ do
            ds = (do @ v.t().contiguous()).sub_((do * o).sum(1, keepdim=True)).mul_(p).mul_(scale)
            out["dQ"][h] = ds @ k
            out["dK"][h] = ds.t().contiguous() @ q
    res = {n: v.reshape(B, H, S, D) for n, v in out.items()}
    if not train:
        return res["O"]
    res["lse"] = lse.reshape(B, H, S)
    return {n: res[n] for n in ("O", "lse", "dQ", "dK", "dV")}


def _xent64(x, targets):
    """Mean of -log(p[target] + 1e-10) and (p - onehot) / M, the loss that the
    reference defines (include/jules/Kernel/FusedKernels.h:766)."""
    p = torch.softmax(x, 1)
    i = targets.long()[:, None]
    loss = -(p.gather(1, i) + 1e-10).log().mean()
    p.scatter_add_(1, i, torch.full_like(i, -1.0, dtype=torch.float64))
    return loss.reshape(1), p.div_(x.shape[0])


def exact(case, seed):
    t = _inputs(case, seed)
    k = case["kind"]
    if k == "gemm":
        v = t["A"].double() @ t["B"].double()
        return _act64(v if t["bias"] is None else v.add_(t["bias"].double()), case["act"])
    if k in ("flash", "flash_train"):
        return _attention64(t, case)
    if k == "w8a16":
        v = (t["x"].double() @ t["W"].double()).mul_(t["scale"].double())
        return _act64(v if t["bias"] is None else v.add_(t["bias"].double()), case["act"])
    if k == "int8":
        v = t["A"].double() @ t["B"].double()
        if case["per_token"]:
            v.mul_(t["sa"].double()[:, None]).mul_(t["sb"].double())
        else:
            v.mul_(0.013 * 0.021)
        return v if t["bias"] is None else v.add_(t["bias"].double())
    if k == "softmax":
        return torch.softmax(t["x"].double(), 1)
    if k == "layernorm":
        n = t["x"].shape[1]
        return torch.nn.functional.layer_norm(t["x"].double(), (n,), t["gamma"].double(),
                                              t["beta"].double(), 1e-5)
    if k == "xent":
        loss, grad = _xent64(t["x"].double(), t["targets"])
        return dict(loss=loss, grad=grad)
    if k == "mlp":
        X, W1, b1, W2, b2 = (t[n].double() for n in ("X", "W1", "b1", "W2", "b2"))
        a = (X @ W1).add_(b1).clamp_min_(0.0)
        o = (a @ W2).add_(b2)
        if not case["backward"]:
            return o
        loss, dO = _xent64(o, t["targets"])
        dH = (dO @ W2.t().contiguous()).mul_(a > 0)
        r = dict(output=o, loss=loss, dW1=X.t().contiguous() @ dH, db1=dH.sum(0),
                 dW2=a.t().contiguous() @ dO, db2=dO.sum(0))
        if case["dX"]:
            r["dX"] = dH @ W1.t().contiguous()
        return r
    return _act64(t["x"].double(), case["act"])
