"""The work that a program on this library has it do, as timed cases.

Every case goes through the ctypes binding (`mlx-runner_amd/qmm.py`), with device memory
held by torch tensors, results written into buffers the program keeps (as the benchmark and
a serving loop do), and work enqueued on torch's current stream without waiting for it.

A case is a dict with an "op" and its sizes:

  qmm        y = x @ deq(W).T                         {mode, M, N, K}
  mlp        down(silu(gate(x)) * up(x))              {mode, M, H, I}
  group      projections of one x, back to back       {mode, M, K, n0..n3}
  gdn_layer  in-projections, recurrence, out-projection of a gated-delta layer
                                                      {mode, M, H, Hk, Hv}
  gdn        the gated-delta recurrence               {B, T, Hk, Hv}
  linear     dense bf16 y = x @ W.T                   {M, N, K}
  convert    quantize a bf16 matrix, dequantize a packed one   {mode, N, K}

Weights are normal with a deviation of 0.02 in bf16, quantized here (group maxima, nearest
codes) without the library; activations are standard normal bf16.
"""
import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "mlx-runner_amd"))
import qmm as Q  # noqa: E402

DK = DV = 128  # head widths of the gated-delta layers
GROUP = {"mxfp8": 32, "nvfp4": 16}
E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)
MODES = ("nvfp4", "mxfp8")
ROWS = 16384  # rows of a weight made or used at a time


def listed():
    return [
        # one token through a linear-attention layer: four projections of one x, the state
        # update and the output projection, all of them short
        dict(name="decode gdn layer nvfp4", op="gdn_layer", mode="nvfp4", M=1, H=5120, Hk=16, Hv=48),
        # three rows (a draft of two being verified) through an MLP block
        dict(name="verify mlp mxfp8 m3", op="mlp", mode="mxfp8", M=3, H=5120, I=17408),
        # the next token's logits: the widest matrix of the model
        dict(name="decode lm_head nvfp4", op="qmm", mode="nvfp4", M=1, N=248320, K=5120),
        # a few sequences decoded together, on a hidden size other than the model's
        dict(name="batch decode nvfp4 m6", op="qmm", mode="nvfp4", M=6, N=14336, K=4096),
        # decode on a checkpoint that is not quantized (or a layer that is left dense)
        dict(name="decode dense m2", op="linear", M=2, N=5120, K=17408),
        # a prompt of a thousand tokens on the same
        dict(name="prefill dense m1000", op="linear", M=1000, N=10240, K=5120),
        # a short last chunk, or the tokens left after a prefix-cache hit
        dict(name="short prefill nvfp4 m48", op="qmm", mode="nvfp4", M=48, N=17408, K=5120),
        # the same, longer and ragged, on the long rows of the down projection
        dict(name="short prefill mxfp8 m200", op="qmm", mode="mxfp8", M=200, N=5120, K=17408),
        # a whole chunk of a prompt through a linear-attention layer's in-projections
        dict(name="prefill group nvfp4 m2048", op="group", mode="nvfp4", M=2048, K=5120, n0=10240, n1=6144, n2=48,
             n3=48),
        # a whole chunk through an MLP block: most of a prompt's time
        dict(name="prefill mlp mxfp8 m2048", op="mlp", mode="mxfp8", M=2048, H=5120, I=17408),
        # the recurrence over a prompt of 1500 tokens
        dict(name="prefill gdn t1500", op="gdn", B=1, T=1500, Hk=16, Hv=48),
        # a checkpoint's matrix converted: one quantized, one dequantized
        dict(name="convert nvfp4", op="convert", mode="nvfp4", N=10240, K=5120),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    op = rng.choice(("qmm", "qmm", "qmm", "mlp", "mlp", "group", "gdn_layer", "gdn", "linear", "linear", "convert"))
    mode = rng.choice(MODES)
    M = _log(rng, 1, 2048)
    kstep = rng.choice((32, 64, 128, 128))
    # half of the shapes are the model's projections, the others any
    if op in ("qmm", "linear"):
        N, K = rng.choice(((12288, 5120), (1024, 5120), (5120, 6144), (10240, 5120), (6144, 5120), (17408, 5120),
                           (5120, 17408), (5120, 10240), (34816, 5120)))
        if rng.random() < 0.5:
            N, K = _log(rng, 256, 34816, rng.choice((1, 8, 64))), _log(rng, 1024, 17408, kstep)
        while M * N * K > 5e11:
            M //= 2
        return dict(op=op, M=M, N=N, K=K, **({"mode": mode} if op == "qmm" else {}))
    if op == "mlp":
        H, I = 5120, 17408
        if rng.random() < 0.5:
            H, I = _log(rng, 1024, 8192, kstep), _log(rng, 2048, 20480, kstep)
        while 3 * M * H * I > 5e11:
            M //= 2
        return dict(op=op, mode=mode, M=M, H=H, I=I)
    if op == "group":
        K, n = 5120, (12288, 1024, 1024, 0)
        if rng.random() < 0.5:
            K, n = _log(rng, 1024, 8192, 128), tuple(_log(rng, 256, 8192, 64) for _ in range(2)) + (64, 64)
        return dict(op=op, mode=mode, M=M, K=K, n0=n[0], n1=n[1], n2=n[2], n3=n[3])
    if op == "gdn_layer":
        Hk = rng.choice((8, 16, 16, 32))
        return dict(op=op, mode=mode, M=rng.randint(1, 4), H=rng.choice((2048, 4096, 5120, 5120)), Hk=Hk,
                    Hv=Hk * rng.choice((1, 2, 3)))
    if op == "gdn":
        Hk = rng.choice((4, 8, 16, 16))
        return dict(op=op, B=rng.choice((1, 1, 1, 2, 4)), T=_log(rng, 1, 2048), Hk=Hk, Hv=Hk * rng.choice((1, 2, 3)))
    return dict(op=op, mode=mode, N=_log(rng, 1024, 17408, rng.choice((1, 64))), K=_log(rng, 1024, 17408, kstep))


# ---------------------------------------------------------------- inputs


def _gen(seed, what):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + what)
    return g


def _normal(seed, what, shape, scale=1.0):
    return (torch.randn(shape, generator=_gen(seed, what), device="cuda") * scale).to(torch.bfloat16)


def _quantize(v, mode):
    """(codes packed in bytes, scale bytes) of a float32 matrix."""
    n, k = v.shape
    g = v.view(n, k // GROUP[mode], GROUP[mode])
    amax = g.abs().amax(-1, keepdim=True)
    if mode == "mxfp8":
        e = torch.floor(torch.log2(amax)) - 8
        q = torch.ldexp(g, -e).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8)
        return q.view(n, k), (e + 127).to(torch.uint8).squeeze(-1)
    s = (amax / 6).to(torch.float8_e4m3fn)
    edges = torch.tensor([(a + b) / 2 for a, b in zip(E2M1, E2M1[1:])], device=v.device)
    code = torch.bucketize((g / s.float()).abs(), edges, out_int32=True).to(torch.uint8)
    code = (code + 8 * (g < 0).to(torch.uint8)).view(n, k // 2, 2)
    return code[..., 0] + 16 * code[..., 1], s.view(torch.uint8).squeeze(-1)


def _packed(seed, what, N, K, mode):
    """A quantized weight: (int32 [N, K * bits / 32], uint8 [N, K / group])."""
    gen = _gen(seed, what)
    w = torch.empty((N, K if mode == "mxfp8" else K // 2), dtype=torch.uint8, device="cuda")
    s = torch.empty((N, K // GROUP[mode]), dtype=torch.uint8, device="cuda")
    for r in range(0, N, ROWS):
        n = min(ROWS, N - r)
        v = (torch.randn((n, K), generator=gen, device="cuda") * 0.02).to(torch.bfloat16).float()
        w[r:r + n], s[r:r + n] = _quantize(v, mode)
    return w.view(torch.int32), s


def _deq64(w, s, mode):
    w, s = w.view(torch.uint8), s
    if mode == "mxfp8":
        v = w.view(torch.float8_e4m3fn).double()
        sc = torch.exp2(s.double() - 127)
    else:
        t = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=torch.float64, device="cuda")
        v = torch.stack((t[(w & 15).int()], t[(w >> 4).int()]), -1).view(w.shape[0], -1)
        sc = s.view(torch.float8_e4m3fn).double()
    return (v.view(s.shape[0], s.shape[1], -1) * sc.unsqueeze(-1)).view(w.shape[0], -1)


def _mm64(x, wq, mode):
    """x (float64) @ deq(w).T in float64, some rows of w at a time."""
    w, s = wq
    step = max(256, (1 << 27) // (x.shape[1] + 1))
    return torch.cat([x @ _deq64(w[r:r + step], s[r:r + step], mode).t() for r in range(0, w.shape[0], step)], 1)


def _parts(case):
    """The projections of a grouped call."""
    if case["op"] == "group":
        return [case[k] for k in ("n0", "n1", "n2", "n3") if case[k]]
    Hk, Hv = case["Hk"], case["Hv"]
    return [2 * Hk * DK + Hv * DV, Hv * DV, Hv, Hv]


def _heads(seed, B, T, Hk, Hv):
    """q, k, v, g, beta, state of the recurrence: normalised q and k, decays in (0.5, 1)."""
    rn = lambda what, *s: torch.randn(s, generator=_gen(seed, what), device="cuda")  # noqa: E731
    q, k = rn(40, B, T, Hk, DK), rn(41, B, T, Hk, DK)
    q = (q / q.pow(2).mean(-1, keepdim=True).sqrt() / DK).to(torch.bfloat16)
    k = (k / k.pow(2).mean(-1, keepdim=True).sqrt() / math.sqrt(DK)).to(torch.bfloat16)
    v = rn(42, B, T, Hv, DV).to(torch.bfloat16)
    g = torch.exp(-0.7 * torch.rand((B, T, Hv), generator=_gen(seed, 43), device="cuda"))
    beta = torch.sigmoid(rn(44, B, T, Hv)).to(torch.bfloat16)
    return q, k, v, g, beta, rn(45, B, Hv, DV, DK) * 0.1


def _tensors(case, seed):
    """The inputs of a case as tensors, by name; packed weights are (words, scales)."""
    op, mode, t = case["op"], case.get("mode"), {}
    if op == "qmm":
        t["x"] = _normal(seed, 0, (case["M"], case["K"]))
        t["w"] = _packed(seed, 1, case["N"], case["K"], mode)
    elif op == "mlp":
        t["x"] = _normal(seed, 0, (case["M"], case["H"]))
        t["gate"], t["up"] = (_packed(seed, i, case["I"], case["H"], mode) for i in (1, 2))
        t["down"] = _packed(seed, 3, case["H"], case["I"], mode)
    elif op == "linear":
        t["x"] = _normal(seed, 0, (case["M"], case["K"]))
        t["w"] = _normal(seed, 1, (case["N"], case["K"]), 0.02)
    elif op == "convert":
        t["dense"] = _normal(seed, 0, (case["N"], case["K"]), 0.02)
        t["w"] = _packed(seed, 1, case["N"], case["K"], mode)
    if op in ("group", "gdn_layer"):
        # the members are row ranges of one matrix, as the loader places them
        K = case["K"] if op == "group" else case["H"]
        t["x"] = _normal(seed, 0, (case["M"], K))
        t["w"] = _packed(seed, 1, sum(_parts(case)), K, mode)
    if op == "gdn_layer":
        t["heads"] = _heads(seed, 1, case["M"], case["Hk"], case["Hv"])
        t["h"] = _normal(seed, 2, (case["M"], case["Hv"] * DV), 0.5)
        t["out"] = _packed(seed, 3, case["H"], case["Hv"] * DV, mode)
    if op == "gdn":
        t["heads"] = _heads(seed, case["B"], case["T"], case["Hk"], case["Hv"])
    return t


# ---------------------------------------------------------------- a program's state and its pass


class State:
    """Inputs, weights and result buffers behind the library's handles."""

    def __init__(self, case, seed):
        self.case, self.op, self.mode = case, case["op"], case.get("mode")
        self.stream = Q.Stream.torch_current()
        self.a, self.out = {}, {}
        for k, v in _tensors(case, seed).items():
            if isinstance(v, tuple):
                self.a[k] = [Q.Array.from_torch(p) for p in v]
            else:
                self.a[k] = Q.Array.from_torch(v)
        op, bf = self.op, torch.bfloat16
        if op in ("qmm", "linear"):
            self._result("y", (case["M"], case["N"]), bf)
        elif op == "mlp":
            self._result("h", (case["M"], case["I"]), bf)
            self._result("y", (case["M"], case["H"]), bf)
        elif op in ("group", "gdn_layer"):
            (w, s), self.ws, self.ss, self.ys, r = [p._keep for p in self.a["w"]], [], [], [], 0
            for i, n in enumerate(_parts(case)):
                self.ws.append(Q.Array.from_torch(w[r:r + n]))
                self.ss.append(Q.Array.from_torch(s[r:r + n]))
                self.ys.append(self._result("p%d" % i, (case["M"], n), bf))
                r += n
        if op in ("gdn", "gdn_layer"):
            B, T = (case["B"], case["T"]) if op == "gdn" else (1, case["M"])
            self._result("o", (B, T, case["Hv"], DV), bf)
            self._result("state", (B, case["Hv"], DV, DK), torch.float32)
        if op == "gdn_layer":
            self._result("y", (case["M"], case["H"]), bf)

    def _result(self, name, shape, dtype):
        self.out[name] = Q.Array.from_torch(torch.empty(shape, dtype=dtype, device="cuda"))
        return self.out[name]

    def results(self):
        return {k: v._keep for k, v in self.out.items()}


class _Device:
    """A library array that torch can look at in place."""

    def __init__(self, array, kind):
        self.array = array
        self.__cuda_array_interface__ = dict(shape=array.shape, typestr=kind, data=(array.ptr, False), version=2)


def _look(array, kind):
    return torch.as_tensor(_Device(array, kind), device="cuda")


def prepare(case, seed):
    return State(case, seed)


def run(s):
    a, o, mode, st = s.a, s.out, s.mode, s.stream
    if s.op == "qmm":
        Q.quantized_matmul(a["x"], *a["w"], mode, out=o["y"], stream=st)
    elif s.op == "mlp":
        Q.mlp_gate_up_silu(a["x"], *a["gate"], *a["up"], mode, out=o["h"], stream=st)
        Q.quantized_matmul(o["h"], *a["down"], mode, out=o["y"], stream=st)
    elif s.op == "linear":
        Q.linear(a["x"], a["w"], out=o["y"], stream=st)
    elif s.op == "convert":
        w, sc = Q.quantize(a["dense"], mode, stream=st)
        d = Q.dequantize(*a["w"], mode, stream=st)
        # bf16 bits as int16, seen as bf16
        return _look(w, "<i4"), _look(sc, "|u1"), _look(d, "<i2").view(torch.bfloat16)
    if s.op in ("group", "gdn_layer"):
        Q.quantized_matmul_group(a["x"], s.ws, s.ss, mode, outs=s.ys, stream=st)
    if s.op in ("gdn", "gdn_layer"):
        Q.gdn_recurrence(*a["heads"], y=o["o"], state_out=o["state"], stream=st)
    if s.op == "gdn_layer":
        Q.quantized_matmul(a["h"], *a["out"], mode, out=o["y"], stream=st)
    return s.results()


# ---------------------------------------------------------------- what a pass cannot do without


def _matmul_work(M, N, K, mode, x=True, y=True):
    w = N * K * 2 if mode is None else N * K if mode == "mxfp8" else N * K // 2
    s = N * K // GROUP[mode] if mode else 0
    return w + s + 2 * M * (K * x + N * y), 2 * M * N * K


def _heads_work(B, T, Hk, Hv):
    state = B * Hv * DV * DK
    return B * T * (4 * Hk * DK + 4 * Hv * DV + 6 * Hv) + 8 * state, 7 * T * state


def work(case):
    op, mode, M = case["op"], case.get("mode"), case.get("M", 0)
    if op in ("qmm", "linear"):
        parts = [_matmul_work(M, case["N"], case["K"], mode)]
    elif op == "mlp":
        H, I = case["H"], case["I"]
        parts = [_matmul_work(M, 2 * I, H, mode, y=False), (2 * M * I, 0), _matmul_work(M, H, I, mode)]
    elif op == "group":
        parts = [_matmul_work(M, sum(_parts(case)), case["K"], mode)]
    elif op == "gdn_layer":
        parts = [_matmul_work(M, sum(_parts(case)), case["H"], mode), _heads_work(1, M, case["Hk"], case["Hv"]),
                 _matmul_work(M, case["H"], case["Hv"] * DV, mode)]
    elif op == "gdn":
        parts = [_heads_work(case["B"], case["T"], case["Hk"], case["Hv"])]
    else:
        n = case["N"] * case["K"]
        packed = (n if mode == "mxfp8" else n // 2) + n // GROUP[mode]
        parts = [(2 * (2 * n + packed), 2 * n)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    # bf16 results measure 1.7e-3 from the exact ones in the 2-norm (a rounding, at most 2^-8
    # of the value), 4.1e-3 through the MLP's several roundings; four times that
    if case["op"] == "convert":
        return {"rel": 1e-6, "differ": 0.0}
    if case["op"] == "mlp":
        return {"rel": 1.6e-2, "max": 7e-2}
    return {"rel": 7e-3, "max": 3e-2}


# ---------------------------------------------------------------- in 64 bits


def _heads64(q, k, v, g, beta, S):
    B, T, Hk, _ = q.shape
    r = v.shape[2] // Hk
    q, k = (t.double().repeat_interleave(r, 2) for t in (q, k))
    v, g, beta, S, y = v.double(), g.double(), beta.double(), S.double().clone(), []
    for i in range(T):
        S = S * g[:, i, :, None, None]
        d = (v[:, i] - (S * k[:, i, :, None, :]).sum(-1)) * beta[:, i, :, None]
        S = S + d.unsqueeze(-1) * k[:, i, :, None, :]
        y.append((S * q[:, i, :, None, :]).sum(-1))
    return torch.stack(y, 1), S


def exact(case, seed):
    t, op, mode = _tensors(case, seed), case["op"], case.get("mode")
    x = t["x"].double() if "x" in t else None
    if op == "qmm":
        return {"y": _mm64(x, t["w"], mode)}
    if op == "mlp":
        g, u = (_mm64(x, t[n], mode) for n in ("gate", "up"))
        h = g * torch.sigmoid(g) * u
        return {"h": h, "y": _mm64(h, t["down"], mode)}
    if op == "linear":
        return {"y": x @ t["w"].double().t()}
    if op == "convert":
        return None, None, _deq64(*t["w"], mode)
    out = {}
    if op in ("group", "gdn_layer"):
        out = {"p%d" % i: v.contiguous() for i, v in enumerate(_mm64(x, t["w"], mode).split(_parts(case), 1))}
    if op in ("gdn", "gdn_layer"):
        out["o"], out["state"] = _heads64(*t["heads"])
    if op == "gdn_layer":
        out["y"] = _mm64(t["h"].double(), t["out"], mode)
    return out
