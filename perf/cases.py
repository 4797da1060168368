"""Cases for timing the framework: what its users have it do, through its public entry points.

Every case is a whole call: a decode step, an inference pass (``newton_apply``) or a training step
(``newton_apply`` or a ``ParaRNN`` stack, forward and backward).  Inputs are ``N(0, 0.5)`` and the
weights are the cells' own initialisation, as in the benchmark.  Two solver settings are in use:

* ``"default"``: ``NewtonConfig()`` -- K = 3, automatic Picard depth, the residual gate and the
  adaptive Picard ladder on.  It is what float32 callers get without asking.
* ``"fixed"``: K, P fixed and no host check, the setting for 16-bit storage, where the rounding of
  the stored state (not the solve) decides the residual that the gate would test.

16-bit sLSTM sequences stay at T <= 2048 (training 1024) and float32 ones at T <= 16384 (training
4096): beyond that the stabiliser slot of the sLSTM outgrows its storage and K Newton steps need not
converge on every channel (the gate raises, or two correct runs differ by any amount).
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "pararnn-torch_amd"))

from pararnn_amd import (  # noqa: E402
    NewtonConfig,
    ParaGRU,
    ParaRNN,
    ParaSLSTM,
    decode_step,
    newton_apply,
)

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}


def listed() -> list[dict]:
    return [
        # serving: one token for each of 64 sessions, the smallest call of all
        dict(name="decode_slstm_bf16", kind="decode", cell="slstm", dtype="bf16", B=64, d=1024),
        # a small model scored in float32 with the library defaults
        dict(name="slstm_f32_small", kind="infer", cell="slstm", dtype="f32", config="default",
             B=2, T=1024, d=64),
        # training a two-layer sLSTM stack in float32, library defaults
        dict(name="slstm_f32_train_stack", kind="stack", cell="slstm", dtype="f32",
             config="default", B=8, T=2048, d=256, layers=2),
        # long documents scored in float32, library defaults
        dict(name="slstm_f32_long", kind="infer", cell="slstm", dtype="f32", config="default",
             B=8, T=16384, d=512),
        # prefill of a large bf16 batch: the largest sLSTM call
        dict(name="slstm_bf16_large", kind="infer", cell="slstm", dtype="bf16", config="fixed",
             B=64, T=2048, d=1024),
        # a bf16 training step of one sLSTM layer
        dict(name="slstm_bf16_train", kind="train", cell="slstm", dtype="bf16", config="fixed",
             B=32, T=1024, d=768),
        # a packed batch of ragged bf16 sequences, each with its own initial state
        dict(name="slstm_bf16_packed", kind="infer", cell="slstm", dtype="bf16", config="fixed",
             N=60013, seqs=53, d=1024, h0=True),
        # a batch of long float32 sequences through the head GRU, library defaults
        dict(name="gru_f32_long", kind="infer", cell="gru", dtype="f32", config="default",
             B=4, T=32768, heads=8, d_head=64),
        # training on one float32 sequence at a time
        dict(name="gru_f32_train_one", kind="train", cell="gru", dtype="f32", config="default",
             B=1, T=4096, heads=8, d_head=64),
        # an ordinary bf16 training batch of the head GRU
        dict(name="gru_bf16_train", kind="train", cell="gru", dtype="bf16", config="fixed",
             B=16, T=1024, heads=8, d_head=64),
        # wide heads, a float32 training step
        dict(name="gru_wide_f32_train", kind="train", cell="gru", dtype="f32", config="default",
             B=4, T=4096, heads=4, d_head=128),
        # narrow heads on a packed ragged float32 batch with initial states, a training step
        dict(name="gru_narrow_packed_train", kind="train", cell="gru", dtype="f32",
             config="default", N=9001, seqs=23, heads=8, d_head=24, h0=True),
    ]


def _log(rng, lo: int, hi: int) -> int:
    """A whole number in [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _batch(rng, T_lo: int, T_hi: int, B_hi: int, width: int, most: int) -> dict:
    """B and T with B * T * width <= most."""
    T = _log(rng, T_lo, min(T_hi, max(T_lo, most // width)))
    return dict(B=_log(rng, 1, max(1, min(B_hi, most // (T * width)))), T=T)


def _ragged(rng, N_lo: int, N_hi: int, width: int, most: int) -> dict:
    N = _log(rng, N_lo, min(N_hi, most // width))
    # uneven lengths, the longest about twice the mean of at most 512 (see _offsets)
    return dict(N=N, seqs=_log(rng, max(2, -(-N // 512)), max(3, N // 64)))


def draw(rng) -> dict:
    what = rng.choice(["decode", "slstm_f32", "slstm_f32", "slstm_16", "slstm_16", "slstm_packed",
                       "gru", "gru", "gru_wide", "gru_packed"])
    if what == "decode":
        c = dict(kind="decode", cell=rng.choice(["slstm", "gru"]),
                 dtype=rng.choice(["bf16", "f16", "f32"]), B=_log(rng, 1, 512))
        return dict(c, d=_log(rng, 64, 2048)) if c["cell"] == "slstm" else \
            dict(c, heads=_log(rng, 1, 16), d_head=64)
    if what == "slstm_f32":
        d = _log(rng, 32, 1024)
        kind = rng.choice(["infer", "train", "stack"])
        c = dict(kind=kind, cell="slstm", dtype="f32", config="default", d=d,
                 **_batch(rng, 64, 16384 if kind == "infer" else 4096, 32, d, 1 << 24))
        return dict(c, layers=rng.randint(1, 2)) if kind == "stack" else c
    if what == "slstm_16":
        d = _log(rng, 64, 1536)
        kind, dtype = rng.choice([("infer", "bf16"), ("infer", "f16"), ("train", "bf16")])
        return dict(kind=kind, cell="slstm", dtype=dtype, config="fixed", d=d,
                    **_batch(rng, 64, 2048 if kind == "infer" else 1024, 64, d, 1 << 25))
    if what == "slstm_packed":
        d = _log(rng, 64, 1024)
        c = dict(kind=rng.choice(["infer", "train"]), cell="slstm",
                 dtype=rng.choice(["bf16", "f32"]), d=d, h0=rng.random() < 0.5)
        return dict(c, config="default" if c["dtype"] == "f32" else "fixed",
                    **_ragged(rng, 512, 65536, d, 1 << 24))
    if what == "gru":
        heads, d_head = _log(rng, 1, 16), rng.choice([64, 64, 64, 32, 48])
        c = dict(kind=rng.choice(["infer", "train"]), cell="gru", dtype=rng.choice(["f32", "bf16"]),
                 heads=heads, d_head=d_head,
                 **_batch(rng, 64, 16384, 64, heads * 64, 1 << 24))
        return dict(c, config="default" if c["dtype"] == "f32" else "fixed")
    if what == "gru_wide":
        heads, d_head = _log(rng, 1, 8), rng.choice([80, 96, 128])
        return dict(kind=rng.choice(["infer", "train"]), cell="gru", dtype="f32",
                    config="default", heads=heads, d_head=d_head,
                    **_batch(rng, 64, 4096, 16, heads * 128, 1 << 23))
    heads, d_head = _log(rng, 1, 12), rng.choice([16, 24, 32, 64])
    return dict(kind=rng.choice(["infer", "train"]), cell="gru", dtype="f32", config="default",
                heads=heads, d_head=d_head, h0=rng.random() < 0.5,
                **_ragged(rng, 256, 32768, heads * 64, 1 << 22))


# ---------------------------------------------------------------------------
# What a user's program holds, and one pass of it
# ---------------------------------------------------------------------------


def _width(case: dict) -> int:
    return case["d"] if case["cell"] == "slstm" else case["heads"] * case["d_head"]


def _config(case: dict) -> NewtonConfig:
    if case["config"] == "default":
        return NewtonConfig()
    slstm = case["cell"] == "slstm"
    return NewtonConfig(max_iters=3, picard_iters=5 if slstm else None, picard_adapt=False,
                        residual_atol=None, residual_fail=None)


def _cell(case: dict) -> torch.nn.Module:
    d = _width(case)
    kw = dict(device=DEVICE, dtype=torch.float32)
    cell = ParaSLSTM(d, d, mix="diag", **kw) if case["cell"] == "slstm" else \
        ParaGRU(d, d, mix="head", n_heads=case["heads"], **kw)
    return cell.to(DTYPES[case["dtype"]])


def _offsets(case: dict, gen: torch.Generator) -> torch.Tensor:
    """cu_seqlens of ``seqs`` sequences of uneven lengths, N steps in all."""
    w = torch.rand(case["seqs"], generator=gen, dtype=torch.float64) * 1.9 + 0.1
    cuts = (torch.cumsum(w, 0) / w.sum() * (case["N"] - case["seqs"])).round().to(torch.int64)
    ends = cuts + torch.arange(1, case["seqs"] + 1)
    ends[-1] = case["N"]
    return torch.cat([torch.zeros(1, dtype=torch.int64), ends])


def prepare(case: dict, seed: int) -> dict:
    torch.manual_seed(seed)
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    dtype, d, kind = DTYPES[case["dtype"]], _width(case), case["kind"]

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=gen, device=DEVICE) * std).to(dtype)

    cell = _cell(case)
    s = dict(case=case, cell=cell)
    if kind == "decode":
        B = case["B"]
        s["x"] = normal(B, d, std=0.5)
        if case["cell"] == "slstm":
            # c, n, m, h as a running session has them: n positive, |c| <= n, |h| < 1
            n = normal(B, 1, d).abs() * 20 + 1
            s["state"] = torch.cat([n * torch.tanh(normal(B, 1, d)), n, normal(B, 1, d) * 8,
                                    torch.tanh(normal(B, 1, d)) * 0.5], 1)
        else:
            s["state"] = torch.tanh(normal(B, d))
        s["out"] = torch.empty_like(s["state"])
        return s
    s["config"] = _config(case)
    rows = (1, case["N"]) if "N" in case else (case["B"], case["T"])
    s["x"] = normal(*rows, d, std=0.5)
    s["cu"] = s["h0"] = None
    if "N" in case:
        s["cu"] = _offsets(case, torch.Generator().manual_seed(seed + 2)).to(DEVICE)
    if case.get("h0"):
        S = case["seqs"]
        if case["cell"] == "slstm":
            n = normal(S, 1, d).abs() + 1
            s["h0"] = torch.cat([n * torch.tanh(normal(S, 1, d)), n, normal(S, 1, d),
                                 torch.tanh(normal(S, 1, d)) * 0.5], 1)
        else:
            s["h0"] = torch.tanh(normal(S, d))
    if kind == "infer":
        return s
    s["x"].requires_grad_(True)
    if s["h0"] is not None:
        s["h0"].requires_grad_(True)
    if kind == "stack":
        # a constructor's own draws: the deeper layers are fresh cells of the template's class
        s["net"] = ParaRNN(cell, num_layers=case["layers"], config=s["config"]).train()
        s["weights"] = list(s["net"].parameters())
        s["grad"] = normal(*rows, d)
    else:
        s["weights"] = list(cell.parameters())
        s["grad"] = normal(*rows, *((4, d) if case["cell"] == "slstm" else (d,)))
    return s


def run(s: dict):
    kind = s["case"]["kind"]
    if kind == "decode":
        with torch.no_grad():
            return decode_step(s["cell"], s["state"], s["x"], out=s["out"])
    if kind == "infer":
        with torch.no_grad():
            return newton_apply(s["cell"], s["x"], s["config"], h0=s["h0"], cu_seqlens=s["cu"])
    out = s["net"](s["x"]) if kind == "stack" else \
        newton_apply(s["cell"], s["x"], s["config"], h0=s["h0"], cu_seqlens=s["cu"])
    leaves = [s["x"], *s["weights"]] + ([] if s["h0"] is None else [s["h0"]])
    return [out.detach(), *torch.autograd.grad(out, leaves, s["grad"])]


def work(case: dict) -> dict:
    d, es = _width(case), 4 if case["dtype"] == "f32" else 2
    slstm = case["cell"] == "slstm"
    gates, slots = (4, 4) if slstm else (3, 1)
    n = case["B"] if case["kind"] == "decode" else case.get("N") or case["B"] * case["T"]
    weights = gates * d * d + (gates * d + 4 * d if slstm else 3 * d + 3 * d * case["d_head"])
    gemm = 2 * n * d * gates * d
    # one evaluation of the recurrent part: elementwise, or three products with a head's matrices
    cell = (40 if slstm else 6 * case["d_head"] + 20) * n * d
    if case["kind"] == "decode":
        return dict(bytes=es * (n * d * (1 + 2 * slots) + weights), flops=gemm + cell)
    P, K = (0, 3) if not slstm else (5, 3) if case["config"] == "fixed" else \
        (3 if case.get("T", case.get("N")) <= 2048 else 5, 3)
    # a Newton iteration: the cell, its Jacobian applied to a vector, the update
    flops = gemm + (P + 1) * (cell if slstm else 0) + K * 2 * cell
    nbytes = es * (n * d * (1 + slots) + weights)
    if case["kind"] != "infer":
        flops += 2 * gemm + 3 * cell + (0 if slstm else 6 * n * d * case["d_head"])
        nbytes += es * (n * d * (1 + slots) + weights)
    layers = case.get("layers", 1)
    return dict(bytes=layers * nbytes, flops=layers * flops)


def tolerance(case: dict):
    """Four times and more what the path differs by from the same in 64 bits (float32), or what a
    flip of the last stored bit does (16 bits: 2^-9 of a bf16 value).  The sLSTM's adjoint
    amplifies a change of rounding in the states with the length of the sequence."""
    if case["dtype"] != "f32":
        return {"rel": 0.01}
    if case["cell"] == "gru" or case["kind"] == "decode":
        return {"rel": 1e-5}
    if case["kind"] == "infer":
        return {"rel": 4e-5}
    return {"rel": 5e-5 if case.get("T", 0) <= 2048 else 1e-4}


# ---------------------------------------------------------------------------
# The same in 64 bits, in plain torch: every sum and product in float64; what a layer keeps between
# its parts in the tensors' own type (the projected input, and the states that the backward reads)
# is rounded to that type, as in any implementation of the same layer.
# ---------------------------------------------------------------------------


class _Stored(torch.autograd.Function):
    """Values rounded to the storage type; the gradient passes."""

    @staticmethod
    def forward(ctx, v, dtype):
        return v.to(dtype).double()

    @staticmethod
    def backward(ctx, g):
        return g, None


def _slstm_step(prev, wx, R, eps):
    """prev, result (B, T, 4, d); wx (B, T, 4 d)."""
    c, n, m, h = prev.unbind(-2)
    d = h.shape[-1]
    zi, zf, zz, zo = (wx[..., g * d:(g + 1) * d] + R[g] * h for g in range(4))
    mn = torch.maximum(zf + m, zi)
    i, f = torch.exp(zi - mn), torch.exp(zf + m - mn)
    nn_, cn = f * n + i, f * c + i * torch.tanh(zz)
    return torch.stack((cn, nn_, mn, torch.sigmoid(zo) * cn / (nn_ + eps)), -2)


def _slstm_jac(prev, wx, R, eps):
    """The 4 x 4 Jacobian, (B, T, 4 out, 4 in, d)."""
    c, n, m, h = prev.unbind(-2)
    d = h.shape[-1]
    zi, zf, zz, zo = (wx[..., g * d:(g + 1) * d] + R[g] * h for g in range(4))
    left = zf + m
    mn = torch.maximum(left, zi)
    a = (left > zi).double() + 0.5 * (left == zi).double()
    i, f, z, o = torch.exp(zi - mn), torch.exp(left - mn), torch.tanh(zz), torch.sigmoid(zo)
    nn_, cn = f * n + i, f * c + i * z
    J = torch.zeros(*h.shape[:-1], 4, 4, d, dtype=torch.float64, device=h.device)
    mh = a * R[1] + (1 - a) * R[0]
    ih, fh = i * (R[0] - mh), f * (R[1] - mh)
    J[..., 0, 0, :] = J[..., 1, 1, :] = f
    J[..., 0, 2, :] = f * (1 - a) * c - i * a * z
    J[..., 0, 3, :] = fh * c + ih * z + i * (1 - z * z) * R[2]
    J[..., 1, 2, :] = f * (1 - a) * n - i * a
    J[..., 1, 3, :] = fh * n + ih
    J[..., 2, 2, :], J[..., 2, 3, :] = a, mh
    den = nn_ + eps
    J[..., 3, :, :] = (o / den).unsqueeze(-2) * J[..., 0, :, :] - \
        (o * cn / den ** 2).unsqueeze(-2) * J[..., 1, :, :]
    J[..., 3, 3, :] += cn / den * o * (1 - o) * R[3]
    return J


def _slstm_frozen(pre, h0, eps):
    """The states when the gates are frozen at ``pre`` (B, T, 4 d): a scan in closed form."""
    d = pre.shape[-1] // 4
    zi, zf, zz, zo = (pre[..., g * d:(g + 1) * d] for g in range(4))
    c0, n0, m0, _ = (t.unsqueeze(1) for t in h0.unbind(1))
    F = torch.cumsum(zf, 1)
    m = torch.maximum(torch.cummax(zi - F, 1).values, m0) + F
    z = torch.tanh(zz)

    def total(w, start):  # sum_s w_s e^{z_i,s - F_s} + start e^{m0}, by sign, in logarithms
        terms = torch.cat((torch.log(start) + m0, torch.log(w) + zi - F), 1)
        return torch.exp(torch.logcumsumexp(terms, 1)[:, 1:] + F - m)

    n = total(torch.ones_like(z), n0)
    c = total(z.clamp(min=0), c0.clamp(min=0)) - total((-z).clamp(min=0), (-c0).clamp(min=0))
    return torch.stack((c, n, m, torch.sigmoid(zo) * c / (n + eps)), 2)


def _shift(H, h0):
    return torch.cat((h0.unsqueeze(1), H[:, :-1]), 1)


def _walk(J, F, reverse=False):
    """delta_t = J_t delta_{t-1} + F_t; reverse: nu_t = J_t^T (F_t + nu_{t+1})."""
    out = torch.empty_like(F)
    v = torch.zeros_like(F[:, 0])
    J = J.transpose(-3, -2) if reverse else J
    for t in (reversed(range(F.shape[1])) if reverse else range(F.shape[1])):
        if reverse:
            v = (J[:, t] * (v + F[:, t]).unsqueeze(-3)).sum(-2)
        else:
            v = (J[:, t] * v.unsqueeze(-3)).sum(-2) + F[:, t]
        out[:, t] = v
    return out


class _SLSTM:
    def __init__(self, cell):
        self.W, self.b, self.R = (p.detach().double().requires_grad_(True)
                                  for p in (cell.W_x.weight, cell.W_x.bias, cell.R))
        self.weights = {"W_x.weight": self.W, "W_x.bias": self.b, "R": self.R}
        self.cap, self.eps, self.tail = cell.max_recurrent_norm, cell.eps, (4, cell.d_h)
        self.dtype = cell.R.dtype

    def wx(self, x):
        return _Stored.apply(x @ self.W.t() + self.b, self.dtype)

    def f(self, prev, x):
        return _slstm_step(prev, self.wx(x), self.R.clamp(-self.cap, self.cap), self.eps)

    def solve(self, x, h0, K, P):
        R, wx = self.R.clamp(-self.cap, self.cap), self.wx(x)
        H = _slstm_frozen(wx, h0, self.eps)
        for _ in range(P):
            h = _shift(H, h0)[..., 3, :]
            H = _slstm_frozen(wx + (R * h.unsqueeze(-2)).flatten(-2), h0, self.eps)
        for _ in range(K):
            prev = _shift(H, h0)
            H = H + _walk(_slstm_jac(prev, wx, R, self.eps), _slstm_step(prev, wx, R, self.eps) - H)
        return H

    def adjoint(self, prev, x, g):
        J = _slstm_jac(prev, self.wx(x), self.R.clamp(-self.cap, self.cap), self.eps)
        return _walk(J, g, reverse=True)


class _GRU:
    def __init__(self, cell):
        self.H, self.dh = cell.n_heads, cell.d_head
        self.W, self.b, *self.A = (p.detach().double().requires_grad_(True) for p in (
            cell.W_x.weight, cell.W_x.bias, cell.A_z, cell.A_r, cell.A_n))
        self.weights = {"W_x.weight": self.W, "W_x.bias": self.b,
                        **dict(zip(("A_z", "A_r", "A_n"), self.A))}
        self.tail, self.dtype = (cell.d_h,), cell.A_z.dtype

    def gates(self, prev, x):
        def mix(v, a):
            rows = v.reshape(-1, self.H, self.dh).transpose(0, 1)
            return torch.matmul(rows, a).transpose(0, 1).reshape(v.shape)

        zx, rx, nx = _Stored.apply(x @ self.W.t() + self.b, self.dtype).chunk(3, -1)
        z = torch.sigmoid(zx + mix(prev, self.A[0]))
        r = torch.sigmoid(rx + mix(prev, self.A[1]))
        return z, r, torch.tanh(nx + mix(prev * r, self.A[2]))

    def f(self, prev, x):
        z, _, n = self.gates(prev, x)
        return prev + z * (n - prev)

    def _rows(self, v):  # (B, T, d) -> (T, H, B, dh)
        B, T, _ = v.shape
        return v.reshape(B, T, self.H, self.dh).permute(1, 2, 0, 3).contiguous()

    def _scalars(self, prev, x):
        z, r, n = self.gates(prev, x)
        return [self._rows(v) for v in (1 - z, (n - prev) * z * (1 - z), z * (1 - n * n), r,
                                        prev * r * (1 - r))]

    def _back(self, v):
        T, _, B, _ = v.shape
        return v.permute(2, 0, 1, 3).reshape(B, T, -1)

    def solve(self, x, h0, K, P):
        prev = _shift(torch.zeros(*x.shape[:2], self.H * self.dh, dtype=x.dtype, device=x.device),
                      h0)
        H = self.f(prev, x)
        zr = torch.cat(self.A[:2], -1)
        for _ in range(K):
            prev = _shift(H, h0)
            d1, d2, d3, r, d5 = self._scalars(prev, x)
            F = self._rows(self.f(prev, x) - H)
            v = torch.zeros_like(F[0])
            out = torch.empty_like(F)
            for t in range(F.shape[0]):
                y = torch.bmm(v, zr)
                u = torch.addcmul(r[t] * v, d5[t], y[..., self.dh:])
                v = torch.addcmul(torch.addcmul(F[t], d1[t], v), d2[t], y[..., :self.dh])
                v = torch.addcmul(v, d3[t], torch.bmm(u, self.A[2]), out=out[t])
            H = H + self._back(out)
        return H

    def adjoint(self, prev, x, g):
        d1, d2, d3, r, d5 = self._scalars(prev, x)
        g = self._rows(g)
        az, ar, an = (a.transpose(1, 2).contiguous() for a in self.A)
        nu, out = torch.zeros_like(g[0]), torch.empty_like(g)
        for t in reversed(range(g.shape[0])):
            mu = g[t] + nu
            u = torch.bmm(d3[t] * mu, an)
            nu = d1[t] * mu + torch.bmm(d2[t] * mu, az) + r[t] * u + torch.bmm(d5[t] * u, ar)
            out[t] = nu
        return self._back(out)


def _pad(v, cu):
    """A packed (1, N, ...) stream as a (S, longest, ...) batch, zeros past each end."""
    n = (cu[1:] - cu[:-1]).tolist()
    out = v.new_zeros(len(n), max(n), *v.shape[2:])
    for q, k in enumerate(n):
        out[q, :k] = v[0, cu[q]:cu[q + 1]]
    return out


def _unpad(v, cu):
    return torch.cat([v[q, :int(cu[q + 1] - cu[q])] for q in range(v.shape[0])]).unsqueeze(0)


def _layer(cell, x, h0, K, P, grad):
    """States, and with ``grad`` the function from dL/dstates to the gradients of x, the weights
    and h0."""
    ref = _SLSTM(cell) if isinstance(cell, ParaSLSTM) else _GRU(cell)
    if h0 is None:
        h0 = torch.zeros(x.shape[0], *ref.tail, dtype=torch.float64, device=x.device)
    with torch.no_grad():
        H = ref.solve(x, h0, K, P).to(ref.dtype).double()
    if grad is None:
        return H, None

    def backward(g):
        prev = _shift(H, h0)
        with torch.no_grad():
            nu = ref.adjoint(prev, x, g)
        mu = g + torch.cat((nu[:, 1:], torch.zeros_like(nu[:, :1])), 1)
        xr = x.detach().requires_grad_(True)
        weights = [ref.weights[n] for n, _ in cell.named_parameters()]
        gx, *gw = torch.autograd.grad(ref.f(prev, xr), [xr, *weights], mu)
        return gx, gw, nu[:, 0]

    return H, backward


def exact(case: dict, seed: int):
    s = prepare(case, seed)
    cell = s["cell"]
    x = s["x"].detach().double()
    if case["kind"] == "decode":
        ref = _SLSTM(cell) if case["cell"] == "slstm" else _GRU(cell)
        with torch.no_grad():
            return ref.f(s["state"].double().unsqueeze(1), x.unsqueeze(1))[:, 0]
    K = int(s["config"].max_iters)
    P = int(work_picard(case))
    cu = s["cu"]
    h0 = None if s["h0"] is None else s["h0"].detach().double()
    pad = (lambda v: v) if cu is None else (lambda v: _pad(v, cu))
    unpad = (lambda v: v) if cu is None else (lambda v: _unpad(v, cu))
    if case["kind"] == "infer":
        return unpad(_layer(cell, pad(x), h0, K, P, None)[0])
    g = pad(s["grad"].double())
    if case["kind"] == "train":
        H, backward = _layer(cell, pad(x), h0, K, P, True)
        gx, gw, gh0 = backward(g)
        return [unpad(H), unpad(gx), *gw] + ([] if h0 is None else [gh0])
    layers, cur = [], x
    for c in s["net"].layers:
        H, backward = _layer(c, cur, None, K, P, True)
        layers.append(backward)
        cur = H[..., 3, :]
    out, grads = cur, []
    for backward in reversed(layers):
        full = torch.zeros(*g.shape[:2], 4, g.shape[-1], dtype=torch.float64, device=g.device)
        full[..., 3, :] = g
        g, gw, _ = backward(full)
        grads = gw + grads
    return [out, g, *grads]


def work_picard(case: dict) -> int:
    """Picard passes of the warm start: none for the GRU; fixed, or by T (library default)."""
    if case["cell"] != "slstm":
        return 0
    if case["config"] == "fixed":
        return 5
    T = case.get("T", case.get("N"))
    return 1 if T <= 64 else 3 if T <= 2048 else 5
