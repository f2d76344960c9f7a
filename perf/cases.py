"""The workloads that a user of fermix_amd runs: batches of Slater determinants and
Pfaffians, as values (Monte Carlo sampling) and with gradients (training), through the
public calls slogdet / slogpf / det / pf and torch.autograd.

A case names the call ("op"), whether the gradient is taken ("grad"), the element type
("dtype"), the batch B, the order n and the options that the call takes: "prec" (None is
the default product mode) and "skew" (skew_symmetrize of slogpf / pf).
"""

import math

import torch

import fermix_amd

DTYPES = {"f32": torch.float32, "f64": torch.float64, "c64": torch.complex64, "c128": torch.complex128}


def _case(op, grad, dtype, B, n, prec=None, skew=True, name=None):
    c = {"op": op, "grad": grad, "dtype": dtype, "B": B, "n": n, "prec": prec, "skew": skew}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # a few walkers of a small system: one call's latency
        _case("slogdet", False, "f32", 16, 12, name="call_slogdet_16x12"),
        # Monte Carlo sampling, values only: the benchmark's two forward workloads
        _case("slogpf", False, "f32", 4096, 128, name="sample_slogpf_4096x128"),
        _case("slogdet", False, "f32", 4096, 128, name="sample_slogdet_4096x128"),
        # sums of many small determinants, det itself differentiated
        _case("det", True, "f32", 16384, 24, name="train_det_16384x24"),
        # training of a small system, an order that is no multiple of a tile
        _case("slogdet", True, "f32", 4096, 100, name="train_slogdet_4096x100"),
        _case("slogpf", True, "f32", 2000, 90, name="train_slogpf_2000x90"),
        # training of middle and large systems: the benchmark's two gradient workloads
        _case("slogdet", True, "f32", 1024, 512, name="train_slogdet_1024x512"),
        _case("slogpf", True, "f32", 64, 2048, name="train_slogpf_64x2048"),
        # double precision: a small and a middle order
        _case("slogdet", True, "f64", 2048, 63, name="train_slogdet_f64_2048x63"),
        _case("slogpf", True, "f64", 48, 302, skew=False, name="train_slogpf_f64_48x302"),
        # complex orbitals and pairing functions
        _case("slogdet", True, "c64", 1024, 100, name="train_slogdet_c64_1024x100"),
        _case("slogpf", False, "c128", 1024, 60, name="sample_slogpf_c128_1024x60"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# One row per use: calls, gradient, types, order range, batch range, largest B n^3.
_USES = [
    (("slogdet", "slogpf"), (False,), ("f32",), (4, 64), (1, 64), 2.0e7),
    (("slogdet", "slogpf"), (False,), ("f32",), (32, 256), (256, 8192), 8.6e9),
    (("det", "pf"), (True,), ("f32",), (4, 32), (1024, 32768), 1.0e9),
    (("slogdet", "slogpf"), (True,), ("f32",), (24, 128), (256, 4096), 8.6e9),
    (("slogdet", "slogpf"), (True,), ("f32",), (129, 1024), (4, 1024), 1.3e11),
    (("slogpf",), (True,), ("f32",), (1024, 2048), (4, 64), 4.0e11),
    (("slogdet", "slogpf"), (False, True), ("f64",), (16, 512), (16, 4096), 4.3e9),
    (("slogdet", "slogpf"), (False, True), ("c64", "c128"), (16, 256), (16, 2048), 2.2e9),
]


def draw(rng):
    ops, grads, dtypes, ns, Bs, most = rng.choice(_USES)
    op, dtype = rng.choice(ops), rng.choice(dtypes)
    n = _log_int(rng, *ns)
    if op in ("slogpf", "pf"):
        n += n % 2  # odd orders have no Pfaffian
    B = _log_int(rng, Bs[0], max(Bs[0], min(Bs[1], int(most / n**3))))
    prec = rng.choice((None, None, "ieee")) if dtype == "f32" and n > 128 else None
    skew = rng.random() < 0.7 or op in ("slogdet", "det")
    return _case(op, rng.choice(grads), dtype, B, n, prec, skew)


def _orbitals(n, pfaffian):
    """The n lowest standing waves on n sites (the orthogonal cosine matrix C), or for the
    Pfaffians the pairing C J C^T of neighbouring waves: dense, no entry dominates."""
    i = torch.arange(n, device="cuda", dtype=torch.float64)
    C = torch.cos((i[:, None] + 0.5) * i[None, :] * (math.pi / n)) * math.sqrt(2.0 / n)
    C[:, 0] /= math.sqrt(2.0)
    if not pfaffian:
        return C
    K = C[:, 0::2] @ C[:, 1::2].t().contiguous()
    return K - K.t()


def _inputs(case, seed):
    """(A, cotangent). Each member is 1.5 (Q + 0.5 G): Q the orbitals at n sites in a random
    order with random signs (phases), G dense N(0, 1/n) from the interaction. The pivoting
    has to search among entries of like size, and the condition number is about ten, so
    that values and gradients are determined to the type's precision. The cotangent is
    what a loss over the batch sends back."""
    B, n, dt = case["B"], case["n"], DTYPES[case["dtype"]]
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    pfaffian = case["op"] in ("slogpf", "pf")
    A = torch.randn(B, n, n, generator=gen, device="cuda", dtype=dt)
    A *= 0.5 / math.sqrt(n)
    order = torch.rand(B, n, generator=gen, device="cuda").argsort(1)
    phase = torch.randn(B, n, generator=gen, device="cuda", dtype=dt)
    phase /= phase.abs()
    Q = _orbitals(n, pfaffian).to(torch.float64 if case["dtype"] in ("f64", "c128") else torch.float32)
    Q = Q[order[:, :, None], order[:, None, :]] if pfaffian else Q[order]
    A += Q * phase[:, :, None] * (phase[:, None, :] if pfaffian else 1.0)
    A *= 1.5
    if pfaffian and not case["skew"]:
        A = (A - A.transpose(1, 2)) / 2  # exactly skew, as skew_symmetrize=False asks
    w = torch.rand(B, generator=gen, device="cuda", dtype=A.real.dtype) + 0.5
    return A.contiguous(), w


def prepare(case, seed):
    A, w = _inputs(case, seed)
    kw = {"prec": case["prec"]}
    if case["op"] in ("slogpf", "pf"):
        kw["skew_symmetrize"] = case["skew"]
    return {"f": getattr(fermix_amd, case["op"]), "A": A.requires_grad_(case["grad"]), "w": w, "kw": kw, "grad": case["grad"]}


def run(state):
    out = state["f"](state["A"], **state["kw"])
    sign, value = out if isinstance(out, tuple) else (None, out)
    got = {"value": value.detach()}
    if sign is not None:
        got["sign"] = sign.detach()
    if state["grad"]:
        (got["grad"],) = torch.autograd.grad(value, state["A"], state["w"])
    return got


def work(case):
    B, n = case["B"], case["n"]
    real, cplx = {"f32": (4, 1), "f64": (8, 1), "c64": (4, 2), "c128": (8, 2)}[case["dtype"]]
    pfaffian = case["op"] in ("slogpf", "pf")
    mats = 2 if case["grad"] else 1
    outs = real if case["op"] in ("det", "pf") else real * (1 + cplx)
    per = (1.0 if pfaffian else 2.0) if case["grad"] else (1.0 / 3 if pfaffian else 2.0 / 3)
    return {"bytes": B * (mats * n * n * real * cplx + outs), "flops": B * per * n**3 * cplx**2}


def tolerance(case):
    """About four times the measured relative error of each output against 64-bit results:
    float32 values 8e-8, the complex sign 3.3e-7, the Pfaffians' gradients 0.3-1.1e-6, the
    determinants' growing with the order (pivot growth of orthogonal matrices): 0.8e-6 at
    n = 24, 1.9e-6 at 100, 1.3e-5 at 430, 2.0e-5 at 512. The 64-bit types' are these times
    the ratio of the roundings (gradients 1.8e-15 at n = 63)."""
    unit = 1.0 if case["dtype"] in ("f32", "c64") else 2.0**-29
    rel = 4.0e-6 if case["dtype"].startswith("c") else 1.5e-6
    if case["grad"]:
        rel = 5.0e-6 if case["op"] in ("slogpf", "pf") else max(5.0e-6, 1.6e-7 * case["n"])
    return {"rel": rel * unit, "max": 100 * rel * unit}


def _parlett_reid(S):
    """(sign, log|pf|) of a batch of skew matrices in their own precision, with pivoting."""
    S = S.clone()
    B, n, _ = S.shape
    at = torch.arange(B, device=S.device)
    sign = torch.ones(B, dtype=S.dtype, device=S.device)
    logabs = torch.zeros(B, dtype=torch.float64, device=S.device)
    for k in range(0, n, 2):
        if k + 2 < n:
            p = k + 1 + S[:, k, k + 1 :].abs().argmax(1)
            row, own = S[at, p].clone(), S[:, k + 1].clone()
            S[:, k + 1] = row
            S[at, p] = own
            col, own = S[at, :, p].clone(), S[:, :, k + 1].clone()
            S[:, :, k + 1] = col
            S[at, :, p] = own
            sign = torch.where(p == k + 1, sign, -sign)
        d = S[:, k, k + 1].clone()
        sign, logabs = sign * d / d.abs(), logabs + d.abs().log()
        if k + 2 < n:
            t, v = S[:, k, k + 2 :] / d[:, None], S[:, k + 2 :, k + 1]
            L, R = torch.stack((t, -v), 2), torch.stack((v, t), 1)
            S[:, k + 2 :, k + 2 :] += torch.matmul(L, R.contiguous())
    return sign, logabs


def exact(case, seed):
    A, w = _inputs(case, seed)
    pfaffian = case["op"] in ("slogpf", "pf")
    log = case["op"] in ("slogdet", "slogpf")
    chunk = case["B"] if case["n"] <= 128 else 8  # torch's batched LU runs out of workspace above
    parts = []
    for a, wa in zip(A.split(chunk), w.split(chunk)):
        a, wa = a.to(torch.complex128 if a.is_complex() else torch.float64), wa.to(torch.float64)
        if pfaffian:
            a = (a - a.transpose(1, 2)) / 2 if case["skew"] else a
            sign, logabs = _parlett_reid(a)
        else:
            sign, logabs = torch.linalg.slogdet(a)
        got = {"value": logabs, "sign": sign} if log else {"value": sign * logabs.exp()}
        if case["grad"]:
            scale = wa if log else wa * got["value"]
            X = torch.linalg.inv(a).transpose(1, 2)
            got["grad"] = (0.5 if pfaffian else 1.0) * scale[:, None, None] * X.conj()
        parts.append(got)
    return {k: torch.cat([p[k] for p in parts]) for k in parts[0]}
