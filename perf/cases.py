"""The measured cases of the CPD-ALS library: the calls a user makes, over the sizes they make them at.

Every case goes through the Python binding (partensor-toolbox_amd/ptn_hip.py), host factors in, host
results out, on a handle whose tensor is already on the device, as a program that calls it keeps it:

  cpd       a whole decomposition (cpd / cpd_dimtree): initial factors to final factors and cost
  mttkrp    one MTTKRP of one mode
  tree      the N MTTKRPs of one dimension-tree sweep
  nnls      one NesterovMNLS solve
  batch     many small independent decompositions advanced together
  train     one epoch of the NNLS warm-start network on a training set held on the device
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "partensor-toolbox_amd"))
import ptn_hip as P  # noqa: E402

ARITH = {"f64": P.ARITH_F64, "f32": P.ARITH_F32, "bf16x3": P.ARITH_BF16X3, "f32_f64": P.ARITH_F32_F64}
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    return [
        # the smallest single call: latency of one FP64 MTTKRP on a tensor of a few tens per mode
        {"name": "mttkrp_37x23x41_r5", "op": "mttkrp", "dims": "37x23x41", "rank": 5, "mode": 1, "arith": "f64"},
        # the default path at the size the plain algorithm is quoted on, nothing divisible by anything
        {"name": "mttkrp_ragged_f64", "op": "mttkrp", "dims": "501x403x307", "rank": 33, "mode": 1, "arith": "f64"},
        # the largest FP64 call: the last mode of the headline tensor
        {"name": "mttkrp_800c_r32_f64", "op": "mttkrp", "dims": "800x800x800", "rank": 32, "mode": 2, "arith": "f64"},
        # an order-4 tensor, per-mode form, FP64: spectral data with two small modes
        {"name": "mttkrp_order4_f64", "op": "mttkrp", "dims": "190x155x61x24", "rank": 12, "mode": 2, "arith": "f64"},
        # the order-4 configuration with FP32 products
        {"name": "tree_200x4_r64_f32", "op": "tree", "dims": "200x200x200x200", "rank": 64, "arith": "f32"},
        # the split-product stream on a tensor whose fibres are not aligned
        {"name": "tree_ragged_bf16x3", "op": "tree", "dims": "701x555x333", "rank": 20, "arith": "bf16x3"},
        # the small configuration: 50 sweeps of 100^3, R = 10, the defaults of cpd()
        {"name": "cpd_100c_r10", "op": "cpd", "dims": "100x100x100", "rank": 10, "arith": "f64", "form": "standard",
         "fuse": False, "sweeps": 50, "cons": "111"},
        # the headline configuration in the form chosen for it, 30 sweeps
        {"name": "cpd_800c_r32_bf16x3", "op": "cpd", "dims": "800x800x800", "rank": 32, "arith": "bf16x3",
         "form": "tree", "fuse": True, "sweeps": 30, "cons": "111"},
        # mixed constraints (nonnegative, orthogonal, unconstrained) on a mid-size ragged tensor, 20 sweeps
        {"name": "cpd_constraints", "op": "cpd", "dims": "301x205x150", "rank": 24, "arith": "f64", "form": "tree",
         "fuse": False, "sweeps": 20, "cons": "120"},
        # one solve at the sizes of the 1000^3, R = 64 configuration
        {"name": "nnls_1000_r64", "op": "nnls", "rows": 1000, "rank": 64},
        # 512 uneven problems, modes 16 .. 128, ranks 4 .. 16, 20 sweeps, launch shape left to the library
        {"name": "batch_512", "op": "batch", "problems": 512, "sweeps": 20, "arith": "f32"},
        # an epoch of the warm-start network on the rows of a few runs
        {"name": "train_8192", "op": "train", "rows": 8192, "batch": 1024},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def dims_of(order, elements):
        # modes of uneven sizes whose product is about `elements`
        w = [rng.uniform(0.6, 1.4) for _ in range(order)]
        return [max(3, int(round(elements ** (x / sum(w))))) for x in w]

    op = rng.choice(["mttkrp", "mttkrp", "tree", "tree", "cpd", "cpd", "nnls", "batch", "train"])
    order = rng.choice([3, 3, 3, 4, 5])
    if op in ("mttkrp", "tree"):
        dims = dims_of(order, log_int(20000, 400000000))
        c = {"op": op, "dims": "x".join(map(str, dims)), "rank": rng.randint(2, 64),
             "arith": rng.choice(["f64", "f64", "f32", "bf16x3", "f32_f64"])}
        if op == "mttkrp":
            c["mode"] = rng.randrange(order)
        return c
    if op == "cpd":
        dims = dims_of(order, log_int(10000, 20000000))
        rank = rng.randint(2, min(32, min(dims)))
        arith = rng.choice(["f64", "f64", "f32", "bf16x3"])
        form = rng.choice(["standard", "tree"])
        cons = "1" * order if arith != "f64" or rng.random() < 0.6 else "".join(rng.choice("0112") for _ in dims)
        return {"op": op, "dims": "x".join(map(str, dims)), "rank": rank, "arith": arith, "form": form,
                "fuse": form == "tree" and arith != "f64" and rng.random() < 0.7, "sweeps": rng.randint(5, 25),
                "cons": cons}
    if op == "nnls":
        return {"op": op, "rows": log_int(30, 20000), "rank": rng.randint(3, 64)}
    if op == "batch":
        return {"op": op, "problems": log_int(8, 600), "sweeps": rng.randint(5, 25), "arith": rng.choice(["f64", "f32"])}
    batch = 32 * rng.randint(2, 64)
    return {"op": op, "rows": batch * rng.randint(2, 8), "batch": batch}


# ------------------------------------------------------------------ inputs

def _dims(case):
    return [int(v) for v in case["dims"].split("x")]


def _rand(case, seed, salt):
    return np.random.default_rng([seed % (1 << 31), salt, case.get("rank", 0)])


def _noisy_tensor(case, seed):
    """[[A]] plus Gaussian noise at 20 dB, FP64 on the torch device, axis k = mode k (mode 0 contiguous).  A mode's
    factor is what its constraint describes: U[0,1) where it is nonnegative, Gaussian columns where it is free,
    orthonormal ones where it is orthogonal."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed % (1 << 31))
    dims, R = _dims(case), case["rank"]
    A = []
    for I, c in zip(dims, case["cons"]):
        draw_k = torch.rand if c == "1" else torch.randn
        a = draw_k(I, R, dtype=torch.float64, device=DEV, generator=g)
        A.append(torch.linalg.qr(a)[0] if c == "2" else a)
    left = A[-1]
    for k in range(len(dims) - 2, 0, -1):
        left = (left[:, None, :] * A[k][None, :, :]).reshape(-1, R)
    X = (left @ A[0].T).reshape(dims[::-1])
    E = torch.randn(X.shape, dtype=torch.float64, device=DEV, generator=g)
    X = X + E * (X.norm() / E.norm() * 0.1)
    return X.permute(*range(len(dims) - 1, -1, -1))


def _start_factors(case, seed):
    r = _rand(case, seed, 1)
    free = [c != "1" for c in case.get("cons", "1" * len(_dims(case)))]
    return [r.standard_normal((I, case["rank"])) if f else r.random((I, case["rank"])) for I, f in zip(_dims(case), free)]


def _nnls_inputs(case, seed):
    r = _rand(case, seed, 2)
    I, R = case["rows"], case["rank"]
    B, C = r.random((I, R)), r.random((I, R))
    Z = (B.T @ B) * (C.T @ C) / I
    true = np.maximum(r.random((I, R)) - 0.2, 0.0)
    return Z, true @ Z + 0.01 * r.standard_normal((I, R)), r.random((I, R))


def _batch_shapes(case, seed):
    r = np.random.default_rng([3, case["problems"]])    # the sizes of the batch; the seed makes its values
    dims = r.integers(16, 129, (case["problems"], 3))
    ranks = r.integers(4, 17, case["problems"])
    return [tuple(int(v) for v in d) for d in dims], [int(v) for v in ranks]


def _training_rows(case, seed):
    """Rows (features, scaled solution, rank) of NNLS updates at ranks 8 .. 64, 256 rows to a Gram matrix."""
    r = _rand(case, seed, 4)
    n = case["rows"]
    X = np.zeros((n, P.MLP_IN), dtype=np.float32)
    T = np.zeros((n, P.MLP_OUT), dtype=np.float32)
    rank = np.zeros(n, dtype=np.uint8)
    upper = np.triu_indices(64)
    for a in range(0, n, 256):
        b, R = min(n, a + 256), int(r.integers(8, 65))
        F = r.random((128, R))
        V = np.zeros((64, 64))
        V[:R, :R] = (F.T @ F) ** 2 / 128
        sv = V.diagonal().max()
        sol = np.maximum(r.random((b - a, R)) - 0.1, 0.0)
        M = sol @ V[:R, :R]
        sm = M.max(axis=1, keepdims=True)
        X[a:b, :2080] = V[upper] / sv
        X[a:b, 2080:2080 + R] = M / sm
        X[a:b, 2144:2144 + R] = (sol + 0.05 * r.standard_normal(sol.shape)) * sv / sm
        T[a:b, :R] = sol * sv / sm
        rank[a:b] = R
    return X, T, rank


def _start_weights(case, seed):
    r = _rand(case, seed, 5)
    w = np.zeros(P.MLP_PARAMS, dtype=np.float32)
    at = 0
    for rows, cols in ((256, 2208), (256, 256), (64, 256)):
        w[at:at + rows * cols] = r.uniform(-1, 1, rows * cols) * math.sqrt(6.0 / cols)
        at += rows * cols + rows
    return w


def _generated(case):
    """The largest tensors come from the library's own generator, the others from host data."""
    return case["op"] in ("mttkrp", "tree") or math.prod(_dims(case)) > 50000000


def prepare(case, seed):
    op, h = case["op"], P.Handle(0)
    s = {"case": case, "h": h}
    if op in ("mttkrp", "tree", "cpd"):
        dims = _dims(case)
        store = P.TENSOR_F64 if case["arith"] == "f64" else P.TENSOR_F32
        if not _generated(case):
            h.set_tensor(_noisy_tensor(case, seed).cpu().numpy(), storage=store)
        else:
            h.generate_tensor(dims, case["rank"], seed=seed, snr_db=20.0 if op == "cpd" else None, storage=store)
        s["factors"] = _start_factors(case, seed)
        if op == "cpd":
            s["options"] = P.default_options(
                max_iter=case["sweeps"], threshold_error=0.0, arith=ARITH[case["arith"]],
                mttkrp_form=P.MTTKRP_DIMTREE if case["form"] == "tree" else P.MTTKRP_STANDARD,
                fuse_accel=int(case["fuse"]), constraints=[int(v) for v in case["cons"]])
    elif op == "nnls":
        s["inputs"] = _nnls_inputs(case, seed)
    elif op == "batch":
        dims, ranks = _batch_shapes(case, seed)
        h.batch_generate(dims, ranks, seed=seed, snr_db=25.0)
        s["factors"] = h.batch_init_factors(seed=seed + 1000)
    else:
        h.mlp_init(0)
        h.mlp_data_add(*_training_rows(case, seed))
        s["weights"] = _start_weights(case, seed)
    return s


def run(s):
    case, h = s["case"], s["h"]
    op = case["op"]
    if op == "mttkrp":
        return h.mttkrp(s["factors"], case["mode"], arith=ARITH[case["arith"]])
    if op == "tree":
        return h.mttkrp_dimtree(s["factors"], arith=ARITH[case["arith"]])
    if op == "cpd":
        F, st, _ = h.cpd(case["rank"], s["factors"], options=s["options"])
        return {"factors": F, "f_value": st["f_value"], "rel_cost": st["rel_cost"], "ao_iter": st["ao_iter"]}
    if op == "nnls":
        A, it, L, mu = h.nesterov(*s["inputs"])
        return {"A": A, "iters": it, "L": L, "mu": mu}
    if op == "batch":
        F, st, _, _ = h.cpd_batch(s["factors"], max_iter=case["sweeps"], arith=ARITH[case["arith"]], with_log=False)
        return {"factors": np.concatenate([P.pack(f) for f in F]), "f_value": np.array([v["f_value"] for v in st]),
                "ao_iter": np.array([v["ao_iter"] for v in st])}
    # from given weights, so that a pass can be repeated
    h.mlp_set_params(s["weights"])
    loss = h.mlp_train(1, batch=case["batch"], lr=1e-3, seed=7)
    return {"loss": loss, "weights": h.mlp_params()}


def work(case):
    op = case["op"]
    if op in ("mttkrp", "tree", "cpd"):
        dims, R = _dims(case), case["rank"]
        n, rows = math.prod(dims), sum(dims)
        size = 8 if case["arith"] == "f64" else 4
        if op == "mttkrp":
            return {"bytes": size * n + 8.0 * R * rows, "flops": 2.0 * R * n}
        if op == "tree":                       # two children of the root, from one reading of the tensor
            return {"bytes": size * n + 16.0 * R * rows, "flops": 4.0 * R * n}
        k = case["sweeps"]                     # two children a sweep, each after the other's factors change
        return {"bytes": 2.0 * k * size * n + 16.0 * R * rows, "flops": 4.0 * k * R * n}
    if op == "nnls":
        I, R = case["rows"], case["rank"]
        return {"bytes": 8.0 * (3 * I * R + R * R), "flops": 2.0 * 50 * I * R * R}
    if op == "batch":
        dims, ranks = _batch_shapes(case, 0)
        el = [math.prod(d) for d in dims]
        return {"bytes": 2.0 * 4 * case["sweeps"] * sum(el),
                "flops": 4.0 * case["sweeps"] * sum(r * e for r, e in zip(ranks, el))}
    n = case["rows"] // case["batch"] * case["batch"]
    return {"bytes": n * (2.0 * P.MLP_IN + 4 * P.MLP_OUT + 1) + 8.0 * P.MLP_PARAMS, "flops": 6.0 * n * P.MLP_PARAMS}


# ------------------------------------------------------------------ the same in 64 bits, without the library

def _philox_uniform(seed, n):
    """The generator's U[0,1) draws 0 .. n-1: Philox4x32-10 on the counter (index, stream 0), the top 53 bits of the
    first two words."""
    i = np.arange(n, dtype=np.uint64)
    low = np.uint64(0xFFFFFFFF)
    c = [i & low, i >> np.uint64(32), np.zeros(n, np.uint64), np.zeros(n, np.uint64)]
    k0, k1 = seed & 0xFFFFFFFF, seed >> 32
    for _ in range(10):
        p0, p1 = np.uint64(0xD2511F53) * c[0], np.uint64(0xCD9E8D57) * c[2]
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k0), p1 & low, (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k1),
             p0 & low]
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    return (((c[1] << np.uint64(32)) | c[0]) >> np.uint64(11)).astype(np.float64) * 2.0 ** -53


def _closed_mttkrp(case, seed):
    """Every mode's MTTKRP of X = [[B]] with factors A: B_n (Hadamard over k != n of B_k^T A_k)."""
    dims, R = _dims(case), case["rank"]
    flat, at, B = _philox_uniform(seed, sum(dims) * R), 0, []
    for I in dims:
        B.append(flat[at:at + I * R].reshape((I, R), order="F"))
        at += I * R
    A = _start_factors(case, seed)
    return [B[n] @ np.prod([B[k].T @ A[k] for k in range(len(dims)) if k != n], axis=0) for n in range(len(dims))]


def _nnls(Z, W, A):
    """Nesterov's projected gradient on min 1/2 <A Z, A> - <W, A> + lambda/2 |A - A0|^2, A >= 0, at most 50 steps."""
    ev = torch.linalg.eigvalsh(Z).abs()
    L, mu = float(ev.max()), float(ev.min())
    q = mu / L
    lam = 10.0 * mu if 1.0 / q > 1e6 else mu if 1.0 / q > 1e3 else mu / 10.0
    Lt = L + lam
    q = (mu + lam) / Lt
    Zt = Z + lam * torch.eye(Z.shape[0], dtype=Z.dtype, device=Z.device)
    Wt = W + lam * A
    Y, alpha, it = A, 1.0, 0
    while True:
        G = Y @ Zt - Wt
        if it >= 50 or (float((G * Y).abs().max()) <= 1e-2 and float(G.min()) >= -1e-2):
            return A, it, L, mu
        new = (Y - G / Lt).clamp(min=0.0)
        b = alpha * alpha - q
        nxt = (-b + math.sqrt(b * b + 4.0 * alpha * alpha)) / 2.0
        beta = alpha * (1.0 - alpha) / (alpha * alpha + nxt)
        Y, A, alpha, it = (1.0 + beta) * new - beta * A, new, nxt, it + 1


def _mttkrp(X, A, n):
    k = max((j for j in range(len(A)) if j != n), key=lambda j: A[j].shape[0])
    Y = torch.tensordot(X, A[k], dims=([k], [0]))            # the other modes in order, then the columns
    left = [j for j in range(len(A)) if j != k]
    for j in [j for j in left if j != n]:
        ax = left.index(j)
        shape = [1] * Y.dim()
        shape[ax], shape[-1] = A[j].shape
        Y = (Y * A[j].reshape(shape)).sum(ax)
        left.pop(ax)
    return Y


def _had(G, skip):
    V = None
    for k, g in enumerate(G):
        if k != skip:
            V = g if V is None else V * g
    return V


def _als(X, A, sweeps, cons):
    """cpd() with its defaults: per-mode updates, the Gram-form cost, Normalize and the line search."""
    N = len(A)
    G = [a.T @ a for a in A]
    frob = float((X * X).sum())
    wf = next((k for k in range(N) if cons[k] != 2), None)
    coeff, fail, old, f = 3, 0, None, 0.0
    for it in range(1, sweeps + 1):
        for n in range(N):
            M, V = _mttkrp(X, A, n), _had(G, n)
            if cons[n] == 1:
                new = _nnls(V, M, A[n])[0]
                A[n] = 0.9 * new + 0.1 * A[n] if float(new.abs().sum(0).min()) == 0.0 else new
            elif cons[n] == 0:
                A[n] = M @ torch.linalg.inv(V)
            else:
                ev, Q = torch.linalg.eigh(M.T @ M)
                A[n] = M @ ((Q / ev.sqrt()) @ Q.T)
            G[n] = A[n].T @ A[n]
        f = math.sqrt(frob - 2.0 * float((M * A[-1]).sum()) + float((V * G[-1]).sum()))
        sweep_f = f
        if wf is not None:
            # every factor but the weight factor and the last to unit columns; the norms are read from the list of
            # the factors other than the weight factor
            rest = [G[k].diagonal().sqrt() for k in range(N) if k != wf]
            on = rest[N - 2] != 0
            scale, gain, used = {}, torch.ones_like(rest[0]), 0
            for j in range(N - 1):
                if j != wf:
                    s = torch.where(on, rest[used], torch.ones_like(rest[used]))
                    scale[j], gain, used = s, gain * s, used + 1
            for j, s in scale.items():
                A[j] = A[j] / s
                G[j] = G[j] / torch.outer(s, s)
            A[wf] = A[wf] * gain
            G[wf] = G[wf] * torch.outer(gain, gain)
        if it == sweeps:
            break
        kept = [a.clone() for a in A]
        if it > 1:
            step = (it + 1.0) ** (1.0 / coeff)
            B = [o + step * (a - o) for o, a in zip(old, A)]
            H = [b.T @ b for b in B]
            fa = frob + float((_had(H, N - 1) * H[-1]).sum()) - 2.0 * float((_mttkrp(X, B, N - 1) * B[-1]).sum())
            fa = math.sqrt(fa) if fa >= 0 else math.nan
            if f > fa:
                A, G, f = B, H, fa
            else:
                fail += 1
            if fail == 5:
                fail, coeff = 0, coeff + 1
        old = kept
    return A, f, sweep_f / math.sqrt(frob)


def exact(case, seed):
    op = case["op"]
    if op == "mttkrp":
        return _closed_mttkrp(case, seed)[case["mode"]]
    if op == "tree":
        return _closed_mttkrp(case, seed)
    if op == "nnls":
        A, it, L, mu = _nnls(*(torch.from_numpy(v).to(DEV) for v in _nnls_inputs(case, seed)))
        return {"A": A.cpu().numpy(), "iters": it, "L": L, "mu": mu}
    if op == "cpd" and not _generated(case):
        # an FP64 run; with an FP32 stream the line search may decide otherwise where two costs are close
        A = [torch.from_numpy(a).to(DEV) for a in _start_factors(case, seed)]
        F, f, rel = _als(_noisy_tensor(case, seed), A, case["sweeps"], [int(v) for v in case["cons"]])
        return {"factors": [a.cpu().numpy() for a in F], "f_value": f, "rel_cost": rel, "ao_iter": case["sweeps"]}
    # the headline run's tensor exists on the device only; hundreds of small runs take too long one after another;
    # the network's weights and activations are bfloat16 by definition
    return None
