"""What this library's users have it do, as cases that can be timed and checked.

Each case is one call (or the few calls that belong together) through the C
ABI of libzt_attn.so, on device buffers the caller owns, as a native program
makes them: a training step's attention, the two reference entry points, a
chunk of a prefill, a decode over a batch of caches, one decode step with its
cache append, and the norm / projections / RoPE that surround the attention in
a block, forward and backward.  Shapes are the repository's own benchmark and
test shapes, or generic odd ones of the same ranges.
"""
import ctypes
import importlib.util
import math
import os

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
THETA = 500000.0
EPS = 1e-5


def _binding():
    spec = importlib.util.spec_from_file_location("zt_attn", os.path.join(ROOT, "z-transformer_amd", "zt_attn.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


zt = _binding()

# (query heads, kv heads, head width): GPT-mini's, the MHA shape, the grouped
# 128-wide and 96-wide ones, the wide-head ones, and a group of three.
HEADS = [(4, 2, 32), (8, 8, 64), (32, 8, 128), (32, 8, 96), (16, 4, 256), (16, 16, 192), (12, 4, 64)]
MAX_UNITS = 32 * 128 * 4096 * 4096  # B H d T^2 of the largest training step below


def listed():
    return [
        # The small model's block at its own context (256 x 128): every launch is a few microseconds.
        dict(name="mini_block", kind="block", T=256, model=128, H=4, Hkv=2, d=32),
        # Its training step's attention.
        dict(name="mini_train", kind="train", B=1, T=256, H=4, Hkv=2, d=32, sigma=1.0),
        # The same model on a long context: few heads, many rows.
        dict(name="mini_train_long", kind="train", B=1, T=4096, H=4, Hkv=2, d=32, sigma=1.0),
        # A grouped 128-wide layer on a short sequence.
        dict(name="gqa128_train_short", kind="train", B=1, T=512, H=32, Hkv=8, d=128, sigma=1.0),
        # Multi-head attention, a small batch of medium sequences.
        dict(name="mha64_train", kind="train", B=4, T=1024, H=8, Hkv=8, d=64, sigma=1.0),
        # The headline training step.
        dict(name="gqa128_train", kind="train", B=1, T=4096, H=32, Hkv=8, d=128, sigma=1.0),
        # Wide heads and a wide range of scores.
        dict(name="gqa256_train", kind="train", B=2, T=2048, H=16, Hkv=4, d=256, sigma=math.sqrt(2.0)),
        # The reference's own two entry points (no saved statistics), an odd length.
        dict(name="gqa96_stateless_odd", kind="stateless", B=1, T=501, H=32, Hkv=8, d=96, sigma=1.0),
        # A chunk of a prompt against a partly filled cache.
        dict(name="prefill_chunk", kind="prefill", B=1, T=333, offset=2007, H=32, Hkv=8, d=128),
        # Serving: 64 sequences of different lengths over 8192-row caches.
        dict(name="decode_batch", kind="decode", B=64, n_ctx=8192, spread=4096, H=32, Hkv=8, d=128),
        # One sequence's decode step with RoPE and the cache append.
        dict(name="decode_step_one", kind="step", B=1, n_ctx=4096, spread=1095, H=32, Hkv=8, d=128),
        # A large block's norm, projections and RoPE, forward and backward.
        dict(name="large_block", kind="block", T=2048, model=4096, H=32, Hkv=8, d=128),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "stateless", "prefill", "decode", "step", "block"])
    if kind == "block":
        H, Hkv, d = rng.choice([(4, 2, 32), (32, 8, 128), (12, 4, 64), (16, 4, 256)])
        model = H * d
        T = _log_int(rng, 32, 2048)
        return dict(kind=kind, T=T, model=model, H=H, Hkv=Hkv, d=d)
    H, Hkv, d = rng.choice(HEADS)
    if kind in ("train", "stateless"):
        B = rng.choice([1, 1, 2, 4])
        T = _log_int(rng, 33, 4096)
        while B * H * d * T * T > MAX_UNITS or (kind == "stateless" and B * H * d * T * T * 3 > MAX_UNITS):
            T = T * 3 // 4
        return dict(kind=kind, B=B, T=T, H=H, Hkv=Hkv, d=d, sigma=rng.choice([1.0, 1.0, math.sqrt(2.0)]))
    if kind == "prefill":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), T=_log_int(rng, 8, 1024), offset=rng.randrange(0, 4096), H=H,
                    Hkv=Hkv, d=d)
    B = _log_int(rng, 1, 64) if kind == "decode" else _log_int(rng, 1, 16)
    n_ctx = _log_int(rng, 256, 8192)
    while B * n_ctx * Hkv * d > 64 * 8192 * 8 * 128:
        n_ctx = n_ctx * 3 // 4
    return dict(kind=kind, B=B, n_ctx=n_ctx, spread=rng.randrange(0, n_ctx), H=H, Hkv=Hkv, d=d)


def _n_keys(case):
    """Visible rows of each sequence: spread below n_ctx, the same for every seed."""
    n_ctx, spread = case["n_ctx"], case["spread"]
    return [n_ctx - (spread * ((i * 37) % 64 + 1) // 64 if spread else 0) for i in range(case["B"])]


def _normal(gen, n, sigma=1.0):
    return torch.randn(n, device="cuda", dtype=torch.float32, generator=gen) * sigma


def _inputs(case, seed):
    """The case's input tensors, from the seed alone."""
    gen = torch.Generator(device="cuda").manual_seed(1000003 * seed + 12345)
    kind = case["kind"]
    H, Hkv, d = case["H"], case["Hkv"], case["d"]
    if kind in ("train", "stateless"):
        n, s = case["B"] * case["T"], case["sigma"]
        return dict(q=_normal(gen, n * H * d, s), k=_normal(gen, n * Hkv * d, s), v=_normal(gen, n * Hkv * d, s),
                    dout=_normal(gen, n * H * d))
    if kind == "prefill":
        n_keys = case["offset"] + case["T"]
        return dict(q=_normal(gen, case["B"] * case["T"] * H * d), k=_normal(gen, case["B"] * n_keys * Hkv * d),
                    v=_normal(gen, case["B"] * n_keys * Hkv * d))
    if kind in ("decode", "step"):
        rows = case["B"] * case["n_ctx"]
        x = dict(q=_normal(gen, case["B"] * H * d), kc=_normal(gen, rows * Hkv * d), vc=_normal(gen, rows * Hkv * d))
        if kind == "step":
            x.update(k_new=_normal(gen, case["B"] * Hkv * d), v_new=_normal(gen, case["B"] * Hkv * d))
        return x
    # block: activations, a gain near 1, fan-in scaled weights, and the gradients that arrive from the attention.
    T, m = case["T"], case["model"]
    s = 1.0 / math.sqrt(m)
    return dict(x=_normal(gen, T * m), g=torch.rand(m, device="cuda", generator=gen) + 0.5,
                wq=_normal(gen, m * H * d, s), wk=_normal(gen, m * Hkv * d, s), wv=_normal(gen, m * Hkv * d, s),
                dq=_normal(gen, T * H * d), dk=_normal(gen, T * Hkv * d), dv=_normal(gen, T * Hkv * d))


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _call(fn, *args):
    rc = fn(*args, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    if rc != 0:
        raise RuntimeError("the library refused a call")


def prepare(case, seed):
    L = zt.lib()
    kind = case["kind"]
    H, Hkv, d = case["H"], case["Hkv"], case["d"]
    x = _inputs(case, seed)
    calls, out = [], {}

    def buf(n):
        return torch.empty(n, device="cuda", dtype=torch.float32)

    keep = dict(x)
    if kind in ("train", "stateless"):
        B, T = case["B"], case["T"]
        out = dict(out=buf(B * T * H * d), dq=buf(B * T * H * d), dk=buf(B * T * Hkv * d), dv=buf(B * T * Hkv * d))
        shape = (B, T, H, Hkv, d)
        if kind == "train":
            out["lse"] = buf(B * T * H)
            nbytes = L.zt_attn_backward_train_workspace(*shape)
            keep["ws"] = ws = torch.empty(nbytes, device="cuda", dtype=torch.uint8)
            calls.append((L.zt_attn_forward_train_ws, _p(x["q"]), _p(x["k"]), _p(x["v"]), _p(out["out"]),
                          _p(out["lse"]), _p(ws), nbytes, *shape))
            calls.append((L.zt_attn_backward_train_ws, _p(x["q"]), _p(x["k"]), _p(x["v"]), _p(out["out"]),
                          _p(x["dout"]), _p(out["lse"]), _p(out["dq"]), _p(out["dk"]), _p(out["dv"]), _p(ws), nbytes,
                          *shape, 3 | zt.ZT_WS_SCORES))
        else:
            rows = keep["rows"] = [buf(B * T * H) for _ in range(3)]
            calls.append((L.zt_attn_forward_batched, _p(x["q"]), _p(x["k"]), _p(x["v"]), _p(out["out"]), B, T, H, Hkv,
                          d, 1, 64, 0, T, T))
            calls.append((L.zt_attn_backward_batched, _p(x["q"]), _p(x["k"]), _p(x["v"]), _p(x["dout"]),
                          _p(out["dq"]), _p(out["dk"]), _p(out["dv"]), *map(_p, rows), B, T, H, Hkv, d, 64))
    elif kind == "prefill":
        B, T, n_keys = case["B"], case["T"], case["offset"] + case["T"]
        out = dict(out=buf(B * T * H * d))
        calls.append((L.zt_attn_forward_batched, _p(x["q"]), _p(x["k"]), _p(x["v"]), _p(out["out"]), B, T, H, Hkv, d,
                      1, 64, case["offset"], n_keys, n_keys))
    elif kind in ("decode", "step"):
        B, n_ctx = case["B"], case["n_ctx"]
        n_keys = _n_keys(case)
        out = dict(out=buf(B * H * d))
        if kind == "decode":
            nbytes = L.zt_attn_decode_workspace(B, n_ctx, H, Hkv, d)
            keep["n"] = n = (ctypes.c_int * B)(*n_keys)
            keep["ws"] = ws = torch.empty(nbytes, device="cuda", dtype=torch.uint8)
            calls.append((L.zt_attn_decode, _p(x["q"]), _p(x["kc"]), _p(x["vc"]), _p(out["out"]), n, B, n_ctx, H, Hkv,
                          d, _p(ws), nbytes))
        else:
            nbytes = L.zt_attn_decode_step_workspace(B, n_ctx, H, Hkv, d)
            keep["n"] = n = (ctypes.c_int * B)(*[k - 1 for k in n_keys])
            keep["ws"] = ws = torch.empty(nbytes, device="cuda", dtype=torch.uint8)
            out.update(kc=x["kc"], vc=x["vc"])  # the caches, one row per sequence appended
            calls.append((L.zt_attn_decode_step, _p(x["q"]), _p(x["k_new"]), _p(x["v_new"]), _p(x["kc"]), _p(x["vc"]),
                          _p(out["out"]), n, B, n_ctx, H, Hkv, d, THETA, _p(ws), nbytes))
    else:
        T, m, nq, nk = case["T"], case["model"], H * d, Hkv * d
        out = dict(xn=buf(T * m), q=buf(T * nq), k=buf(T * nk), v=buf(T * nk))
        # One flat gradient buffer, cleared once a step as a training loop does, since the products add into it.
        sizes = dict(gx=T * m, gwq=m * nq, gwk=m * nk, gwv=m * nk)
        keep["grads"] = grads = buf(sum(sizes.values()))
        out.update(zip(sizes, torch.split(grads, list(sizes.values()))))
        keep["dqr"], keep["dkr"] = dqr, dkr = buf(T * nq), buf(T * nk)
        calls.append((L.zt_rmsnorm_forward, _p(x["x"]), _p(x["g"]), _p(out["xn"]), T, m, EPS))
        for w, y, n in (("wq", "q", nq), ("wk", "k", nk), ("wv", "v", nk)):
            calls.append((L.zt_matmul, _p(out["xn"]), _p(x[w]), _p(out[y]), T, m, n))
        calls.append((L.zt_rope_qk_forward, _p(out["q"]), _p(out["k"]), _p(out["q"]), _p(out["k"]), 1, T, H, Hkv, d, 0,
                      THETA))
        calls.append((L.zt_rope_qk_backward, _p(x["dq"]), _p(x["dk"]), _p(dqr), _p(dkr), 1, T, H, Hkv, d, 0, THETA))
        for w, dy, gw, n in (("wq", dqr, "gwq", nq), ("wk", dkr, "gwk", nk), ("wv", x["dv"], "gwv", nk)):
            calls.append((L.zt_weight_grad, _p(out[gw]), _p(out["xn"]), _p(dy), T, m, n))
            calls.append((L.zt_input_grad, _p(out["gx"]), _p(dy), _p(x[w]), T, n, m))
    return dict(calls=calls, out=out, keep=keep)


def run(state):
    grads = state["keep"].get("grads")
    if grads is not None:
        grads.zero_()
    for call in state["calls"]:
        _call(*call)
    return state["out"]


def work(case):
    kind = case["kind"]
    H, Hkv, d = case["H"], case["Hkv"], case["d"]
    if kind in ("train", "stateless"):
        B, T = case["B"], case["T"]
        unit = B * H * d * T * (T + 1)  # one causal T x T x d product
        rows, kv = B * T * H * d, B * T * Hkv * d
        # q, k, v, dO read, O, dq, dk, dv written (and each row's log-sum-exp).
        return dict(bytes=4 * (4 * rows + 4 * kv + (B * T * H if kind == "train" else 0)), flops=7 * unit)
    if kind == "prefill":
        B, T, off = case["B"], case["T"], case["offset"]
        pairs = T * off + T * (T + 1) // 2
        return dict(bytes=4 * B * (2 * T * H * d + 2 * (off + T) * Hkv * d), flops=4 * B * H * d * pairs)
    if kind in ("decode", "step"):
        keys, B = sum(_n_keys(case)), case["B"]
        extra = 4 * B * Hkv * d if kind == "step" else 0  # the new key and value read and appended
        return dict(bytes=4 * (2 * keys * Hkv * d + 2 * B * H * d + extra), flops=4 * H * d * keys)
    T, m, n = case["T"], case["model"], (H + 2 * Hkv) * d
    # x, the gain, the weights and the three gradients in; xn, q, k, v, the input and weight gradients out.
    return dict(bytes=4 * (T * m + m + m * n + T * n + T * m + T * n + T * m + m * n), flops=3 * 2 * T * m * n)


def tolerance(case):
    # f32 inputs, products and sums: about four times the largest difference from 64-bit sums that was measured over
    # the listed shapes and drawn ones (1.3e-6 for the training steps, whose wide range of scores at d = 256 is the
    # worst, 9.3e-7 for a prefill, 5.1e-7 and 2.3e-7 for the decodes, 1.1e-6 for products over 4096).
    return {"train": {"rel": 5e-6}, "stateless": {"rel": 5e-6}, "prefill": {"rel": 4e-6}, "decode": {"rel": 2e-6},
            "step": {"rel": 1.5e-6}, "block": {"rel": 4.5e-6}}[case["kind"]]


def _rope64(x, pos, sign=1.0):
    """Rotates x [rows, heads, d] at the rows' positions, column i paired with column i + d / 2."""
    half = x.shape[-1] // 2
    i = torch.arange(half, device=x.device, dtype=torch.float64)
    ang = pos.to(torch.float64)[:, None] / THETA ** (i / half)[None, :]
    c, s = torch.cos(ang)[:, None, :], sign * torch.sin(ang)[:, None, :]
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def exact(case, seed):
    kind = case["kind"]
    H, Hkv, d = case["H"], case["Hkv"], case["d"]
    g = H // Hkv
    scale = 1.0 / math.sqrt(d)
    x = {n: t.double() for n, t in _inputs(case, seed).items()} if kind != "decode" else _inputs(case, seed)
    if kind in ("train", "stateless", "prefill"):
        B, T, off = case["B"], case["T"], case.get("offset", 0)
        S = off + T
        q, k, v = x["q"].view(B, T, H, d), x["k"].view(B, S, Hkv, d), x["v"].view(B, S, Hkv, d)
        keys, rows = torch.arange(S, device="cuda"), torch.arange(T, device="cuda") + off
        mask = keys[None, :] > rows[:, None]
        o = torch.empty_like(q)
        lse = torch.empty(B, T, H, device="cuda", dtype=torch.float64)
        if kind != "prefill":
            do = x["dout"].view(B, T, H, d)
            dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
        for b in range(B):
            for h in range(H):
                qh = q[b, :, h].contiguous()
                kh, vh = k[b, :, h // g].contiguous(), v[b, :, h // g].contiguous()
                s = (qh @ kh.t().contiguous()) * scale
                s.masked_fill_(mask, -math.inf)
                l = torch.logsumexp(s, 1)
                p = torch.exp(s - l[:, None])
                del s
                oh = p @ vh
                o[b, :, h], lse[b, :, h] = oh, l
                if kind != "prefill":
                    doh = do[b, :, h].contiguous()
                    ds = p * (doh @ vh.t().contiguous() - (doh * oh).sum(1, keepdim=True))
                    dq[b, :, h] = (ds @ kh) * scale
                    dk[b, :, h // g] += (ds.t().contiguous() @ qh) * scale
                    dv[b, :, h // g] += p.t().contiguous() @ doh
                    del ds
                del p
        if kind == "prefill":
            return dict(out=o.flatten())
        y = dict(out=o.flatten(), dq=dq.flatten(), dk=dk.flatten(), dv=dv.flatten())
        if kind == "train":
            y["lse"] = lse.flatten()
        return y
    if kind in ("decode", "step"):
        B, n_ctx, n_keys = case["B"], case["n_ctx"], _n_keys(case)
        q, kc, vc = x["q"].view(B, H, d), x["kc"].view(B, n_ctx, Hkv, d), x["vc"].view(B, n_ctx, Hkv, d)
        if kind == "step":
            pos = torch.tensor([n - 1 for n in n_keys], device="cuda")
            q = _rope64(q, pos)
            at = torch.arange(B, device="cuda")
            kc[at, pos] = _rope64(x["k_new"].view(B, Hkv, d), pos)
            vc[at, pos] = x["v_new"].view(B, Hkv, d)
        o = torch.empty(B, H, d, device="cuda", dtype=torch.float64)
        for b in range(B):
            for j in range(Hkv):
                kk, vv = kc[b, :n_keys[b], j].double().contiguous(), vc[b, :n_keys[b], j].double().contiguous()
                qq = q[b, j * g:(j + 1) * g].double()
                o[b, j * g:(j + 1) * g] = torch.softmax((qq @ kk.t().contiguous()) * scale, 1) @ vv
        y = dict(out=o.flatten())
        if kind == "step":
            y.update(kc=kc.flatten(), vc=vc.flatten())
        return y
    T, m = case["T"], case["model"]
    xx = x["x"].view(T, m)
    xn = xx / torch.sqrt((xx * xx).mean(1, keepdim=True) + EPS) * x["g"]
    w = {n: x[n].view(m, -1) for n in ("wq", "wk", "wv")}
    pos = torch.arange(T, device="cuda")
    y = dict(xn=xn.flatten(), q=_rope64((xn @ w["wq"]).view(T, H, d), pos).flatten(),
             k=_rope64((xn @ w["wk"]).view(T, Hkv, d), pos).flatten(), v=(xn @ w["wv"]).flatten())
    dq = _rope64(x["dq"].view(T, H, d), pos, -1.0).reshape(T, H * d)
    dk = _rope64(x["dk"].view(T, Hkv, d), pos, -1.0).reshape(T, Hkv * d)
    dv = x["dv"].view(T, Hkv * d)
    grads = dict(wq=dq, wk=dk, wv=dv)
    y["gx"] = sum(dy @ w[n].t().contiguous() for n, dy in grads.items()).flatten()
    xt = xn.t().contiguous()
    for n, dy in grads.items():
        y["g" + n] = (xt @ dy).flatten()
    return y
