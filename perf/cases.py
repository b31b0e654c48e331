"""The workloads that this framework's speed is judged on, through its public entry points
(``aideen_amd.backend.GpuDeqBackend``): what each stands for in use, how its inputs are made, what
one pass runs, the work it cannot do without, and the same results in 64 bits.

Sizes are the repository's own presets (``synth.PRESETS``: C1, C2, NS, C3, C4 and the wide rows of
C5), the reference's evaluation shape (d = 192, 8 slots, 65 symbols, ctx = 128, 6 fixed steps) and
generic ragged ones.  Weights are signal-driven as a trained model's are (the ranges of
``synth.make_token_sensitive_weights``): every token has its own fixed point, so iteration counts
vary from token to token.  They are drawn on the GPU; a Xavier-uniform matrix has its largest
singular value near 2, so the spectral scale is applied in closed form.
"""
import math

import numpy as np
import torch

from aideen_amd import synth
from aideen_amd.backend import GpuDeqBackend

PREC = {"f16x3": 0, "bf16x3": synth.F_GEMM_BF16X3, "fp32": synth.F_GEMM_FP32, "bf16": synth.F_GEMM_BF16}
SAMPLE = dict(temperature=0.8, top_p=0.9, top_k=40, repetition_penalty=1.1)  # the reference binaries' settings

# the fields that a kind of case may leave out
DEFAULTS = dict(d=512, H=8, V=50257, N=16, prec="f16x3", m=0, sigma=0.5, iters=20, eps=0.0, ctx=0, long=False,
                want="pooled,logits,argmax", typical=10, bias=False, adj=2, new=0)


def _c(name, **kw):
    return dict(name=name, **kw)


def listed():
    return [
        # One serving step: the query of one 256-token window, ten fixed steps, its next-token logits.
        # The smallest call: launches and latency.
        _c("serve_1", kind="query", B=1, T=256, iters=10),
        # The same step for a batch of 24 requests.
        _c("serve_24", kind="query", B=24, T=256, iters=10),
        # A sampled reply of 24 tokens to a 200-token prompt (host arrays, blocking), then the logits
        # of the position that follows it.
        _c("generate_24", kind="generate", B=1, T=200, new=24, iters=10, ctx=256),
        # Evaluation of a character model as the reference's benchmark runs it: the context query of
        # every position, six fixed steps.
        _c("eval_char", kind="forward", B=1, T=128, d=192, V=65, N=1, iters=6, ctx=128),
        # One document window with the carrier (preset C2): an ordinary single request.
        _c("window_256", kind="forward", B=1, T=256, eps=1e-4,
           want="h_star,pooled,logits,argmax,iters,converged,scan_y,scan_state"),
        # The throughput batch (preset NS) with every output.
        _c("batch_8192", kind="forward", B=32, T=256, eps=1e-4,
           want="h_star,pooled,logits,argmax,iters,converged,scan_y,scan_state"),
        # Throughput with bf16 inputs, which a caller chooses for speed; ragged sizes.
        _c("batch_bf16", kind="forward", B=24, T=250, prec="bf16", iters=8, want="h_star,pooled,logits"),
        # The Anderson-mixed solve of a less contractive model (preset C3's block), ragged sizes.  Depth
        # 3: deeper rings run into Gram matrices so near singular that rounding sets some tokens'
        # coefficients (depth 5, eight updates: 1e-3 off the 64-bit result, depth 3: 4e-7).
        _c("anderson", kind="forward", B=9, T=333, sigma=0.7, m=3, iters=8, want="h_star,pooled,logits,argmax"),
        # Long documents through the carrier (preset C4): the scan's share is at its largest.
        _c("carrier_8k", kind="forward", B=4, T=8192, eps=1e-4, long=True, want="pooled,iters,scan_y,scan_state"),
        # The memory-coupled forward: every position waits for the one before it.
        _c("memory_64", kind="memory", B=32, T=64, N=1, eps=1e-4, want="h_star,logits,argmax,iters,scan_y,scan_state"),
        # A training step's forward and backward: pooled fixed points, then the adjoint of the loss
        # gradient (v) and the source gradient, two adjoint steps as the reference runs.
        _c("train_4096", kind="train", B=8, T=512, iters=6, want="h_star,pooled"),
        # Wide rows and twice the slots, a few hundred ragged tokens.
        _c("wide_531", kind="forward", B=3, T=177, d=1024, H=16, N=32, iters=8, want="h_star,pooled,logits,argmax"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["query", "query", "generate", "forward", "forward", "forward", "forward", "memory", "train"])
    d = rng.choice([64, 128, 192, 256, 320, 512, 512, 512, 1024])
    H = rng.choice([2, 3, 4, 6, 8, 8, 8, 16]) if d <= 512 else rng.choice([4, 8])
    c = dict(kind=kind, d=d, H=H, V=rng.choice([65, 512, 2100, 50257]), N=rng.choice([1, 4, 16, 32]),
             prec=rng.choice(["f16x3"] * 5 + ["bf16x3", "fp32", "bf16"]), bias=rng.random() < 0.25)
    if kind == "query":
        c.update(B=_log_int(rng, 1, 300), T=_log_int(rng, 16, 512), iters=10)
    elif kind == "generate":
        c.update(B=_log_int(rng, 1, 12), T=_log_int(rng, 8, 300), new=_log_int(rng, 4, 24), iters=10, ctx=256,
                 V=50257, prec="f16x3")
    elif kind == "memory":
        c.update(B=_log_int(rng, 2, 40), T=_log_int(rng, 5, 64), N=1, iters=rng.choice([6, 10]),
                 want="h_star,logits,argmax,scan_y,scan_state")
    else:
        most = min(8192, 8192 * 8 * 512 * 512 // (H * d * d))
        n = _log_int(rng, 20, most)
        T = _log_int(rng, 4, n)
        c.update(B=max(1, n // T), T=T)
        if kind == "train":
            c.update(iters=6, want="h_star,pooled", adj=rng.choice([1, 2, 3]))
        else:
            c.update(iters=rng.choice([6, 8, 10]), m=rng.choice([0, 0, 0, 3]), ctx=rng.choice([0, 0, 128]),
                     want=rng.choice(["pooled,logits,argmax", "h_star,pooled,logits,argmax",
                                      "pooled,logits,argmax,scan_y,scan_state"]))
            if c["m"]:
                c["sigma"] = 0.7
    if c["prec"] == "bf16":  # near-ties of the arg-max turn on the rounding of the inputs
        c.update(m=0, want=c.get("want", DEFAULTS["want"]).replace(",argmax", ""))
    return c


def _full(case):
    return {**DEFAULTS, **case}


def _model(c):
    flags = PREC[c["prec"]] | (synth.F_MEMORY if c["kind"] == "memory" else synth.F_SCAN_SELECTIVE)
    return synth.ModelConfig(d=c["d"], H=c["H"], V=c["V"], N=c["N"], flags=flags, max_iters=c["iters"], eps=c["eps"],
                             anderson_m=c["m"], sigma=c["sigma"])


def _weights(c, seed):
    """The model's tensors as float32 on the GPU, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 1)
    d, H, V, N, r = c["d"], c["H"], c["V"], c["N"], 32
    dev = dict(device="cuda", generator=g, dtype=torch.float32)

    def uni(shape, lo, hi):
        return torch.rand(shape, **dev) * (hi - lo) + lo

    xr = math.sqrt(3.0 / d)
    w = {k: uni((H, d, d), -xr, xr) * (c["sigma"] / 2) for k in ("w_q", "w_k", "w_v", "w_o")}
    w["w_in"] = uni((H, d, d), -xr, xr) * 1.5
    w["q_bias"] = uni((H, d), -0.08, 0.08) if c["bias"] else None
    w["k_bias"] = uni((H, d), -0.08, 0.08) if c["bias"] else None
    w["anchor"] = uni((H, d), -0.02, 0.02)
    w["norm_scale"] = torch.ones(d, device="cuda")
    w["embed"] = uni((V, d), -0.2, 0.2)
    w["lm_w"] = uni((V, d), -xr, xr)
    w["lm_b"] = uni((V,), -0.05, 0.05)
    w["lm_g"] = uni((d,), 0.75, 1.25)
    alpha = torch.linspace(0, 1, H, device="cuda") if H > 1 else torch.full((1,), 0.5, device="cuda")
    base = (0.80 + alpha * 0.199)[:, None].expand(H, d)
    if c["long"]:  # decay bases from long memory to almost none across the channels
        base = torch.linspace(0.999, 0.01, d, device="cuda")[None].expand(H, d)
    w["a_log"] = torch.log((1 - base) / base) if c["long"] else torch.log(base / (1 - base))
    gate = 1.0 if c["long"] else 0.0
    w["b_delta"] = torch.randn((H, d), **dev) * gate
    w["w_kw"] = torch.randn((H, d, r), **dev) / math.sqrt(d) if gate else uni((H, d, r), -0.01, 0.01)
    w["w_vw"] = torch.randn((H, r, d), **dev) / math.sqrt(r) if gate else uni((H, r, d), -0.01, 0.01)
    w["wx_diag"] = uni((H, d), -0.01, 0.01)
    w["w_out"] = uni((H, d, d), -0.01, 0.01)
    w["w_b"] = uni((H, N, d), -xr, xr) if N > 1 else None
    w["w_c"] = uni((H, N, d), -xr, xr) if N > 1 else None
    if c["kind"] == "memory":
        w["w_hist"] = torch.eye(d, device="cuda") * 0.15 + uni((d, d), -0.01, 0.01)
        w["hist_slot_scale"] = uni((H, d), -1e-2, 1e-2)
        w["hist_gate_logit"] = uni((H,), -1.3, -1.1)
    return {k: None if v is None else v.contiguous() for k, v in w.items()}


def _inputs(c, seed):
    """Token ids (Zipf-distributed ranks), the loss gradient and the sampling draws."""
    rng = np.random.default_rng(int(seed) * 2 + 2)
    p = 1.0 / np.arange(1, c["V"] + 1) ** 1.1
    cdf = np.cumsum(p / p.sum())
    toks = np.minimum(np.searchsorted(cdf, rng.random((c["B"], c["T"])), side="right"), c["V"] - 1).astype(np.int32)
    uni = (rng.integers(0, 1 << 24, (c["B"], max(1, c["new"]))) * 2.0 ** -24).astype(np.float32)
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 2 + 3)
    dl = torch.randn((c["B"], c["T"], c["d"]), device="cuda", generator=g) if c["kind"] == "train" else None
    return toks, uni, dl


_STREAM = []


def _stream():
    """The one stream that every context and torch's copies between its calls run on."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def prepare(case, seed):
    c = _full(case)
    mc = _model(c)
    B, T, d, H = c["B"], c["T"], c["d"], c["H"]
    w = {k: None if v is None else v.cpu().numpy() for k, v in _weights(c, seed).items()}
    toks, uni, dl = _inputs(c, seed)
    be = GpuDeqBackend(mc, B, T)
    be.upload_weights(w)
    be._weights_keepalive = None  # the device holds them
    s = dict(c=c, be=be, toks=toks, uni=uni)
    if c["kind"] == "generate":
        return s
    be.set_stream(_stream().cuda_stream)
    n = 1 if c["kind"] == "query" else T  # positions solved
    f32, i32 = dict(device="cuda", dtype=torch.float32), dict(device="cuda", dtype=torch.int32)
    shapes = dict(h_star=(B, n, H, d), pooled=(B, n, d), logits=(B, n, c["V"]), scan_y=(B, n, H, d),
                  scan_state=(B, H, d, c["N"]))
    s["out"] = {k: torch.empty(shapes[k], **f32) if k in shapes else torch.empty((B, n), **i32)
                for k in c["want"].split(",")}
    s["tok"] = torch.from_numpy(toks).cuda()
    if c["kind"] == "query" or c["ctx"]:
        s["q"] = torch.empty((B, T, d), **f32)
    if c["kind"] == "query":
        s["last"] = torch.empty((B, 1, d), **f32)
    if c["kind"] == "train":
        s["dl"] = dl
        s["v"] = torch.empty((B, T, H, d), **f32)
        s["src"] = torch.empty((B, T, d), **f32)
    torch.cuda.synchronize()
    return s


def run(s):
    c, be = s["c"], s["be"]
    if c["kind"] == "generate":
        reply = be.decode_sample(s["toks"], c["new"], c["ctx"], uniforms=s["uni"], **SAMPLE)
        window = np.concatenate([s["toks"], reply], axis=1)[:, -min(c["T"], c["ctx"]):]
        q = be.embed_context(window, c["ctx"])[:, -1:]
        return dict(reply=reply, **be.forward(s_in=q, max_iters=c["iters"], eps=0.0, want=("pooled", "logits")))
    if c["kind"] == "query":
        be.embed_context_async(s["tok"], c["T"], s["q"])
        if c["B"] > 1:
            with torch.cuda.stream(_stream()):
                s["last"].copy_(s["q"][:, -1:])
        be.forward_async(s_in=s["last"] if c["B"] > 1 else s["q"][:, -1:], outputs=s["out"])
        return s["out"]
    if c["ctx"]:
        be.embed_context_async(s["tok"], c["ctx"], s["q"])
        be.forward_async(s_in=s["q"], outputs=s["out"])
    else:
        be.forward_async(s["tok"], outputs=s["out"])
    if c["kind"] == "train":
        be.adjoint_async(c["B"] * c["T"], s["dl"], c["adj"], be.model.beta, s["v"], s["src"])
        return dict(s["out"], v=s["v"], src=s["src"])
    return s["out"]


def work(case):
    """Weights read once, inputs read once, outputs written once; the operations of the solve (the
    typical number of updates where tokens exit on the tolerance), the head, the carrier and the
    adjoint.  A product of fp32 values counts once, however many products carry it."""
    c = _full(case)
    B, T, d, H, V, N, r = c["B"], c["T"], c["d"], c["H"], c["V"], c["N"], 32
    n = B if c["kind"] == "query" else B * T
    if c["kind"] == "generate":
        n = B * (c["new"] + 1)
    k = c["typical"] if c["eps"] > 0 else c["iters"]
    want = ["pooled", "logits"] if c["kind"] == "generate" else c["want"].split(",")
    rows = B if c["kind"] == "generate" else n
    sizes = dict(h_star=H * d, pooled=d, logits=V, scan_y=H * d, argmax=1, iters=1, converged=1)
    flops = n * (2 * H * d * d + k * (8 * H * d * d + 4 * H * H * d + 10 * H * d))
    by = 4 * (5 * H * d * d + 2 * H * d)
    by += 4 * sum(rows * sizes[o] for o in want if o in sizes)
    by += 4 * min(B * T, V) * d + 4 * B * T  # embedding rows and token ids
    if "logits" in want:
        flops += 2 * n * V * d
        by += 4 * V * (d + 1)
    if "scan_y" in want and c["kind"] != "memory":
        flops += n * H * d * (2 * (r + 2 * N) + 2 * r + 4 * N + 2 * d)
        by += 4 * (H * d * d + 2 * H * d * (r + N) + 2 * B * H * d * N)
    if c["kind"] == "memory":
        flops += n * H * d * 4 * d
        by += 4 * (H * d * d + d * d + B * H * d)
    if c["kind"] == "train":
        flops += n * H * d * (8 * c["adj"] + 6)
        by += 4 * n * d * (H + 2)
    return {"bytes": by, "flops": flops}


def tolerance(case):
    c = _full(case)
    if c["prec"] == "bf16":
        return {"rel": 1e-2, "differ": 0.01}
    # largest errors seen against 64 bits: 9e-7 (fp16 pairs, fp32), 7e-6 (bf16 pairs), 3e-3 (bf16); where
    # tokens exit on the tolerance, a residual within rounding of it moves a token by one update
    return {"rel": 4e-5 if c["prec"] == "bf16x3" else 5e-6, "differ": 0.01}


# ---------------------------------------------------------------------------------------------
# the same results in 64 bits
# ---------------------------------------------------------------------------------------------
def _rms(x, eps):
    return torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _anderson64(ring, k, m):
    """The mixed iterate of step k from the ring of iterates [H][n][d]."""
    nr = min(k, m - 1)
    xs = [ring[(k - i) % m] for i in range(nr + 1)]
    f = [xs[i] - xs[i + 1] for i in range(nr)]
    G = torch.stack([torch.stack([(a * b).sum((0, 2)) for b in f], -1) for a in f], -2)  # [n][nr][nr]
    tr = G.diagonal(dim1=-2, dim2=-1).abs().sum(-1)
    A = G + torch.clamp(1e-4 * tr, min=1e-8)[:, None, None] * torch.eye(nr, device=G.device, dtype=G.dtype)
    low = 1e-10 if nr == 2 else 1e-8

    def det(M):
        k_ = M.shape[-1]
        if k_ == 1:
            return M[:, 0, 0]
        cols = list(range(k_))
        return sum((-1) ** j * M[:, 0, j] * det(M[:, 1:, [q for q in cols if q != j]]) for j in cols)

    dt = det(A)
    dt = torch.where(dt < 0, dt.clamp(max=-low), dt.clamp(min=low))
    beta = []
    for j in range(nr):
        M = A.clone()
        M[:, :, j] = 1.0
        beta.append((det(M) / dt).clamp(-2.0, 3.0))
    s = sum(beta)
    bad = s.abs() < 1e-6
    beta = [torch.where(bad, torch.full_like(b, float(i == 0)), b / s) for i, b in enumerate(beta)]
    return sum(b[None, :, None] * x for b, x in zip(beta, xs))


def _solve64(c, w, x, hist=None):
    """x [n][d] -> h [H][n][d], signal [H][n][d]."""
    H, d, beta = c["H"], c["d"], 0.70
    n = x.shape[0]
    sig = torch.bmm(x[None].expand(H, n, d).contiguous(), w["w_in_t"])
    h = x[None] + w["anchor"][:, None]
    live = torch.ones(n, dtype=torch.bool, device=x.device)
    ring = [None] * max(1, c["m"])
    for k in range(c["iters"]):
        q, kk, v = (torch.bmm(h, w[t]) for t in ("w_q_t", "w_k_t", "w_v_t"))
        if c["bias"]:
            q, kk = q + w["q_bias"][:, None], kk + w["k_bias"][:, None]
        q, kk, v = (t.transpose(0, 1).contiguous() for t in (q, kk, v))  # [n][H][d]
        a = torch.softmax(torch.bmm(q, kk.transpose(1, 2).contiguous()) / math.sqrt(d), -1)
        o = torch.bmm(torch.bmm(a, v).transpose(0, 1).contiguous(), w["w_o_t"])
        s = o + sig + w["anchor"][:, None]
        if hist is not None:
            s = s + hist
        nxt = (w["norm_scale"] * s / _rms(s, 1e-6)) * beta + h * (1 - beta)
        done = (nxt - h).abs().amax((0, 2)) < c["eps"]
        mixed = nxt
        if c["m"] >= 3:
            ring[k % c["m"]] = nxt
            if k >= 2:
                mixed = torch.where(done[None, :, None], nxt, _anderson64(ring, k, c["m"]))
        h = torch.where(live[None, :, None], mixed, h)
        live = live & ~done
        if not bool(live.any()):
            break
    return h, sig


def _head64(c, w, h, out, lead):
    pooled = h.mean(0)
    out["pooled"] = pooled.reshape(*lead, -1)
    out["logits"] = (((pooled / _rms(pooled, 1e-5)) * w["lm_g"]) @ w["lm_w"].t() + w["lm_b"]).reshape(*lead, -1)


def _queries64(c, w, toks):
    """The context query of the last position of every window, [B][d]; toks [B][L]."""
    e = w["embed"][toks]
    r = (e * torch.arange(1, toks.shape[1] + 1, device=e.device, dtype=e.dtype)[:, None]).sum(1) / toks.shape[1]
    return r / r.norm(dim=-1, keepdim=True)


def _carrier64(c, w, h):
    """h [B][T][H][d] -> the carrier's outputs [B][T][H][d] and last state [B][H][d][N]."""
    B, T, H, d = h.shape
    N = c["N"]
    m = torch.zeros((B, H, d, N), device=h.device, dtype=h.dtype)
    ys = []
    ln_base = torch.log(torch.clamp(torch.sigmoid(-w["a_log"]), min=1e-6))
    for t0 in range(0, T, 256):
        u = h[:, t0:t0 + 256]
        u = u / _rms(u, 1e-6)
        us = u.permute(2, 0, 1, 3).reshape(H, -1, d)  # [H][B*t][d]
        x = u * (1 + 0.5 * torch.tanh(w["wx_diag"]))
        pre = torch.bmm(torch.bmm(us, w["w_kw"]), w["w_vw"]) + w["b_delta"][:, None]
        ab = 0.1 + 0.9 * torch.exp(torch.log1p(torch.exp(pre)) * ln_base[:, None])
        ab = ab.reshape(H, B, -1, d).permute(1, 2, 0, 3)
        bc = [torch.ones((B, u.shape[1], H, 1), device=h.device, dtype=h.dtype)] * 2
        if N > 1:
            bc = [torch.bmm(us, w[k].transpose(1, 2).contiguous()).reshape(H, B, -1, N).permute(1, 2, 0, 3)
                  for k in ("w_b", "w_c")]
        zx = (1 - ab) * x
        for t in range(u.shape[1]):
            m = ab[:, t, :, :, None] * m + zx[:, t, :, :, None] * bc[0][:, t, :, None]
            ys.append((m * bc[1][:, t, :, None]).sum(-1))
    y = torch.stack(ys, 1)
    wy = torch.bmm(y.permute(2, 0, 1, 3).reshape(H, -1, d), w["w_out_t"])
    return y + wy.reshape(H, B, T, d).permute(1, 2, 0, 3), m


def _memory64(c, w, toks, out):
    B, T, H, d = c["B"], c["T"], c["H"], c["d"]
    ab = torch.sigmoid(-w["a_log"])[:, None]
    alpha = 0.07 + 0.13 * torch.sigmoid(w["hist_gate_logit"])[:, None, None]
    hs, ms, m = [], [], None
    for t in range(T):
        x = w["embed"][toks[:, t]]
        hist = None
        if m is not None:
            sig = torch.bmm(x[None].expand(H, B, d).contiguous(), w["w_in_t"])
            u = m @ w["w_hist"].t() + w["hist_slot_scale"][:, None] * m / _rms(m, 1e-6)
            hist = u * alpha * torch.clamp(_rms(sig, 1e-6) / _rms(u, 1e-6), max=1.0)
        h, _ = _solve64(c, w, x, hist)
        inner = (1 - ab) * (h / _rms(h, 1e-6)) * (1 + 0.5 * torch.tanh(w["wx_diag"]))[:, None]
        inner = inner if m is None else ab * m + inner
        m = inner + torch.bmm(inner, w["w_out_t"])
        hs.append(h)
        ms.append(m)
    h, m = torch.stack(hs, 2), torch.stack(ms, 2)  # [H][B][T][d]
    out["h_star"], out["scan_y"] = h.permute(1, 2, 0, 3), m.permute(1, 2, 0, 3)
    out["scan_state"] = m[:, :, -1].permute(1, 0, 2)[..., None]
    return h.reshape(H, B * T, d)


def _adjoint64(c, w, h, sig, dl, out):
    H, d, beta = c["H"], c["d"], 0.70
    g = w["norm_scale"]
    pre = sig + h
    rhs = (dl.double().reshape(-1, d) / H)[None]
    rms = _rms(pre, 1e-6)

    def vjp(v):
        up = beta * v
        return g / rms * up - pre * ((up * g * pre).sum(-1, keepdim=True) / (d * rms ** 3))

    v = rhs.expand(H, -1, d)
    for _ in range(c["adj"]):
        v = rhs + vjp(v) + (1 - beta) * v
    lead = (c["B"], c["T"])
    out["v"], out["src"] = v.transpose(0, 1).reshape(*lead, H, d), vjp(v).sum(0).reshape(*lead, d)


def _draw64(c, logits, context, u):
    """One token of the sampling rule at SAMPLE's settings, in 64 bits."""
    lg = logits.clone()
    seen = torch.unique(context)
    lg[seen] = torch.where(lg[seen] < 0, lg[seen] * SAMPLE["repetition_penalty"], lg[seen] / SAMPLE["repetition_penalty"])
    p, ix = torch.sort(torch.softmax(lg / SAMPLE["temperature"], -1), descending=True, stable=True)
    p = p[:SAMPLE["top_k"]].cpu().numpy()
    cut = np.nonzero(np.cumsum(p) > SAMPLE["top_p"])[0]
    p = p[:cut[0] + 1] if len(cut) else p
    hit = np.nonzero(np.float64(u) <= np.cumsum(p / p.sum()))[0]
    return int(ix[hit[0] if len(hit) else 0])


def exact(case, seed):
    c = _full(case)
    w = {k: None if v is None else v.double() for k, v in _weights(c, seed).items()}
    for k in ("w_q", "w_k", "w_v", "w_o", "w_in", "w_out"):
        w[k + "_t"] = w.pop(k).transpose(1, 2).contiguous()
    toks, uni, dl = _inputs(c, seed)
    tok = torch.from_numpy(toks).cuda().long()
    B, T, H, d = c["B"], c["T"], c["H"], c["d"]
    out = {}
    if c["kind"] == "generate":
        seq = tok
        for j in range(c["new"]):
            win = seq[:, -c["ctx"]:]
            _head64(c, w, _solve64(c, w, _queries64(c, w, win))[0], out, (B,))
            nxt = [_draw64(c, out["logits"][b], win[b], uni[b, j]) for b in range(B)]
            seq = torch.cat([seq, torch.tensor(nxt, device=seq.device)[:, None]], 1)
        win = seq[:, -min(T, c["ctx"]):]
        _head64(c, w, _solve64(c, w, _queries64(c, w, win))[0], out, (B, 1))
        return dict(reply=None, pooled=out["pooled"], logits=out["logits"])
    if c["kind"] == "memory":
        h = _memory64(c, w, tok, out)
        sig = None
    else:
        if c["kind"] == "query":
            x = _queries64(c, w, tok)
        elif c["ctx"]:
            x = torch.cat([_queries64(c, w, tok[:, max(0, i + 1 - c["ctx"]):i + 1])[:, None] for i in range(T)], 1)
            x = x.reshape(B * T, d)
        else:
            x = w["embed"][tok.reshape(-1)]
        h, sig = _solve64(c, w, x)
        lead = (B, 1) if c["kind"] == "query" else (B, T)
        out["h_star"] = h.transpose(0, 1).reshape(*lead, H, d)
    lead = (B, 1) if c["kind"] == "query" else (B, T)
    want = c["want"].split(",")
    if "logits" in want:
        _head64(c, w, h, out, lead)
    out["pooled"] = h.mean(0).reshape(*lead, d)
    if "scan_y" in want and c["kind"] != "memory":
        out["scan_y"], out["scan_state"] = _carrier64(c, w, out["h_star"])
    if c["kind"] == "train":
        _adjoint64(c, w, h, sig, dl, out)
        want = want + ["v", "src"]
    return {k: out[k].contiguous() if k in out else None for k in want}
