"""The calls that a program built on this package makes, as cases for measuring their time and outputs.

A case is a dict of plain values; `op` names the entry point:
    scan     kv_scan_c, hard and detached address: the writer layer's scan, forward and backward
    mem      kv_scan_mem: the same scan with the writer epilogue (bits = 0) or the storage quantiser (bits > 0)
    soft     kv_scan_g with its default modes: soft write address, attached address gradient
    stream   kv_scan_stream (bits = 0) / kv_scan_stream_q: one chunk of a long stream, the state carried in and out
    read     shared_read: a reader layer's cosine read, one block of copies per G tokens
    frozen   slot_read of one frozen store (one block for the whole sequence)
    readout  shared_read_out: the reader layer's read and its output projection into the residual
    window   window: the exact short-term attention of every layer

`train` runs the forward and the backward against given upstream gradients, otherwise the forward alone without
autograd.  Sizes are those of the benchmark's workloads and of the tests, and what lies between them.  prepare()
draws every input from its seed on the GPU; exact() states each path in float64 with plain torch.
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "smal-memory-llm_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import slotkern_hip as KH  # noqa: E402
import slotread_hip as RH  # noqa: E402
import slotwin_hip as WH  # noqa: E402

EPS = 1e-4           # occupancy threshold, the entry points' default
TEMP = 16.0          # write temperature
RSHARP = 2.0         # the bound C of the read multiplier exp(C tanh(s / C))
BF = torch.bfloat16


def listed():
    train = dict(dtype="bf16", train=True)
    return [
        # the smallest training scan that the tests and the CPU baseline use: launches and the serial chain
        dict(name="scan_small", op="scan", B=2, T=128, H=1, N=64, D=64, G=8, dtype="f32", train=True),
        # the main memory's scan at full length and one GPU's share of the batch: the headline workload
        dict(name="scan_train", op="scan", B=64, T=1024, H=6, N=192, D=128, G=8, **train),
        # the encoder memory half way through the length curriculum, with the writer epilogue
        dict(name="mem_curriculum", op="mem", B=256, T=256, H=6, N=96, D=128, G=8, bits=0, group=16, **train),
        # the quantisation-aware phase of training at a small batch and a length that fills no whole window
        dict(name="mem_qat", op="mem", B=16, T=1000, H=6, N=192, D=128, G=8, bits=3, group=16, **train),
        # soft write addresses (the entry point's default), full length, half a batch
        dict(name="soft_train", op="soft", B=32, T=1024, H=6, N=192, D=128, G=8, **train),
        # long-context inference: a 1,024-token chunk, copies emitted as int8 codes with a scale per row
        dict(name="stream_chunk", op="stream", B=8, T=1024, H=6, N=192, D=128, G=8, bits=8, group=128, dtype="bf16",
             train=False),
        # the same stream as it is generated: one block of 8 tokens for 4 sequences
        dict(name="stream_step", op="stream", B=4, T=8, H=6, N=192, D=128, G=8, bits=0, group=128, dtype="bf16",
             train=False),
        # a reader layer in training
        dict(name="read_train", op="read", B=64, T=1024, H=6, NQ=2, N=192, D=128, G=8, **train),
        # a later layer's read of a store that no longer changes
        dict(name="read_frozen", op="frozen", B=64, T=1024, H=6, NQ=1, N=192, D=128, dtype="bf16", train=False),
        # a reader layer in training with its projection into the residual, quarter batch
        dict(name="readout_train", op="readout", B=16, T=1024, H=6, NQ=2, N=192, D=128, G=8, DM=2048, **train),
        # the same layer while 8 sequences generate a block of 8 tokens
        dict(name="readout_step", op="readout", B=8, T=8, H=6, NQ=2, N=192, D=128, G=8, DM=2048, dtype="bf16",
             train=False),
        # every layer's window in training: the extra queries' call, 3 query heads per key/value head
        dict(name="window_train", op="window", B=64, T=1024, Hk=4, Hq=12, D=128, W=16, **train),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["scan", "scan", "mem", "soft", "stream", "stream", "read", "frozen", "readout", "readout",
                     "window"])
    D = rng.choice([64, 128, 128])
    H = rng.choice([1, 2, 4, 6, 6, 8])
    N = rng.choice([32, 48, 64, 96, 100, 128, 160, 192, 192])
    G = rng.choice([4, 5, 8, 8, 8, 16])
    T = _log(rng, 32, 1024)
    if op in ("scan", "mem", "soft"):
        # tokens x heads of one call: 256 up to the headline's 393,216 (soft: the soft case's 196,608)
        per = _log(rng, 256, 196608 if op == "soft" else 393216)
        # no more copy bytes than the headline's (a copy every 8 tokens, 192 x 128)
        per = min(per, int(393216 * (192 * 128 / 8) / (N * D / G)))
        B = max(1, min(512, per // (T * H)))
        c = dict(op=op, B=B, T=T, H=H, N=N, D=D, G=G, dtype=rng.choice(["bf16", "bf16", "f32"]),
                 train=rng.random() < 0.8)
        if op == "mem":
            c["bits"], c["group"] = rng.choice([(0, 16), (3, 16), (4, 32), (8, 64)])
        return c
    if op == "stream":
        bits, group = rng.choice([(0, D), (8, D), (8, 64), (4, 32)])
        return dict(op=op, B=_log(rng, 1, 32), T=_log(rng, 1, 1024), H=H, N=N, D=D, G=G, bits=bits, group=group,
                    dtype=rng.choice(["bf16", "bf16", "f32"]), train=False)
    if op == "read":
        NQ = rng.choice([1, 2, 2])
        # no more copy bytes than the listed reader layer's
        B = _log(rng, 1, max(1, min(64, int(65536 * 6 * 192 * 128 / 8 / (T * H * N * D / G)))))
        return dict(op=op, B=B, T=T, H=H, NQ=NQ, N=N, D=D, G=G, dtype="bf16", train=rng.random() < 0.7)
    if op == "frozen":
        return dict(op=op, B=_log(rng, 1, 64), T=_log(rng, 1, 1024), H=H, NQ=rng.choice([1, 1, 2]), N=N, D=D,
                    dtype="bf16", train=rng.random() < 0.3)
    if op == "readout":
        H, D = rng.choice([(2, 128), (4, 64), (4, 128), (6, 128), (6, 128), (8, 128)])
        train = rng.random() < 0.5
        T = _log(rng, 32, 1024) if train else _log(rng, 1, 1024)
        G = rng.choice([5, 8, 8, 16])
        return dict(op=op, B=_log(rng, 1, max(1, min(32, 16384 // T))), T=T, H=H, NQ=2, N=N, D=D, G=G,
                    DM=rng.choice([512, 1024, 2048, 2048]), dtype="bf16", train=train)
    Hk = rng.choice([1, 2, 4, 4, 8])
    T = _log(rng, 16, 2048)
    return dict(op=op, B=_log(rng, 1, max(1, min(64, 65536 * 4 // (T * Hk)))), T=T, Hk=Hk, Hq=Hk * rng.choice([1, 2, 3]),
                D=D, W=rng.choice([8, 15, 16, 16]), dtype="bf16", train=rng.random() < 0.7)


def _unit(x):
    return x / x.norm(dim=-1, keepdim=True)


def _blocks(c):
    return 1 if c["op"] == "frozen" else -(-c["T"] // c["G"])


def prepare(case, seed):
    c = case
    dev = torch.device("cuda:0")
    gen = torch.Generator(device=dev).manual_seed(int(seed) * 7919 + 11)
    rn = lambda *s: torch.randn(*s, device=dev, generator=gen)
    ru = lambda *s: torch.rand(*s, device=dev, generator=gen)
    dt = BF if c["dtype"] == "bf16" else torch.float32
    op, B, T, D = c["op"], c["B"], c["T"], c["D"]
    s = dict(case=c)
    if op == "window":
        # token-major activations as the layer's projection leaves them, seen as (B, heads, T, D)
        s["cq"], s["ck"], s["cv"] = (rn(B, T, h, D).to(BF).transpose(1, 2) for h in (c["Hq"], c["Hk"], c["Hk"]))
        s["up"] = [rn(B, T, c["Hq"], D).to(BF).transpose(1, 2)] if c["train"] else None
        s["leaves"] = [s["cq"], s["ck"], s["cv"]]
    elif op in ("scan", "mem", "soft", "stream"):
        H, N = c["H"], c["N"]
        s["k"], s["q"] = (_unit(rn(B, T, H, D)).to(dt) for _ in range(2))
        s["v"] = rn(B, T, H, D).to(dt)
        s["gate"] = torch.sigmoid(rn(B, T, H) * 1.5).to(dt)
        s["fr"] = (ru(B, T, H) * 2).to(dt)
        s["temp"] = torch.tensor(TEMP, device=dev)
        s["leaves"] = [s[x] for x in ("k", "q", "v", "gate", "fr", "temp")]
        if op == "stream":
            # what an earlier chunk left: rows blended from several unit keys, the last eighth still free
            used = (torch.arange(N, device=dev) < max(1, N - N // 8)).float()
            o = (0.3 + 0.7 * ru(B * H, N)) * used
            s["state"] = (_unit(rn(B * H, N, D)) * o.unsqueeze(-1), rn(B * H, N, D) * o.unsqueeze(-1), o)
        elif c["train"]:
            NB = _blocks(c)
            udt = BF if op == "mem" else torch.float32
            s["up"] = [rn(B, NB, H, N, D).to(BF).to(udt) for _ in range(2)] + ([rn(B, NB, H, N)] if op == "mem" else [])
    else:
        H, N, NQ, NB = c["H"], c["N"], c["NQ"], _blocks(c)
        # In training the store fills while the sequence goes on: the free rows are zero, and the first block is
        # empty.  A frozen store and that of a sequence being continued are whole.
        if op == "frozen" or not c["train"]:
            fill = torch.full((NB,), N, device=dev)
        else:
            fill = (torch.arange(NB, device=dev) * c["G"]).clamp_max(N)
        live = (torch.arange(N, device=dev) < fill.unsqueeze(-1)).view(1, NB, 1, N)
        o = (0.3 + 0.7 * ru(B, NB, H, N)) * live
        kb = _unit(rn(B, NB, H, N, D)).mul_(o.unsqueeze(-1))
        nsq = kb.pow(2).sum(-1)
        s["kinv"], s["valid"] = torch.rsqrt(nsq.clamp_min(1e-12)), nsq > 1e-12
        s["kb"] = kb.to(BF)
        del kb
        s["vb"] = rn(B, NB, H, N, D).mul_(o.unsqueeze(-1)).to(BF)
        if op == "frozen":
            s["q"] = _unit(rn(B, T, H, NQ, D)).to(BF)
            s["scale"] = F.softplus(rn(B, T, H, NQ)) + 1.0
            s["leaves"] = [s[x] for x in ("q", "kb", "vb", "kinv", "scale")]
        else:
            s["q"] = rn(B, T, H, NQ, D).to(BF)                 # as tk_q leaves them, not yet normalised
            s["log_rsel"] = torch.tensor(math.log(8.0), device=dev)
            s["s"] = rn(B, T, H, NQ)
            s["leaves"] = [s[x] for x in ("q", "kb", "vb", "kinv", "log_rsel", "s")]
        if op == "readout":
            KD = H * NQ * D
            s["wo"] = (rn(c["DM"], KD) / KD ** 0.5).to(BF)
            s["delta"] = rn(B, T, c["DM"]).to(BF)
            s["leaves"] += [s["wo"], s["delta"]]
            s["up"] = [rn(B, T, c["DM"]).to(BF)]
        else:
            s["up"] = [rn(B, T, H, NQ, D).to(BF)]
    if c["train"]:
        for x in s["leaves"]:
            x.requires_grad_()
    return s


def _call(s):
    c = s["case"]
    op = c["op"]
    if op == "window":
        return [WH.window(s["cq"], s["ck"], s["cv"], c["W"])]
    if op == "read":
        return [RH.shared_read(s["q"], s["kb"], s["vb"], s["kinv"], s["valid"], s["log_rsel"], c["G"], s=s["s"],
                               rsharp=RSHARP)]
    if op == "frozen":
        return [RH.slot_read(s["q"], s["kb"], s["vb"], s["kinv"], s["valid"], s["scale"], c["T"])]
    if op == "readout":
        return [RH.shared_read_out(s["q"], s["kb"], s["vb"], s["kinv"], s["valid"], s["log_rsel"], c["G"], s["wo"],
                                   s=s["s"], rsharp=RSHARP, delta=s["delta"])]
    tok = (s["k"], s["v"], s["gate"], s["fr"], c["N"], s["temp"])
    if op == "soft":
        return list(KH.kv_scan_g(*tok, G=c["G"], q=s["q"]))
    if op == "scan":
        return list(KH.kv_scan_c(*tok, G=c["G"], hard=True, detach_addr=True, q=s["q"], occ_bin=True))
    if op == "mem":
        return list(KH.kv_scan_mem(*tok, G=c["G"], hard=True, detach_addr=True, q=s["q"], occ_bin=True, bits=c["bits"],
                                   group=c["group"]))
    kw = dict(G=c["G"], q=s["q"], occ_bin=True, state=s["state"])
    if c["bits"]:
        kc, vc, st = KH.kv_scan_stream_q(*tok, bits=c["bits"], group=c["group"], **kw)
        return [*kc, *vc, *st]
    kb, vb, st = KH.kv_scan_stream(*tok, **kw)
    return [kb, vb, *st]


def run(state):
    s = state
    if not s["case"]["train"]:
        with torch.no_grad():
            return _call(s)
    outs = _call(s)
    diff = [o for o in outs if o.dtype != torch.bool]
    return [o.detach() for o in outs] + list(torch.autograd.grad(diff, s["leaves"], s["up"]))


def work(case):
    """Each input read once, each output written once; the products that the path consists of."""
    c = case
    op, B, T, D, tr = c["op"], c["B"], c["T"], c["D"], c["train"]
    e = 2 if c["dtype"] == "bf16" else 4
    both = 2 if tr else 1                  # every input has a gradient, every output an upstream one
    if op == "window":
        q, kv = B * T * c["Hq"] * D, B * T * c["Hk"] * D
        band = 2 * B * T * c["Hq"] * c["W"] * D
        return dict(bytes=both * e * (2 * q + 2 * kv), flops=band * (7 if tr else 2))
    H, N = c["H"], c["N"]
    NB = _blocks(c)
    if op in ("scan", "mem", "soft", "stream"):
        tok = B * T * H * (3 * D + 2) * e
        rows = B * NB * H * N
        if op == "mem":
            out = rows * (2 * D * 2 + 4)
            got = rows * (2 * D * 2 + 5)
        elif op == "stream":
            st = B * H * N * (2 * D + 1) * 4
            got = rows * (2 * D + 2 * (D // c["group"]) * 4 if c["bits"] else 2 * D * 4) + 2 * st
            out = 0
        else:
            out = got = rows * 2 * D * 4
        # scores; the backward's row sums <k, dK> + <v, dV> and the query gradient; a soft write moves every row
        per = 2 * N * D * ((4 if tr else 1) + (0 if op != "soft" else 10 if tr else 4))
        return dict(bytes=both * tok + got + (out if tr else 0), flops=B * T * H * per)
    M = B * T * H * c["NQ"]
    store = B * NB * H * N * (2 * D * 2 + 4)
    by = both * (M * (D * 2 + 4) + store) + B * NB * H * N
    fl = 2 * M * N * D * (7 if tr else 2)
    if op == "readout":
        KD, DM = H * c["NQ"] * D, c["DM"]
        by += both * (B * T * DM * 2 * 2 + DM * KD * 2) - (B * T * DM * 2 if tr else 0)   # delta's gradient is the
        fl += 2 * B * T * DM * KD * (3 if tr else 1)                                      # upstream one itself
    else:
        by += both * M * D * 2
    return dict(bytes=by, flops=fl)


def tolerance(case):
    """About four times the error against exact() of the listed and some drawn cases, at most 3e-2 and 1."""
    op = case["op"]
    if op in ("read", "readout"):
        # bf16 scores and probabilities under a multiplier of up to 60: 0.7-1.0e-2; single values of the rows of
        # small norm 0.9
        return dict(rel=3e-2, max=0.95)
    if op in ("frozen", "window"):
        # the same roundings under a multiplier of about 2 (frozen: 2.4e-3, 1.2e-2) or none (window: 2.5e-3, 5e-2);
        # with gradients of a frozen store up to 5e-3
        return dict(rel=2e-2 if op == "frozen" and case["train"] else 1e-2, max=0.2)
    if case["dtype"] == "bf16" or op == "mem":
        # results rounded to bf16: 1.7e-3, single values 3.9e-3; a quantiser's value that falls on the other side
        # of a threshold is a step off (0.4), one in a million
        return dict(rel=7e-3, max=0.95 if case.get("bits") else 1.6e-2, differ=1e-5)
    # sums in 32 bits: 4e-6, single values 4e-5 (a soft address over a long sequence 2e-6 and 4e-4)
    return dict(rel=2e-5, max=1.6e-3, differ=1e-5)


# ---- the same in float64, with plain torch ----------------------------------------------------------------


def _scan_steps(K, V, o, k, q, v, g, fr, temp, hard):
    """The write of every given step (k, q, v (B,t,H,D), g, fr (B,t,H)) on the state K, V (B,H,N,D), o (B,H,N)."""
    n = torch.arange(K.shape[2], device=K.device)
    for t in range(k.shape[1]):
        Ka = K.detach() if hard else K
        kn = Ka / Ka.norm(dim=-1, keepdim=True).clamp_min(1e-6)
        qn = q[:, t] / q[:, t].norm(dim=-1, keepdim=True).clamp_min(1e-6)
        occ = (o >= EPS).double() if hard else o
        z = (kn @ qn.unsqueeze(-1)).squeeze(-1) * temp - fr[:, t].unsqueeze(-1) * occ
        free = o < EPS
        first = torch.where(free, n, n.numel()).amin(-1, keepdim=True)
        a = torch.softmax(z.masked_fill(free & (n != first), -1e30), -1)
        if hard:
            hot = F.one_hot(z.masked_fill(free & (n != first), -1e30).argmax(-1), n.numel()).double()
            a = hot + (a - a.detach())
        w = g[:, t].unsqueeze(-1) * a
        o = torch.lerp(o, torch.ones_like(o), w)
        w = w.unsqueeze(-1)
        K = K + w * (k[:, t].unsqueeze(2) - K)
        V = V + w * (v[:, t].unsqueeze(2) - V)
    return K, V, o


def _quantised(x, bits, group):
    """(value, code, scale) of the midrise quantiser over groups of channels; its thresholds are float32's."""
    xg = x.float().reshape(*x.shape[:-1], -1, group)
    half = float(2 ** (bits - 1))
    a = xg.abs().amax(-1, keepdim=True)
    sc = (a / half).clamp_min(1e-30)
    code = torch.floor(xg / sc).clamp(-half, half - 1)
    val = torch.where(a > 0, (code.double() + 0.5) * sc.double(), 0.0)
    return val.reshape(x.shape), code.to(torch.int8).reshape(x.shape), torch.where(a > 0, sc, 0.0).squeeze(-1)


def _exact_scan(s):
    c = s["case"]
    B, T, H, N, D, G, op = (c[x] for x in ("B", "T", "H", "N", "D", "G", "op"))
    hard = op != "soft"
    tok = [s[x].detach().double() for x in ("k", "q", "v", "gate", "fr")]
    temp = s["temp"].detach().double()
    z = lambda *sh: torch.zeros(*sh, device=temp.device, dtype=torch.float64)
    if op == "stream":
        st = tuple(x.double().reshape(B, H, *x.shape[1:]) for x in s["state"])
    else:
        st = (z(B, H, N, D), z(B, H, N, D), z(B, H, N))
    keep, at = [], list(range(0, T, G))
    with torch.no_grad():
        for t in at:
            keep.append(st)
            st = _scan_steps(*st, *(x[:, t:t + G] for x in tok), temp, hard)
        kbuf, vbuf = (torch.stack([x[i] for x in keep], 1) for i in range(2))
        if op != "stream":
            keep = [(None, None, x[2]) for x in keep]     # the copies hold the rest
    if op == "stream":
        fin = [x.reshape(B * H, *x.shape[2:]) for x in st]
        if not c["bits"]:
            return [kbuf, vbuf, *fin]
        (_, kc, ks), (_, vc, vs) = (_quantised(x, c["bits"], c["group"]) for x in (kbuf, vbuf))
        return [kc, ks.double(), vc, vs.double(), *fin]
    outs = [kbuf, vbuf]
    if op == "mem":
        vals = [_quantised(x, c["bits"], c["group"])[0] if c["bits"] else x for x in outs]
        nsq = vals[0].pow(2).sum(-1)
        outs = [*vals, torch.rsqrt(nsq.clamp_min(1e-12)), nsq > 1e-12]
    if not c["train"]:
        return outs
    up = [x.double() for x in s["up"]]
    if op == "mem":                        # the quantiser's gradient goes straight through
        dn = torch.where(nsq >= 1e-12, -0.5 * outs[2].pow(3) * up[2], 0.0)
        up = [up[0] + 2.0 * vals[0] * dn.unsqueeze(-1), up[1]]
    got = [torch.zeros_like(x) for x in tok]
    d = (z(B, H, N, D), z(B, H, N, D), z(B, H, N))
    for j in range(len(at) - 1, -1, -1):
        t = at[j]
        seg = [x[:, t:t + G].detach().requires_grad_() for x in tok]
        st = [x.detach().requires_grad_() for x in (kbuf[:, j], vbuf[:, j], keep[j][2])]
        with torch.enable_grad():
            gr = torch.autograd.grad(_scan_steps(*st, *seg, temp, hard), seg + st, d)
        for x, y in zip(got, gr):
            x[:, t:t + G] = y
        d = (gr[5] + up[0][:, j], gr[6] + up[1][:, j], gr[7])
        del gr, st, seg
    # The temperature's gradient sums mixed-sign terms of every token to one number: its error is one draw of the
    # rounding of all of them and says nothing about precision, so it has no exact value here.
    return outs + got + [None]


def _exact_read(s):
    """One slice of the batch: (rd, s, scale leaves) -> the read's value in float64."""
    c = s["case"]
    B, T, H, NQ, N, D = (s["q"].shape[0],) + tuple(c[x] for x in ("T", "H", "NQ", "N", "D"))
    NB = _blocks(c)
    G = T if c["op"] == "frozen" else c["G"]
    q = s["q"]
    if c["op"] == "frozen":
        scale = s["scale"]
    else:
        q = q / q.norm(dim=-1, keepdim=True).clamp_min(1e-6)
        scale = torch.exp(s["log_rsel"] + RSHARP * torch.tanh(s["s"] / RSHARP))
    pad = NB * G - T
    q = F.pad(q, (0, 0, 0, 0, 0, 0, 0, pad)).reshape(B, NB, G, H, NQ, D).permute(0, 1, 3, 2, 4, 5).reshape(B, NB, H, G * NQ, D)
    scale = F.pad(scale, (0, 0, 0, 0, 0, pad)).reshape(B, NB, G, H, NQ).permute(0, 1, 3, 2, 4).reshape(B, NB, H, G * NQ)
    sc = (q @ s["kb"].transpose(-1, -2)) * s["kinv"].unsqueeze(-2) * scale.unsqueeze(-1)
    ok = s["valid"].unsqueeze(-2)
    att = torch.softmax(sc.masked_fill(~ok, -1e30), -1) * ok
    rd = att @ s["vb"]
    rd = rd.reshape(B, NB, H, G, NQ, D).permute(0, 1, 3, 2, 4, 5).reshape(B, NB * G, H, NQ, D)[:, :T]
    if c["op"] != "readout":
        return rd
    return s["delta"] + rd.reshape(B, T, -1) @ s["wo"].t()


def _exact_window(s):
    c = s["case"]
    W, rep = c["W"], c["Hq"] // c["Hk"]
    band = lambda x: F.pad(x.repeat_interleave(rep, dim=1), (0, 0, W - 1, 0)).unfold(2, W, 1)     # (B, Hq, T, D, W)
    t = torch.arange(c["T"], device=s["cq"].device)
    ok = t.unsqueeze(-1) - (W - 1) + torch.arange(W, device=t.device) >= 0
    sc = (s["cq"].unsqueeze(-1) * band(s["ck"])).sum(-2) * c["D"] ** -0.5
    att = torch.softmax(sc.masked_fill(~ok, -1e30), -1)
    return (band(s["cv"]) * att.unsqueeze(-2)).sum(-1)


def exact(case, seed):
    s = prepare(case, seed)
    c = case
    if c["op"] in ("scan", "mem", "soft", "stream"):
        return _exact_scan(s)
    if c["op"] == "window":
        fn, names, size = _exact_window, ["cq", "ck", "cv"], 3 * c["T"] * c["Hq"] * c["D"] * c["W"]
    else:
        fn, size = _exact_read, c["T"] * c["H"] * c["NQ"] * 4 * c["N"] + 4 * _blocks(c) * c["H"] * c["N"] * c["D"]
        names = dict(frozen=["q", "kb", "vb", "kinv", "scale"], read=["q", "kb", "vb", "kinv", "log_rsel", "s"],
                     readout=["q", "kb", "vb", "kinv", "log_rsel", "s", "wo", "delta"])[c["op"]]
    step = max(1, int(3e9 / size))                     # sequences at once
    outs, grads = [], {x: [] for x in names}
    for b in range(0, c["B"], step):
        part = dict(case=c)
        whole = ("wo", "log_rsel")
        for x in names + ["valid"] * (c["op"] != "window"):
            y = s[x].detach() if x in whole else s[x].detach()[b:b + step]
            part[x] = y if y.dtype == torch.bool else y.double().requires_grad_(c["train"])
        out = fn(part)
        outs.append(out.detach())
        if c["train"]:
            for x, y in zip(names, torch.autograd.grad(out, [part[x] for x in names], s["up"][0][b:b + step].double())):
                grads[x].append(y)
        del out, part
    got = [torch.cat(outs)]
    if c["train"]:
        # (as for the scan's temperature: one number summed from every query's mixed-sign terms)
        got += [None if x == "log_rsel" else sum(grads[x]) if x == "wo" else torch.cat(grads[x]) for x in names]
    return got
