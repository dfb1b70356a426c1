"""The register-resident forward chain, which runs where there are more chains than a round of the other one's workgroups:
batch rows of such a scan, run alone (few chains: the one-wave chain), give bitwise the same outputs, states and
gradients in every contract, and the fp64 oracle's values.  test_host_streams.py checks on the CPU that every case here
takes the register chain, and their rows alone do not."""
import pytest
import torch

from oracle import scan_oracle as SO
from scan_inputs import np64, scan_inputs

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotkern_hip as KH

F32, BF = torch.float32, torch.bfloat16
# mode, B, T, H, N, D, G, token dtype, per-token fr, occ_bin, start state
CASES = [
    ("f32", 257, 40, 1, 97, 128, 8, F32, True, False, False),
    ("f32", 129, 37, 2, 130, 128, 5, BF, False, True, True),
    ("f32", 257, 16, 1, 191, 128, 16, BF, True, False, True),
    ("f32", 257, 1, 1, 192, 128, 8, F32, False, False, False),
    # the pipeline's chunks and a ragged end; both routes cut at multiples of the 16-step window, at which they form the
    # scores anew (519 = 4 x 128 + 7 = 256 + 128 + 64 + 32 + 39), so that the logged cosines are the same bits too
    ("f32", 257, 519, 1, 100, 128, 8, BF, True, True, False),
    ("f32", 300, 21, 1, 177, 64, 8, F32, True, False, True),
    ("f32", 512, 33, 1, 96, 128, 4, F32, False, False, False),
    ("mem", 300, 41, 1, 130, 128, 8, BF, True, False, False),
    ("mem", 512, 24, 1, 192, 64, 8, F32, False, True, False),
    ("mem", 512, 13, 1, 81, 128, 4, F32, True, False, False),
    ("memq", 300, 15, 1, 130, 128, 8, BF, True, True, False),
    ("memq", 512, 8, 1, 96, 128, 3, F32, True, False, False),
    ("codes", 300, 16, 1, 177, 128, 8, BF, False, True, True),
    ("codes", 512, 7, 1, 90, 128, 2, F32, True, False, True),
]


def _forward(mode, x, frt, N, G, occb, state):
    """Every output of one forward with its logs (codes: without), batch row first."""
    k, v, g, fr, q = x
    B, T, H, D = k.shape
    rows = lambda t: t.reshape(B, H, *t.shape[1:])
    if mode == "codes":
        kc, vc, fin = KH.kv_scan_stream_q(k, v, g, fr, N, 16.0, G=G, q=q, occ_bin=occb, state=state)
        return [*kc, *vc, *map(rows, fin)]
    dt, k_, q_, v_, g_, fr_, _, temp = KH._prep(k, q, v, g, fr, 16.0, False)
    out = KH._fwd(k_, q_, v_, g_, fr_, frt, temp, N, G, 1e-4, occb, dt, True, state=state, mem=mode != "f32",
                  bits=3 if mode == "memq" else 0)
    copies = list(out[:2]) if mode == "f32" else list(out[0])
    am, kold, vold, oold, cslog, kfin, vfin, ofin = out[-8:]
    return copies + [rows(kfin), rows(vfin), rows(ofin), am, kold, vold, oold, rows(cslog)]


def _gradients(mode, x, N, G, occb):
    x = [t.requires_grad_() for t in x]
    k, v, g, fr, q = x
    kw = dict(G=G, q=q, occ_bin=occb, hard=True, detach_addr=True)
    out = KH.kv_scan_c(k, v, g, fr, N, 16.0, **kw) if mode == "f32" else \
        KH.kv_scan_mem(k, v, g, fr, N, 16.0, bits=3 if mode == "memq" else 0, group=16, **kw)
    diff = [o for o in out if o.dtype != torch.bool]
    up = [torch.cos(torch.arange(o[0].numel(), device="cuda") * 0.37).reshape(1, *o.shape[1:]).expand(o.shape).to(o.dtype)
          for o in diff]
    return list(torch.autograd.grad(diff, [t for t in x if t.dim() > 1], up))      # (a scalar fr sums over the batch)


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_reg_chain_equals_rows_alone(case):
    mode, B, T, H, N, D, G, dt, frt, occb, has_state = case
    print("reg chain", case, flush=True)
    k, q, v, g, fr = scan_inputs(B, T, H, D, 1000 + N + T, frt=frt, dtype=dt)
    tok = [x.cuda() for x in (k, v, g, fr, q)]
    gen = torch.Generator().manual_seed(N)
    r = lambda *s: torch.randn(*s, generator=gen)
    st = None
    if has_state:
        o = torch.rand(B, H, N, generator=gen) * (torch.rand(B, H, N, generator=gen) < 0.8)
        st = [(r(B, H, N, D) * 0.1 * o[..., None]).cuda(), (r(B, H, N, D) * o[..., None]).cuda(), o.cuda()]

    def run(rows):
        pick = lambda t: (t if rows is None or t.dim() == 1 else t[rows]).detach().clone()
        x = [pick(t) for t in tok]
        res = _forward(mode, x, frt, N, G, occb, None if st is None else [pick(t).flatten(0, 1) for t in st])
        if mode != "codes" and st is None:
            res += _gradients(mode, x, N, G, occb)
        return res

    full = run(None)
    for rows in ([0], [1, B // 2, B - 2], [B - 1]):
        for a, b in zip(full, run(rows)):
            assert torch.equal(a[rows], b)

    if mode == "f32" and N > 1 and T > 1:                                # and the oracle, on two rows
        rows = [0, B - 1]
        os = None if st is None else tuple(np64(t[rows]) for t in st)
        frn = np64(fr[rows]) if frt else np64(fr)
        okb, ovb, info = SO.scan_forward(np64(k[rows]), np64(v[rows]), np64(g[rows]), frn, N, 16.0, G=G, hard=True,
                                         q=np64(q[rows]), occ_bin=occb, state=os)
        for got, ref in zip(full, (okb, ovb)):
            assert abs(np64(got[rows]) - ref).max() <= 1e-5 * max(abs(ref).max(), 1e-30)
        for got, ref in zip(full[2:5], (info["kfin"], info["vfin"], info["ofin"])):
            assert abs(np64(got[rows]) - ref).max() <= 1e-5 * abs(ref).max()
        assert (full[5][rows].cpu().numpy() == info["am"]).all()
