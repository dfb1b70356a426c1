"""A short scan of more chains than one round of the forward chain's workgroups runs as a pipeline over groups of
batch rows: rows around the group boundary, run alone (one group), give bitwise the same outputs, states and
gradients in every contract."""
import pytest
import torch

from scan_inputs import scan_inputs

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotkern_hip as KH

B, T, D = 300, 200, 128          # one workgroup per CU at these row counts: 256 chains a round
ROWS = ([0, 1], [254, 255, 256, 257], [299])


def _tokens(H, seed, dtype):
    k, q, v, g, fr = scan_inputs(B, T, H, D, seed, dtype=dtype)
    return [x.cuda() for x in (k, v, g, fr, q)]


@pytest.mark.parametrize("N,dtype,mode", [(70, torch.float32, "f32"), (130, torch.bfloat16, "mem"),
                                          (130, torch.bfloat16, "memq")])
def test_groups_equal_rows_alone(N, dtype, mode):
    tok = _tokens(1, 900 + N, dtype)

    def run(rows):
        x = [(t if rows is None else t[rows]).detach().clone().requires_grad_() for t in tok]
        k, v, g, fr, q = x
        kw = dict(G=8, hard=True, detach_addr=True, q=q, occ_bin=True)
        if mode == "f32":
            out = KH.kv_scan_c(k, v, g, fr, N, 16.0, **kw)
        else:
            out = KH.kv_scan_mem(k, v, g, fr, N, 16.0, bits=3 if mode == "memq" else 0, group=16, **kw)
        diff = [o for o in out if o.dtype != torch.bool]
        up = [torch.cos(torch.arange(o[0].numel(), device="cuda") * 0.37).reshape(1, *o.shape[1:]).expand(o.shape).to(o.dtype)
              for o in diff]
        return [o.detach() for o in out] + list(torch.autograd.grad(diff, x, up))

    full = run(None)
    for rows in ROWS:
        for a, b in zip(full, run(rows)):
            assert torch.equal(a[rows], b)


def test_groups_stream_codes_with_state():
    N, H = 130, 2
    k, v, g, fr, q = _tokens(H, 950, torch.bfloat16)
    gen = torch.Generator().manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=gen).cuda()
    st = (r(B * H, N, D) * 0.1, r(B * H, N, D), torch.rand(B * H, N, generator=gen).cuda())

    def run(rows):
        s = [x if rows is None else x.reshape(B, H, *x.shape[1:])[rows].reshape(-1, *x.shape[1:]) for x in st]
        x = [t if rows is None else t[rows] for t in (k, v, g, fr, q)]
        kc, vc, fin = KH.kv_scan_stream_q(*x[:4], N, 16.0, G=8, q=x[4], occ_bin=True, state=s)
        n = B if rows is None else len(rows)
        return [*kc, *vc] + [f.reshape(n, H, *f.shape[1:]) for f in fin]

    full = run(None)
    for rows in ROWS:
        for a, b in zip(full, run(rows)):
            assert torch.equal(a[rows], b)
