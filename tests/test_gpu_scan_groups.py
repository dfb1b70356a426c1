"""A short scan of more chains than one round of the forward chain's workgroups runs as a pipeline over groups of
batch rows: rows around the group boundary, run alone (one group), give bitwise the same outputs, states and
gradients in every contract."""
import pytest
import torch

from scan_inputs import scan_inputs

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotkern_hip as KH

F32, BF = torch.float32, torch.bfloat16
# mode, token dtype, B, T, H, N, D, G, batch rows of a group; test_host_streams.py checks on the CPU that these groups run
GROUPS = [
    ("f32", F32, 300, 200, 1, 70, 128, 8, 256),          # one workgroup per CU at these row counts: 256 chains a round
    ("mem", BF, 300, 200, 1, 130, 128, 8, 256),
    ("memq", BF, 300, 200, 1, 130, 128, 8, 256),
    ("f32", BF, 520, 200, 1, 70, 128, 5, 512),           # two per CU
    ("f32", F32, 1030, 193, 1, 40, 64, 8, 1024),         # four
    ("mem", BF, 519, 200, 3, 40, 64, 8, 426),            # five, and a group that ends between them (1,280 / 3)
    ("mem", BF, 520, 90, 1, 130, 128, 8, 512),           # 192 / 90: two rounds a group
    ("f32", BF, 2600, 33, 1, 70, 128, 16, 2560),         # 192 / 33: five
]


def _rows(B, group):
    return [0, 1], [x for x in range(group - 2, group + 2) if x < B], [B - 1]


@pytest.mark.parametrize("case", GROUPS, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
@pytest.mark.parametrize("frt", [True, False])
def test_groups_equal_rows_alone(case, frt):
    mode, dtype, B, T, H, N, D, G, group = case
    print("groups", case, frt, flush=True)
    k, q, v, g, fr = scan_inputs(B, T, H, D, 900 + N, dtype=dtype, frt=frt)
    tok = [x.cuda() for x in (k, v, g, fr, q)]

    def run(rows):
        x = [(t if rows is None or t.dim() == 1 else t[rows]).detach().clone().requires_grad_() for t in tok]
        k, v, g, fr, q = x
        kw = dict(G=G, hard=True, detach_addr=True, q=q, occ_bin=True)
        if mode == "f32":
            out = KH.kv_scan_c(k, v, g, fr, N, 16.0, **kw)
        else:
            out = KH.kv_scan_mem(k, v, g, fr, N, 16.0, bits=3 if mode == "memq" else 0, group=16, **kw)
        diff = [o for o in out if o.dtype != torch.bool]
        up = [torch.cos(torch.arange(o[0].numel(), device="cuda") * 0.37).reshape(1, *o.shape[1:]).expand(o.shape).to(o.dtype)
              for o in diff]
        leaves = [t for t in x if t.dim() > 1]           # (a scalar fr sums over the batch)
        return [o.detach() for o in out] + list(torch.autograd.grad(diff, leaves, up))

    full = run(None)
    for rows in _rows(B, group):
        for a, b in zip(full, run(rows)):
            assert torch.equal(a[rows], b)


def test_groups_stream_codes_with_state():
    B, T, N, H, D = 300, 200, 130, 2, 128
    k, q, v, g, fr = (x.cuda() for x in scan_inputs(B, T, H, D, 950, dtype=torch.bfloat16))
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
    for rows in _rows(B, 128):
        for a, b in zip(full, run(rows)):
            assert torch.equal(a[rows], b)
