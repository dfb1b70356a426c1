"""The read's query preparation kernels against float64, and against the torch expressions they replace."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotread_hip as RH


def _inputs(B, T, H, NQ, D, seed):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    q = (r(B, T, H, NQ, D) * torch.exp(3 * r(B, T, H, NQ, 1))).to(torch.bfloat16)
    q[0, 0, 0, 0] = 0                                   # |q| below the clamp
    q[-1, -1, -1, -1] *= 1e-9
    return q, r(B, T, H, NQ) * 2, r(B, T, H, NQ, D).to(torch.bfloat16), r(B, T, H, NQ)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("B,T,H,NQ", [(1, 1, 1, 1), (1, 3, 5, 1), (2, 9, 6, 2), (3, 33, 4, 2)])
@pytest.mark.parametrize("sharp", [2.0, 0, None, "no s"])
def test_prep_matches_float64(B, T, H, NQ, D, sharp):
    q, s, dqn, dsc = _inputs(B, T, H, NQ, D, 7 * T + D)
    has_s = sharp != "no s"
    lr = torch.tensor(0.7, device="cuda", requires_grad=True)
    qq = q.cuda().requires_grad_()
    ss = s.cuda().requires_grad_() if has_s else None
    qn, sc = RH._prep(qq, lr, ss, sharp if has_s else None)
    assert qn.grad_fn.name().startswith("_PrepHip")
    leaves = [qq, lr] + ([ss] if has_s else [])
    got = torch.autograd.grad([qn, sc], leaves, [dqn.cuda(), dsc.cuda()])
    x, d, sd = q.double(), dqn.double(), s.double()
    nrm = x.norm(dim=-1, keepdim=True)
    nb = nrm.clamp_min(1e-6)
    # two bf16 roundings (the norm, the quotient) of unit roundoff 2^-8 each (8 significant bits), and fp32 noise
    e = 2.0 ** -7 * 1.02
    ref = x / nb
    assert ((qn.double().cpu() - ref).abs() <= e * ref.abs() + 1e-30).all()
    f = sd * 0
    if has_s:
        f = sharp * torch.tanh(sd / sharp) if sharp else sd
    ref = torch.exp(lr.double().cpu() + f)
    assert ((sc.double().cpu() - ref).abs() <= 2e-6 * ref).all()
    p = dsc.double() * ref
    # dq: each of the two terms carries the norm's bf16 rounding (2 and 3 times) and the result's: at most 4 x 2^-8
    a, b = d / nb, torch.where(nrm >= 1e-6, x * (d * x).sum(-1, keepdim=True) / (nb * nb * nrm.clamp_min(1e-30)), 0.0)
    mag = (d * x).abs().sum(-1, keepdim=True) * x.abs() / (nb * nb * nrm.clamp_min(1e-30))
    assert ((got[0].double().cpu() - (a - b)).abs() <= 2 * e * (a.abs() + torch.where(nrm >= 1e-6, mag, 0.0)) + 1e-30).all()
    assert abs(got[1].item() - p.sum().item()) <= 1e-5 * p.abs().sum().item()
    if has_s:
        ref = p * (1 - torch.tanh(sd / sharp) ** 2) if sharp else p
        assert ((got[2].double().cpu() - ref).abs() <= 1e-5 * p.abs()).all()


def test_prep_takes_views_and_leaves_broadcasts_to_torch():
    """A view at an odd offset or with strides takes the kernel; a log_rsel or s that broadcasts, and other dtypes,
    take the torch expressions -- with the same values (bf16 queries: at most one rounding apart)."""
    q, s, _, _ = (x.cuda() for x in _inputs(2, 6, 4, 2, 64, 3))
    lr = torch.tensor(0.3, device="cuda")
    base = RH._prep(q, lr, s, 2.0)
    flat = torch.empty(q.numel() + 1, device="cuda", dtype=q.dtype)
    odd = flat[1:].view(q.shape).copy_(q)
    strided = q.transpose(1, 2).contiguous().transpose(1, 2)
    for v in (odd, strided):
        assert all(torch.equal(a, b) for a, b in zip(RH._prep(v, lr, s, 2.0), base))
    for args in ((q, lr.expand(4, 2).contiguous(), s, 2.0), (q.float(), lr, s, 2.0)):
        qn, sc = RH._prep(*args)
        torch.testing.assert_close(sc, base[1], rtol=2e-6, atol=0)
        torch.testing.assert_close(qn.float(), base[0].float(), rtol=2.0 ** -7, atol=1e-30)
    qn, sc = RH._prep(q, lr, s[:, :, :1, :1], 2.0)
    torch.testing.assert_close(sc[:, :, 0, 0], base[1][:, :, 0, 0], rtol=2e-6, atol=0)


@pytest.mark.parametrize("D", [64, 128])
def test_prep_passes_nan_and_infinity_on(D):
    """A NaN in a query makes its norm NaN, and with it the whole unit query and its gradient; an infinity leaves 0 and NaN.
    As the torch expressions; the other queries are untouched."""
    q, s, dqn, dsc = (x.cuda() for x in _inputs(2, 5, 3, 2, D, 11))
    lr = torch.tensor(0.3, device="cuda")
    bad = q.clone()
    bad[0, 1, 2, 0, 5] = float("nan")
    bad[1, 3, 0, 1, D - 1] = float("inf")

    def run(x, prep):
        x = x.clone().requires_grad_()
        qn, sc = prep(x)
        return qn.detach(), sc, torch.autograd.grad([qn], [x], [dqn])[0]

    a, b = run(bad, lambda x: RH._prep(x, lr, s, 2.0)), run(q, lambda x: RH._prep(x, lr, s, 2.0))
    t = run(bad, lambda x: (x / x.float().norm(dim=-1, keepdim=True).clamp_min(1e-6).to(x.dtype), None))
    assert a[0][0, 1, 2, 0].isnan().all() and a[2][0, 1, 2, 0].isnan().all()
    for i in (0, 2):
        assert torch.equal(a[i].isnan(), t[i].isnan())
    same = torch.ones(q.shape[:-1], dtype=torch.bool, device="cuda")
    same[0, 1, 2, 0] = same[1, 3, 0, 1] = False
    assert torch.equal(a[0][same], b[0][same]) and torch.equal(a[1], b[1]) and torch.equal(a[2][same], b[2][same])


@pytest.mark.parametrize("D", [64, 128])
def test_prep_gradient_error_is_no_larger_than_the_torch_expressions(D):
    """dq is formed in fp32 and rounded to bf16 once, where the torch expressions round every intermediate result: the two
    differ (2.9e-3, 2-norm), and the kernel's is the one closer to float64 (2.3e-3 against 2.9e-3)."""
    gen = torch.Generator().manual_seed(9)
    q = torch.randn(4, 256, 6, 2, D, generator=gen).to(torch.bfloat16).cuda()
    d = torch.randn(q.shape, generator=gen).to(torch.bfloat16).cuda()
    lr = torch.tensor(0.0, device="cuda")
    norm = lambda x: x / x.float().norm(dim=-1, keepdim=True).clamp_min(1e-6).to(x.dtype)
    exact = lambda x: x / x.norm(dim=-1, keepdim=True).clamp_min(1e-6)

    def grad(x, f):
        x = x.clone().requires_grad_()
        return torch.autograd.grad(f(x), x, d.to(x.dtype))[0].double()

    ref = grad(q.double(), exact)
    err = lambda f: ((grad(q, f) - ref).norm() / ref.norm()).item()
    kern, expr = err(lambda x: RH._prep(x, lr, None, None)[0]), err(norm)
    print(f"dq against float64: kernel {kern:.2e}, torch expressions {expr:.2e}")
    # the norm's rounding, common to a query, and the result's: each uniform within 2^-8 of the value at most
    assert kern <= expr and kern <= 2 * 2.0 ** -8 / 3 ** 0.5


def test_prep_refuses_a_log_rsel_that_does_not_expand():
    """One value in more dimensions than the multiplier (B, T, H, NQ) has was never accepted."""
    q, s, _, _ = (x.cuda() for x in _inputs(2, 3, 2, 1, 64, 5))
    base = RH._prep(q, torch.tensor(0.3, device="cuda"), s, 2.0)
    for n in range(5):
        assert all(torch.equal(a, b) for a, b in zip(RH._prep(q, torch.full((1,) * n, 0.3, device="cuda"), s, 2.0), base))
    with pytest.raises(RuntimeError):
        RH._prep(q, torch.full((1,) * 5, 0.3, device="cuda"), s, 2.0)
