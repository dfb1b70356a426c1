"""The projection's few-row kernel and both sides of the rule that chooses it, forward, with and without the residual, and
the backward's products at the same row counts, which the tile kernels form, against float64.  Guard rows behind the
output stay untouched.  test_host_streams.py checks on the CPU which kernel each case here runs."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotread_hip as RH
    import slotscan_lib as L


def _bound(ref, mag, K):
    """One bf16 rounding of a K-term fp32 sum (unit roundoff 2^-8; the sum's own error at most K 2^-24 of the sum of
    magnitudes), with a residual a second one."""
    return 2.0 ** -8 * 1.02 * ref.abs() + K * 2.0 ** -24 * mag


# (M, N, K), whether the few-row kernel runs
FORWARD = [
    ((1, 256, 32), True), ((15, 256, 64), True), ((16, 256, 224), True), ((17, 512, 256), True), ((32, 256, 1536), True),
    ((33, 256, 288), True), ((64, 2048, 1536), True), ((65, 512, 512), True), ((128, 1024, 96), True),
    ((256, 2048, 64), True), ((257, 2048, 64), False), ((300, 2048, 96), False), ((2048, 256, 64), True),
    ((2049, 256, 64), False),
]
BACKWARD = [(5, 256, 256), (40, 512, 1024), (70, 2048, 256), (700, 256, 1024)]


@pytest.mark.parametrize("M,N,K", [s for s, _ in FORWARD])
@pytest.mark.parametrize("res", [True, False])
def test_proj_rows_matches_float64(M, N, K, res):
    gen = torch.Generator().manual_seed(M + N + K)
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=gen) / K ** 0.5).to(torch.bfloat16).cuda()
    d = torch.randn(M, N, generator=gen).to(torch.bfloat16).cuda() if res else None
    out = torch.full((M + 3, N), 7.0, device="cuda", dtype=torch.bfloat16)
    rc = L.lib().slotproj_fwd(L.ptr(x), L.ptr(w), L.ptr(d), M, N, K, L.ptr(out), L.stream_of(x.device))
    L.check(rc, "slotproj_fwd")
    ref = x.double() @ w.double().t()
    tol = _bound(ref, x.double().abs() @ w.double().abs().t(), K)
    if res:
        ref = ref + d.double()
        tol = tol + 2.0 ** -8 * 1.02 * (ref.abs() + tol)
    assert ((out[:M].double() - ref).abs() <= tol).all()
    assert (out[M:] == 7.0).all()


@pytest.mark.parametrize("M,N,K", BACKWARD)
def test_few_rows_backward(M, N, K):
    gen = torch.Generator().manual_seed(3 * M + K)
    g = torch.randn(M, N, generator=gen).to(torch.bfloat16).cuda()
    x = torch.randn(M, K, generator=gen).to(torch.bfloat16).cuda()
    w = (torch.randn(N, K, generator=gen) / K ** 0.5).to(torch.bfloat16).cuda()
    dx, dw = RH._proj_bwd(g, x, w)
    for got, a, b, n in ((dx, g.double(), w.double(), N), (dw, g.double().t(), x.double(), M)):
        ref = a @ b
        assert ((got.double() - ref).abs() <= _bound(ref, a.abs() @ b.abs(), n)).all()
