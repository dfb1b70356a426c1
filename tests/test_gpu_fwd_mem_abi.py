"""slotscan_fwd_mem through the C-ABI: the outputs, states and logs of slotscan_fwd_memq with bits = 0, bitwise, although it
runs long scans as one chunk (it has no key carry); on the one-wave chain, in batch groups, and on the register chain."""
import pytest
import torch

from scan_inputs import scan_inputs

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotscan_lib as L


# the longer ones are cut at multiples of the 16-step window by the other entry point (512 = 256 + 128 + 64 + 32 + 32)
@pytest.mark.parametrize("B,T,H,N,D,G,dtype", [
    (2, 37, 3, 70, 64, 5, torch.float32), (1, 512, 2, 192, 128, 8, torch.bfloat16), (3, 519, 2, 40, 64, 8, torch.float32),
    (300, 200, 1, 130, 128, 8, torch.bfloat16), (300, 40, 1, 130, 128, 8, torch.bfloat16),
])
@pytest.mark.parametrize("logs", [True, False])
@pytest.mark.parametrize("has_state", [True, False])
def test_fwd_mem_equals_memq_without_bits(B, T, H, N, D, G, dtype, logs, has_state):
    print("fwd_mem", B, T, H, N, D, G, dtype, logs, has_state, flush=True)
    dev = torch.device("cuda:0")
    k, q, v, g, fr = (x.to(dev) for x in scan_inputs(B, T, H, D, 70 + N, dtype=dtype))
    temp = torch.tensor([16.0], device=dev)
    gen = torch.Generator().manual_seed(4)
    o0 = torch.rand(B * H, N, generator=gen).to(dev)
    st = [torch.randn(B * H, N, D, generator=gen).to(dev) * o0[..., None] for _ in range(2)] + [o0] if has_state else [None] * 3
    NB, P, f32 = -(-T // G), L.ptr, torch.float32
    e = lambda *s, dt=f32: torch.full(s, 3, device=dev, dtype=dt)

    def run(memq):
        out = [e(B, NB, H, N, D, dt=torch.bfloat16), e(B, NB, H, N, D, dt=torch.bfloat16), e(B, NB, H, N),
               e(B, NB, H, N, dt=torch.uint8), e(B, T, H, dt=torch.int32)]
        log = [e(B, T, H, D), e(B, T, H, D), e(B, T, H), e(B * H, T, N)] if logs else [None] * 4
        fin = [e(B * H, N, D), e(B * H, N, D), e(B * H, N)]
        head = (P(k), P(q), P(v), L.dtype_code(dtype), P(g), P(fr), 1, P(temp), B, T, H, N, D, G, 1e-4, 1)
        tail = tuple(map(P, st + out + log + fin))
        if memq:
            nb = L.lib().slotscan_fwd_carry_bytes(B, T, H, N, D, G)
            car = torch.empty(nb // 4, device=dev) if nb else None
            L.check(L.lib().slotscan_fwd_memq(*head, 0, 16, *tail, P(car), L.stream_of(dev)), "slotscan_fwd_memq")
        else:
            L.check(L.lib().slotscan_fwd_mem(*head, *tail, L.stream_of(dev)), "slotscan_fwd_mem")
        torch.cuda.synchronize()
        return [t for t in out + log + fin if t is not None]

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)
