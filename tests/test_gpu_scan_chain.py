"""The forward chain at the edges of its layout, against the fp64 oracle: row counts around a lane's share of the
rows (NR = 1, 2, 3 at 64 and 128) and around the 16-row score tiles, lengths around the 16-step window and its
turns of four steps, and occupancies that stay below, at or next to the threshold.  check_case's bars: addresses
and final occupancy exact, snapshots 1e-5, gradients 1e-4 of each tensor's largest value."""
import numpy as np
import pytest
import torch

from oracle import scan_oracle as SO
from scan_inputs import np64, scan_inputs
from test_gpu_scan import check_case

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    import slotkern_hip as KH


@pytest.mark.parametrize("N", [2, 15, 16, 17, 63, 64, 65, 96, 97, 127, 128, 129, 130, 191, 192])
@pytest.mark.parametrize("D", [64, 128])
def test_chain_row_counts(N, D):
    # longer than N, so that every row is written and the scan goes on with none free
    check_case(1, 37 if N < 32 else 230, 2, N, D, 8, True, True, True, False, seed=300 + N)


@pytest.mark.parametrize("T", [3, 4, 5, 15, 16, 17, 31, 33])
@pytest.mark.parametrize("occb", [True, False])
def test_chain_lengths(T, occb):
    check_case(2, T, 1, 70, 128, 5, True, occb, True, False, seed=400 + T, dtype=torch.float32)


@pytest.mark.parametrize("N,T", [(1, 20), (1, 1), (70, 1), (192, 2)])
def test_chain_one_competing_row(N, T):
    """Forward only: with one row the softmax adjoint is exactly 0, so a relative gradient bar says nothing."""
    B, H, D = 2, 3, 128
    k, q, v, g, fr = scan_inputs(B, T, H, D, 450 + N)
    kb, vb, st = KH.kv_scan_stream(*(x.cuda() for x in (k, v, g, fr)), N, 16.0, G=4, q=q.cuda(), occ_bin=True)
    okb, ovb, info = SO.scan_forward(np64(k), np64(v), np64(g), np64(fr), N, 16.0, G=4, hard=True, q=np64(q),
                                     occ_bin=True, teacher=np.zeros((B, T, H), int) if N == 1 else None)
    for got, ref in ((kb, okb), (vb, ovb), (st[0].reshape(B, H, N, D), info["kfin"]),
                     (st[1].reshape(B, H, N, D), info["vfin"]), (st[2].reshape(B, H, N), info["ofin"])):
        assert abs(np64(got) - ref).max() <= 1e-5 * max(abs(ref).max(), 1e-30)


@pytest.mark.parametrize("occb", [True, False])
def test_chain_occupancy_next_to_the_threshold(occb):
    """Gates around eps: rows whose first writes leave them free, and exact zeros and ones.  Without occ_bin the scores take
    the occupancy of every write, while the rows that compete change only where one crosses the threshold."""
    B, T, H, N, D = 2, 80, 2, 24, 64
    k, q, v, g, fr = scan_inputs(B, T, H, D, 500, gate_mix=True)
    g = torch.where(torch.rand(B, T, H, generator=torch.Generator().manual_seed(7)) < 0.5, g * 1.5e-4, g)
    run = lambda lo, hi, st: KH.kv_scan_stream(*(x[:, lo:hi].cuda() for x in (k, v, g, fr)), N, 16.0, G=8,
                                               q=q[:, lo:hi].cuda(), occ_bin=occb, state=st)
    kb, vb, st = run(0, T, None)
    okb, ovb, info = SO.scan_forward(np64(k), np64(v), np64(g), np64(fr), N, 16.0, G=8, hard=True, q=np64(q),
                                     occ_bin=occb)
    # every value of the state is a blend of at most T unit-scale tokens in fp32: 1e-5 of the largest
    for got, ref in ((kb, okb), (vb, ovb), (st[2].reshape(B, H, N), info["ofin"])):
        assert abs(np64(got) - ref).max() <= 1e-5 * abs(ref).max()
    assert ((np64(st[2]).reshape(B, H, N) >= 1e-4) == (info["ofin"] >= 1e-4)).all()
    # and in pieces that start and end inside a window
    st2, parts = None, []
    for lo, hi in ((0, 8), (8, 32), (32, 80)):
        p = run(lo, hi, st2)
        st2 = p[2]
        parts.append(p[0])
    assert abs(np64(torch.cat(parts, 1)) - okb).max() <= 1e-5 * abs(okb).max()
