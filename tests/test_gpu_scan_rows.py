"""The row backward's counted-load variant where T cuts the last 16-step chunk short and where a chunk holds one
snapshot (G = 16), against the fp64 oracle with the bars of the scan and writer-epilogue checks they reuse."""
import pytest
import torch

from test_gpu_scan import check_case
from test_gpu_scan_mem import _check, _check_q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [7, 8, 9, 15, 16, 17, 24, 25, 40, 63])
@pytest.mark.parametrize("G,D", [(8, 64), (8, 128), (16, 128), (16, 64)])
def test_rows_bwd_short_last_chunk(T, G, D):
    check_case(2, T, 1, 33, D, G, True, True, True, False, seed=600 + T,
               dtype=torch.bfloat16 if T % 2 else torch.float32)


@pytest.mark.parametrize("T,G", [(9, 8), (24, 8), (40, 8), (41, 8), (15, 16), (32, 16), (50, 16)])
def test_rows_bwd_short_last_chunk_epilogue(T, G):
    _check(2, T, 2, 40, 128, G, True, True, True, False, seed=700 + T)


@pytest.mark.parametrize("T,G", [(24, 8), (41, 8), (50, 16)])
def test_rows_bwd_short_last_chunk_quantised(T, G):
    _check_q(2, T, 2, 40, 128, G, True, True, True, False, 3, 16, seed=800 + T)
