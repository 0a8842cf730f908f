"""GPU tests of how the attention work is dealt out over workgroups: the launch order of the tiles, the key splits and
the variants that a shape selects, each at the sizes where its bookkeeping has an edge.  Every case is compared with the
oracle over all (batch, head) pairs at the operator's bar, so a tile that is visited twice, never, or for the
wrong pair shows."""
import pytest
import torch

from test_gpu_parity import fa, run_case  # noqa: F401  (fa is a fixture)

pytestmark = pytest.mark.gpu


# (pairs, length, head dim): one group or several, of equal or unequal size, pairs that divide over the XCDs or do not;
# grids that just fill two workgroups per CU (32 tiles x 16 pairs: the folded order) and just exceed that
@pytest.mark.parametrize("B,H,T,D", [(1, 136, 2048, 128), (1, 131, 2048, 128), (1, 24, 4096, 128), (1, 16, 4096, 32),
                                     (1, 15, 4300, 32), (3, 11, 2000, 16), (1, 1, 4096, 64)])
def test_launch_order(fa, B, H, T, D):
    torch.cuda.empty_cache()
    run_case(fa, B, H, T, T, D, seed=H + T, gate_mean=1.0)


# few query rows behind many keys: key splits that fill the chip once, also where one split more would not fit
@pytest.mark.parametrize("B,H,M,N,D", [(2, 16, 333, 1100, 32), (1, 8, 129, 3000, 64), (3, 7, 300, 2000, 16)])
def test_key_splits(fa, B, H, M, N, D):
    run_case(fa, B, H, M, N, D, seed=M + N, gate_mean=2.0)
