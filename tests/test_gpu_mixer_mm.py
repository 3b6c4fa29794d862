"""The mixers' many-token kernels at the edges of their tiles, through the C
ABI against the oracle, with the bars of tests/test_gpu_deltanet.py and
tests/test_gpu_attention.py (outputs 2e-2 max-abs and 1e-3 relative L2,
states and caches 1e-4; the indexer bit for bit)."""
import pytest

import test_gpu_attention as ta
import test_gpu_deltanet as td

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_dev(gpu):
    import torch
    return torch, gpu


# token counts around the first matrix call, the 32- and 64-row tiles and the
# K-split kernel's last count; hidden 320 and 448 have odd numbers of groups
@pytest.mark.parametrize("shape", [(320, 1, 2, 32, 32, 7), (448, 3, 6, 64, 64, 5), (256, 2, 4, 128, 128, 16)])
@pytest.mark.parametrize("calls", [[5, 6, 31], [32, 33, 1, 64], [65, 1, 129], [320, 1, 321]])
def test_deltanet_token_counts(torch_dev, shape, calls):
    torch, dev = torch_dev
    td.run_steps(torch, dev, shape, calls, seed=8)


@pytest.mark.parametrize("case", [(320, 5, 1, 64, 3, 68, 12, 3, 768, 1.0), (256, 4, 2, 64, 2, 64, 4096, 4, 768, 0.25)])
@pytest.mark.parametrize("calls", [[8, 9, 31], [32, 33, 1, 64], [65, 1, 129], [320, 1, 321]])
def test_attention_token_counts(torch_dev, case, calls):
    torch, dev = torch_dev
    ta.run_calls(torch, dev, case, calls, seed=9)
