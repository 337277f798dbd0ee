"""The stand-alone sort with the launch shape it chooses itself, on both sides of every size and key width at
which the choice changes, against a stable sort on the host."""
import numpy as np
import pytest
import torch

from torpedo_amd.engine import GaussianEngine, sort_pairs_device

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [65_535, 65_537, 524_287, 524_289, 1_499_999, 1_500_001, 3_145_728, 3_145_729])
@pytest.mark.parametrize("bits", [17, 27, 32, 64])  # 9-bit digits save a pass at 17 and 27 bits
def test_chosen_shape(n, bits):
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 2 ** bits, n, dtype=np.uint64, endpoint=False)
    keys[n // 3:n // 2] = keys[n // 3]  # a run of equal keys keeps its order
    eng = GaussianEngine()
    k = torch.from_numpy(keys.view(np.int64)).cuda()
    v = torch.arange(n, dtype=torch.int32, device="cuda")
    ka, va = torch.empty_like(k), torch.empty_like(v)
    torch.cuda.synchronize()
    in_alt = sort_pairs_device(eng, k.data_ptr(), v.data_ptr(), ka.data_ptr(), va.data_ptr(), n, bits)
    torch.cuda.synchronize()
    order = np.argsort(keys, kind="stable")
    assert np.array_equal((va if in_alt else v).cpu().numpy(), order)
    assert np.array_equal((ka if in_alt else k).cpu().numpy().view(np.uint64), keys[order])
    eng.close()
