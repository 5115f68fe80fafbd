"""Delta rule step with more heads and batch rows than the chip has CUs, where the kernel takes fewer registers."""

import pytest
import torch

from tests.test_zufadra_ops_gpu import Y_REL, _close, _Delta

pytestmark = pytest.mark.gpu

# (heads, kv_heads, dk, dv, taps, ranks of decay and gate): four rows of S per thread, eight, edges of both, and a size that stays with one workgroup per CU
SIZES = [(4, 2, 64, 64, 4, 16, 8), (4, 4, 128, 128, 4, 128, 128), (4, 1, 100, 72, 2, 72, 136), (8, 1, 16, 4, 1, 8, 8), (2, 2, 256, 128, 4, 64, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", range(len(SIZES)))
@pytest.mark.parametrize("more", [0, 1])
def test_one_workgroup_per_cu_and_two(case, more, dtype):
    d = _Delta(dtype, *SIZES[case], seed=case)
    batch = torch.cuda.get_device_properties(0).multi_processor_count // d.heads + more
    pads = torch.zeros(batch, dtype=torch.int64)
    pads[batch // 2] = 2
    proj = d.inputs(batch, 5)
    y, s = d.run(proj, [1, 3, 1], pads)
    for b in (0, 1, batch // 2, batch - 1):
        ref, s_ref = d.reference(proj[b, pads[b]:])
        _close(y[b, pads[b]:], ref, Y_REL[dtype], b)
        _close(s[b], s_ref, 2e-5, b)
