"""tpt_guide_infer at the edges of its tiles: 16-row groups, 128-row blocks, one
grid of blocks, and output rows that are not 16-byte aligned.  A row's outputs
do not depend on the batch it is in, so every size must give the same bits as
the rows of one large batch (checked against the oracle in test_gpu_guide)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 127, 128, 129, 1280 * 128 - 1, 1280 * 128 + 1])
@pytest.mark.parametrize("offset", [0, 1])
def test_infer_rows_do_not_depend_on_the_batch(tpt, device, n, offset):
    import torch

    g = tpt.Guide(seed=3)
    rng = np.random.default_rng(4)
    x = rng.uniform(-1, 1, (200000, 9)).astype(np.float32)
    xt = torch.from_numpy(x).to(device)
    want = g.infer(xt)
    first = 200000 - n if n < 1000 else 0
    rows = xt[first:first + n].contiguous()
    buf = torch.full((n * 40 + 8,), -7.0, dtype=torch.float32, device=device)
    L = tpt.lib()
    rc = L.tpt_guide_infer(g.h, rows.data_ptr(), n, buf.data_ptr() + 4 * offset, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    got = buf[offset:offset + n * 40].view(n, 40)
    assert torch.equal(got, want[first:first + n])
    assert bool((buf[offset + n * 40:] == -7.0).all()) and bool((buf[:offset] == -7.0).all())
