"""pm_scan_u32 around its tiles' edges and at 4,194,304 elements, where the
two-level form begins, inclusive and exclusive, from addresses
that are and are not 16-byte aligned: whole numbers, equal to numpy's sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 4095, 4097, 8191, 8192, 8193, 262_145, 4_186_113, 4_194_303, 4_194_304, 4_194_305]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("inclusive", [False, True])
def test_edges(ctx, n, off, inclusive):
    import torch

    a = np.random.default_rng(n).integers(0, 1 << 20, n + off, dtype=np.uint32)
    x = torch.from_numpy(a.view(np.int32)).cuda()[off:]
    out, tot = ctx.scan_u32(x, inclusive=inclusive, with_total=True)
    ctx.sync()
    s = np.cumsum(a[off:], dtype=np.uint32)
    want = s if inclusive else np.concatenate([[np.uint32(0)], s[:-1]])
    assert np.array_equal(out.cpu().numpy().view(np.uint32), want)
    assert int(tot.item()) & 0xFFFFFFFF == int(s[-1])
