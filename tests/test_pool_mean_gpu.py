"""Mean pooling with many rows at once: widths that fill 1024 threads and that don't, counts around the rows in flight."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("D", [8, 384, 768, 1000, 1024, 2048, 2056])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_mean(D, dtype):
    lens = [1, 2, 7, 8, 9, 31, 32, 33, 65, 512, 0, 3]
    g = torch.Generator(device="cuda").manual_seed(D)
    h = torch.randn(sum(lens), D, device="cuda", generator=g).to(dtype)
    cu = torch.tensor([0] + lens, device="cuda").cumsum(0).int()
    fn = K.pool_l2norm if dtype == torch.bfloat16 else K.pool_l2norm_f16
    got = fn(h, cu, 1)
    for b, n in enumerate(lens):
        rows = h[int(cu[b]):int(cu[b]) + max(n, 1)].double()  # (an empty text: the row that follows)
        want = torch.nn.functional.normalize(rows.mean(0), dim=0)
        # sums of up to 512 terms and of D squares in fp32, the reciprocal root to 2^-22
        scale = rows.abs().mean(0) / rows.mean(0).norm()
        assert ((got[b].double() - want).abs() <= (n + 8) * 2.0 ** -24 * scale + (D + 8) * 2.0 ** -22 * want.abs()).all()
