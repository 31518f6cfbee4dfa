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


@pytest.mark.parametrize("D", [8, 384, 1000, 1024, 2048])
@pytest.mark.parametrize("B,lens", [(512, [3]), (513, [1]), (700, [1, 2, 3]), (600, [12, 13]), (520, [60, 0, 3, 200])])
def test_many_texts(D, B, lens):
    """Workgroups sized by the mean length: of one row to more rows than texts have, around the count where that begins."""
    lens = [lens[i % len(lens)] for i in range(B)]
    g = torch.Generator(device="cuda").manual_seed(D + B)
    h = torch.randn(sum(lens) + 1, D, device="cuda", generator=g).bfloat16()
    cu = torch.tensor([0] + lens, device="cuda").cumsum(0).int()
    got = K.pool_l2norm(h, cu, 1).double()
    seg = torch.repeat_interleave(torch.arange(B, device="cuda"), torch.tensor(lens, device="cuda"))
    n = torch.tensor(lens, device="cuda").double()[:, None].clamp_min(1)
    mean, mag = (torch.zeros(B, D, device="cuda", dtype=torch.float64).index_add_(0, seg, x[:sum(lens)].double()) / n
                 for x in (h, h.abs()))
    empty = (torch.tensor(lens, device="cuda") == 0)[:, None]
    first = h[cu[:-1].long()].double()  # (an empty text: the row that follows)
    mean, mag = torch.where(empty, first, mean), torch.where(empty, first.abs(), mag)
    want = torch.nn.functional.normalize(mean, dim=1)
    # (as above)
    scale = mag / mean.norm(dim=1, keepdim=True)
    assert ((got - want).abs() <= (n + 8) * 2.0 ** -24 * scale + (D + 8) * 2.0 ** -22 * want.abs()).all()
