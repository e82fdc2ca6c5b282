"""What latent attention keeps of the matrices it is bound with: no GPU is needed."""
import pytest
import torch

from transformer_amd.config.spec import LatentAttentionSpec
from transformer_amd.parts.base import build_part

BF = torch.bfloat16


def _off(t, start, extra):
    """The same values at ``start`` numbers behind 16 bytes, in rows ``extra`` numbers longer."""
    n, k = t.shape
    return torch.zeros(n * (k + extra) + 8, dtype=t.dtype)[start:start + n * (k + extra)].view(n, k + extra)[:, :k].copy_(t)


@pytest.mark.parametrize("start,extra", [(0, 0), (1, 0), (4, 0), (0, 8), (3, 5)])
def test_the_heads_maps_lie_in_whole_pieces(start, extra):
    H, dn, dv, rank, d = 3, 24, 16, 40, 64
    spec = LatentAttentionSpec(hidden=d, num_heads=H, nope_dim=dn, rope_dim=0, value_dim=dv, q_rank=None, kv_rank=rank, scale=0.1,
                               eps=1e-5, rot_dims=0, rot_base=1e4)
    part = build_part(spec, BF, torch.device("cpu"))
    g = torch.Generator().manual_seed(start + extra)
    tensors = {n: torch.randn(*p.shape, generator=g).to(torch.float32 if p.role == "vector" else BF) for n, p in part.params().items()}
    uk, uv = tensors["uk.weight"].view(H, dn, rank), tensors["uv.weight"].view(H, dv, rank)
    for n in ("uk.weight", "uv.weight"):
        tensors[n] = _off(tensors[n], start, extra)
        assert (tensors[n].data_ptr() % 16 == 0) == (start == 0) and tensors[n].is_contiguous() == (extra == 0)
    part.bind(tensors)
    for got, want in ((part.uk_op, uk), (part.uv_op, uv.transpose(1, 2))):
        assert torch.equal(got, want) and got.is_contiguous() and got.data_ptr() % 16 == 0
    assert (part.uk_op.data_ptr() == tensors["uk.weight"].data_ptr()) == (start == 0 and extra == 0)     # no copy without a reason
