"""32-bit prompt attention with one, two and four waves for 16 rows: a sequence gives the same bits alone, where its few blocks are split, and
beside enough others that they are not, and its last token the same as a step of its own; and it is what 64 bits give."""
import pytest
import torch

from transformer_amd import kernels
from transformer_amd.parts.linear import Workspace

pytestmark = pytest.mark.gpu

PAGE = 64
OTHERS = [300] * 40          # 12,000 tokens: past every line of the rule at the heads below


def _g(*shape, seed=0):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, generator=gen, device="cuda")


def _exact(q, k, v, nh, nkv, scale, first, window, keep, chunk, cap, sink):
    """One sequence in 64 bits: q [n, nh, dk] at positions first .., k [t, nkv, dk], v [t, nkv, dv]."""
    q, k, v, g = q.double(), k.double(), v.double(), nh // nkv
    at = first + torch.arange(q.shape[0], device="cuda")[:, None]
    key = torch.arange(k.shape[0], device="cuda")[None]
    seen = key <= at
    if window:
        seen &= (key > at - window) | (key < keep)
    if chunk:
        seen &= key >= at // chunk * chunk
    out = []
    for h in range(nh):
        s = q[:, h] @ k[:, h // g].t() * scale
        s = cap * torch.tanh(s / cap) if cap else s
        s = s.masked_fill(~seen, -float("inf"))
        if sink is not None:
            s = torch.cat([s, sink[h].double().expand(s.shape[0], 1)], 1)
        p = torch.softmax(s, 1)
        out.append(p[:, :k.shape[0]] @ v[:, h // g])
    return torch.cat(out, 1)


@pytest.mark.parametrize("n,first", [(5, 0), (67, 61), (130, 0), (513, 64), (1021, 0)])
@pytest.mark.parametrize("nh,nkv,dk,dv,options", [(16, 4, 128, 128, {}), (8, 8, 64, 64, {"window": 100, "keep_first": 4}), (6, 2, 96, 48, {"softcap": 30.0, "sink": True}),
                                                  (8, 2, 48, 64, {"chunk": 96}), (12, 4, 64, 64, {"softcap": 20.0, "window": 64})])
def test_the_same_however_many_waves(n, first, nh, nkv, dk, dv, options):
    lens, cached = [n] + OTHERS, [first] + [0] * len(OTHERS)
    pages = [-(-(l + c) // PAGE) for l, c in zip(lens, cached)]
    perm = torch.randperm(sum(pages), generator=torch.Generator().manual_seed(n)).int()
    table = torch.zeros(len(lens), max(pages), dtype=torch.int32)
    for b, m in enumerate(pages):
        table[b, :m] = perm[sum(pages[:b]):sum(pages[:b]) + m]
    kc, vc = _g(sum(pages), nkv, PAGE, dk, seed=1), _g(sum(pages), nkv, dv, PAGE, seed=2)
    tail = (first + n) % PAGE
    if tail:                                       # keys that were never written
        last = int(table[0, pages[0] - 1])
        kc[last, :, tail:] = float("nan")
        vc[last, :, :, tail:] = float("nan")
    q, sink = _g(sum(lens), nh * dk, seed=3), _g(nh, seed=4) if options.get("sink") else None
    opt = {**options, "sink": sink}
    table, pos0 = table.cuda(), torch.tensor(cached, dtype=torch.int32, device="cuda")
    cu = torch.tensor([0] + lens, device="cuda").cumsum(0).int()
    scale = dk ** -0.5

    def run(rows, batch, cu_q, pos, longest, ws=None):
        out = torch.full((rows.shape[0], nh * dv), float("nan"), device="cuda")
        return kernels.attention_sink(rows, out, kc, vc, table[:batch].contiguous(), cu_q, pos, longest, nh, nkv, dk, dv, scale, ws=ws, **opt)

    alone = run(q[:n], 1, cu[:2].contiguous(), pos0[:1].contiguous(), n)
    beside = run(q, len(lens), cu, pos0, max(lens))
    assert torch.equal(alone, beside[:n])
    single = run(q[n - 1:n], 1, torch.tensor([0, 1], dtype=torch.int32, device="cuda"), pos0[:1] + n - 1, 1, Workspace("cuda"))
    assert torch.equal(single[0], alone[-1])
    own = table[0, :pages[0]].long()
    k = kc[own].transpose(1, 2).reshape(-1, nkv, dk)[:first + n]
    v = vc[own].permute(0, 3, 1, 2).reshape(-1, nkv, dv)[:first + n]
    want = _exact(q[:n].view(n, nh, dk), k, v, nh, nkv, scale, first, options.get("window"), options.get("keep_first", 0), options.get("chunk"),
                  options.get("softcap"), sink)
    # sums of up to 1,085 products in 32 bits, rounded 2^-24 each of either sign, and scores of some 4 with the same
    assert float((alone.double() - want).norm() / want.norm()) < 2e-6
