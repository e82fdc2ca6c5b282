"""float32 models wide enough for the products of up to 8 rows that take the norm in front or the add behind: a row's bits follow
from its own sequence whatever shares its steps."""
import numpy as np
import pytest

import plain_linonex
import plain_llama
import plain_saredra

pytestmark = pytest.mark.gpu


def _engine(plain, cfg, seed, folder):
    import transformer_amd as ta
    plain.make_model_folder(folder, cfg, seed, storage="F32")
    return ta.load_model(str(folder), "float32", "cuda:0")


def _logits(engine, tokens, cuts, beside=0):
    """Logits of a sequence given in steps of ``cuts`` tokens, beside others that bring a token each step."""
    from transformer_amd import Entry
    cache = engine.new_cache(64 * 16, max_slots=16)
    slots, at, out = [cache.alloc_slot() for _ in range(1 + beside)], 0, []
    for n in cuts:
        entries = [Entry(slots[0], tokens[at:at + n], range(n))]
        entries += [Entry(s, [tokens[(at + i) % len(tokens)]], []) for i, s in enumerate(slots[1:])]
        out.append(engine.step(cache, entries)[:n].float().cpu().numpy())
        at += n
    return np.concatenate(out)


def _tokens(vocab, n):
    return [int(t) for t in np.random.default_rng(1).integers(0, vocab, n)]


# a feed-forward whose product adds itself to the stream, in front of rows that join it before the next pass: eight rows and nine
@pytest.mark.parametrize("stop", [1, 2, 3])
def test_loops_with_wide_feed_forwards(tmp_path, stop):
    memory = {"type": "mlstm", "mixer": {"heads": 2, "dim": 16, "vdim": 12, "gate_cap": 8.0}}
    cfg = {"architecture": "Linonex", "vocab": 60, "width": 72, "max_positions": 100, "norm": {"eps": 1e-5},
           "loop": {"start": 0, "stop": stop, "times": 3},
           "layers": [{**memory, "mlp": {"kind": "dense", "ff": ff}} for ff in (1540, 2048, 4100)]}
    engine = _engine(plain_linonex, cfg, 5, tmp_path)
    from transformer_amd import kernels
    assert all(kernels.add_takes(8, b.ffn.w["down.weight"]) and not kernels.add_takes(9, b.ffn.w["down.weight"]) for b in engine.blocks)
    tokens = _tokens(60, 12)
    want = _logits(engine, tokens, [1] * 12)
    for beside in (3, 7, 8, 11):
        assert np.array_equal(_logits(engine, tokens, [1] * 12, beside), want), beside


# hidden sizes whose products go over the norm by four waves' rows and by eight
def _llama(hidden, layers=2):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": layers, "hidden_size": hidden,
            "num_attention_heads": 12, "num_key_value_heads": 2, "head_dim": 128, "intermediate_size": 1600, "vocab_size": 300,
            "rope_theta": 5e5, "rms_norm_eps": 1e-5, "tie_word_embeddings": False, "max_position_embeddings": 256}


def _saredra(width):
    m = {"heads": 12, "kv_heads": 2, "dim": 16, "vdim": 128, "scale": 0.25, "rot": {"base": 1000.0, "dims": 6}}
    return {"architecture": "Saredra", "vocab": 300, "width": width, "norm": {"eps": 1e-5},
            "layers": [{"type": "attention", "mixer": m, "mlp": {"kind": "dense", "ff": ff}} for ff in (2000, 1600)]}


def _linonex(width):
    m = {"heads": 12, "dim": 16, "vdim": 128, "gate_cap": 8.0}
    return {"architecture": "Linonex", "vocab": 300, "width": width, "max_positions": 100, "norm": {"eps": 1e-5},
            "loop": {"start": 0, "stop": 2, "times": 2},
            "layers": [{"type": "mlstm", "mixer": m, "mlp": {"kind": "dense", "ff": ff}} for ff in (1600, 1540)]}


@pytest.mark.parametrize("plain,cfg", [(plain_llama, _llama(1536)), (plain_llama, _llama(2044)), (plain_llama, _llama(3072)),
                                       (plain_saredra, _saredra(1536)), (plain_linonex, _linonex(2048))],
                         ids=["llama-1536", "llama-2044", "llama-3072", "saredra-1536", "linonex-2048"])
def test_norms_inside_the_products(tmp_path, monkeypatch, plain, cfg):
    """Up to eight rows, eagerly and in a recorded step, the products go over the norms in front of them and add themselves to the
    stream; nine rows take the norm's own kernel and leave the add to it."""
    from transformer_amd import kernels
    engine = _engine(plain, cfg, 4, tmp_path)
    rows = {}
    for name in ("gemm_normed", "gemm_add"):
        def counted(*a, _call=getattr(kernels, name), _name=name, **kw):
            n = (a[0].x if _name == "gemm_normed" else a[0]).shape[0]
            rows.setdefault(_name, set()).add(n)
            return _call(*a, **kw)
        monkeypatch.setattr(kernels, name, counted)
    tokens = _tokens(300, 12)
    # the matrix memory takes a piece's tokens together: there the sequence comes token by token beside others
    if plain is plain_linonex:
        want = _logits(engine, tokens, [1] * 12, 8)
        others = [([1] * 12, beside) for beside in (0, 2, 3, 7)]
    else:
        want = _logits(engine, tokens, [12])
        others = [([1] * 12, 0), ([8, 4], 0), ([9, 3], 0), ([1] * 12, 7), ([1] * 12, 8), ([3, 9], 5)]
    assert not rows
    for cuts, beside in others:
        assert np.array_equal(_logits(engine, tokens, cuts, beside), want), (cuts, beside)
    assert rows["gemm_normed"] >= {1, 3, 4, 8} and rows["gemm_add"] >= {1, 3, 4} and max(max(r) for r in rows.values()) == 8


def test_norm_weights_that_start_off_16_bytes(tmp_path):
    """A product does not go over such a norm; the norm's own kernel takes it, in steps of any size."""
    import torch
    engine = _engine(plain_llama, _llama(1536), 3, tmp_path)
    tokens = _tokens(300, 12)
    want = _logits(engine, tokens, [12])
    tensors = dict(engine.tensors)
    for n, t in tensors.items():
        if "norm" in n:
            tensors[n] = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].copy_(t)
            assert tensors[n].data_ptr() % 16 == 4
    engine.bind(tensors)
    got = _logits(engine, tokens, [12])
    # the same formulas with the squares of a row added in another order
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    for cuts, beside in (([1] * 12, 0), ([8, 4], 0), ([9, 1, 1, 1], 7)):
        assert np.array_equal(_logits(engine, tokens, cuts, beside), got), cuts
