"""float32 models wide enough for the products of up to 8 rows that take the norm in front or the add behind: a row's bits follow
from its own sequence whatever shares its steps."""
import numpy as np
import pytest

import plain_linonex
import plain_llama

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
