"""float32 models wide enough for the products of up to 8 rows that take the norm in front or the add behind: a row's bits follow
from its own sequence whatever shares its steps."""
import numpy as np
import pytest

import plain_linonex

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
