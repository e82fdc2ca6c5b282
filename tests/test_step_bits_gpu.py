"""What a float32 engine's result depends on: a row's own sequence, not who shares a step with it nor how it was cut into
steps, also where layers keep a state of fixed size."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("name", ["A", "C", "D"])
@pytest.mark.parametrize("model", ["kunitar", "luduvik", "saredra"])
def test_float32_bits_of_models_with_matrix_states(model, name):
    """A prompt of 40 tokens and three more, alone, beside shorter, longer and many sequences, beside prompts that come in while
    it decodes, and in pieces: the same logits bit for bit."""
    from transformer_amd import Entry
    U = importlib.import_module(model + "_util")
    engine, toks = U.engine(name, "float32"), [[int(t) for t in U.tokens(name, 64, 50 + i)] for i in range(6)]

    def run(cuts, beside):
        cache = engine.new_cache(64 * 24, max_slots=8)
        at, slots, out = [0] * (1 + len(beside)), [cache.alloc_slot() for _ in range(1 + len(beside))], []
        for i, n in enumerate(cuts):
            entries = []
            for j, s in enumerate(slots):
                m = n if j == 0 else beside[j - 1][i]
                if m:
                    entries.append(Entry(s, toks[j][at[j]:at[j] + m], range(m)))
                    at[j] += m
            out.append(engine.step(cache, entries)[:n].float().cpu().numpy())
        return np.concatenate(out)

    want = run([40, 1, 1, 1], [])
    for beside in ([[9, 1, 1, 1]], [[50, 1, 1, 1], [40, 3, 1, 1], [30, 1, 12, 1]], [[40, 1, 1, 1]] * 5):
        assert np.array_equal(run([40, 1, 1, 1], beside), want)
    for cuts in ([20, 20, 1, 1, 1], [7, 33, 1, 1, 1], [1] * 43):
        assert np.array_equal(run(cuts, []), want)


@pytest.mark.parametrize("lens", [[1] * 8, [3, 40], [200]])
def test_float32_gates_of_the_diagonal_recurrence(lens):
    """Decays and inputs of a step's tokens, and of the same tokens one by one in steps of their own."""
    from transformer_amd import kernels as K
    nb, size = 2, 128
    C, nt, B = nb * size, sum(lens), len(lens)
    g = torch.Generator(device=DEV).manual_seed(nt)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    yx, gw, xb, cb, lam, gb, tp, mem = r(nt, 2 * C), r(2 * nb, size, size) / size ** 0.5, r(C), r(C), r(C), r(2 * nb, size), r(C, 4), r(B, 3, C)
    cu = np.concatenate([[0], np.cumsum(lens)])

    def gates(rows, bounds, slots):
        a, b = torch.empty(len(rows), C, device=DEV), torch.empty(len(rows), C, device=DEV)
        K.rglru_gates(rows, C, xb, tp, cb, mem, gw, gb, lam, 8.0, torch.tensor(bounds, dtype=torch.int32, device=DEV),
                      torch.tensor(slots, dtype=torch.int32, device=DEV), a, b)
        return a, b

    whole = gates(yx, cu.tolist(), list(range(B)))
    for i in range(B):                                            # every sequence's first four tokens by themselves
        n = min(lens[i], 4)
        for got, want in zip(gates(yx[cu[i]:cu[i] + n].contiguous(), [0, n], [i]), whole):
            assert torch.equal(got, want[cu[i]:cu[i] + n])
