"""A context whose tensors are uploaded and finalized again (include/mlh.h) against a context that only ever had the new ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def config(pkg, bf16=0, **kw):
    hp = pkg.config(3, dim=256, attnHeads=4, headDim=64, ffnDim=704, transformers=4, vocabSize=1000, gdnHeads=4, pleDim=64, maxL=160,
                    weightDtype=bf16, **kw)
    pkg.set_layer_pattern(hp, 1)
    return hp


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("nseq,graph", [(1, 1), (3, 1), (3, 4), (9, 2)])
def test_graphs_follow_a_repeated_finalize(pkg, bf16, nseq, graph):
    """A finalize replaces the operands whose addresses a captured step holds: the next decode must not replay the old capture."""
    hp = config(pkg, bf16, maxSeqs=nseq)
    old, new = (pkg.Model.generate(hp, seed).randomize_gains(seed) for seed in (5, 6))
    prompts = [pkg.random_tokens(5, s, hp.vocabSize, 20 + 3 * s) for s in range(nseq)]

    def decode(dev):
        dev.reset()
        dev.prefill_batch(list(range(nseq)), prompts)
        firsts = [dev.greedy_token(s) for s in range(nseq)]
        runs = [dev.decode_loop(firsts, 9)]  # whole replays and a remainder
        for _ in range(2):
            dev.synchronize()
            runs.append(dev.decode_loop(runs[-1][-1], 9))
        return np.concatenate(runs), np.stack([dev.logits(s) for s in range(nseq)])

    def device(model):
        dev = pkg.Device(hp, 0)
        dev.set_persistent(0)
        dev.set_graph(graph)
        dev.upload(model)
        return dev

    dev = device(old)
    before = decode(dev)
    dev.upload(new)
    got = decode(dev)
    dev.close()
    dev = device(new)
    want = decode(dev)
    dev.close()
    assert not np.array_equal(before[1], want[1])
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


@pytest.mark.parametrize("bf16", [0, 1])
def test_without_copies_of_the_matrices(pkg, bf16):
    """A context that may not spend memory on them (or has none left for them) answers as the token-by-token path does."""
    hp = config(pkg, bf16, maxSeqs=3)
    model = pkg.Model.generate(hp, 5).randomize_gains(5)
    prompts = [pkg.random_tokens(5, s, hp.vocabSize, n) for s, n in enumerate((20, 70, 1))]

    def answers(dev):
        out = []
        dev.reset()
        out.extend(dev.forward_full(0, prompts[1]))
        dev.reset()
        dev.prefill_batch([0, 1, 2], prompts)
        out.append(dev.decode_loop([dev.greedy_token(s) for s in range(3)], 6))
        out.append(np.stack([dev.logits(s) for s in range(3)]))
        dev.reset()
        dev.prefill(0, prompts[0])
        out.append(dev.decode_loop([3], 6))
        out.append(dev.logits(0))
        return out

    dev = pkg.Device(hp, 0)
    dev.upload(model)
    d, per = hp.dim, 4 if bf16 else 10
    rows = sum((d * 3 if hp.layerKinds[t] == 0 else d * 3 + 8) + hp.pleDim for t in range(4))
    exact = ((1000 + rows + 4 * 2 * hp.ffnDim) * d + 4 * d * (d + hp.pleDim + hp.ffnDim)) * per + 4 * d * (d + hp.pleDim) * (2 if bf16 else 4)
    full = dev.operand_bytes()
    assert exact <= full <= exact * 1.02  # (packed rows are padded to 16)
    fast = answers(dev)
    dev.set_prefill_mode(1)
    want = answers(dev)
    dev.set_prefill_mode(0)
    for limit in (0, full - full // 16):
        dev.limit_operands(limit)
        dev.finalize()
        assert dev.operand_bytes() == 0
        for a, b in zip(answers(dev), want):
            assert np.array_equal(a, b)
    dev.limit_operands(2 * full)
    dev.finalize()
    assert dev.operand_bytes() == full
    for a, b in zip(answers(dev), fast):
        assert np.array_equal(a, b)
    dev.close()


@pytest.mark.parametrize("bf16", [0, 1])
def test_room_for_a_prefill_over_every_position(pkg, bf16):
    """What finalize keeps free for prefill calls is what the largest one allocates: to 2 % and the granularity of a dozen allocations (2 MB each)."""
    import torch

    hp = pkg.config(3, dim=512, attnHeads=4, headDim=128, ffnDim=512, transformers=2, vocabSize=256, gdnHeads=16, gdnDk=128, gdnDv=128, pleDim=64,
                    maxL=2100, maxSeqs=8, weightDtype=bf16)
    pkg.set_layer_pattern(hp, 1)
    dev = pkg.Device(hp, 0)
    dev.upload(pkg.Model.generate(hp, 5))
    before = torch.cuda.mem_get_info()[0]
    dev.prefill_batch(list(range(8)), [pkg.random_tokens(5, s, hp.vocabSize, hp.maxL) for s in range(8)])
    took = before - torch.cuda.mem_get_info()[0]
    assert abs(took - dev.prefill_bytes()) <= 0.02 * took + (24 << 20), (took, dev.prefill_bytes())
    dev.close()


@pytest.mark.parametrize("bf16", [0, 1])
def test_a_limit_just_below_the_copies(pkg, bf16):
    """What the copies take never exceeds the limit, their rows' exponents included (widths of whole tiles: no padding in between)."""
    hp = pkg.config(3, dim=512, attnHeads=8, headDim=64, ffnDim=1024, transformers=2, vocabSize=1024, gdnHeads=8, pleDim=64, maxL=100, maxSeqs=2, weightDtype=bf16)
    pkg.set_layer_pattern(hp, 1)
    dev = pkg.Device(hp, 0)
    dev.upload(pkg.Model.generate(hp, 5))
    full = dev.operand_bytes()
    for limit in (full - 1, full - 4096):
        dev.limit_operands(limit)
        dev.finalize()
        assert dev.operand_bytes() <= limit
    dev.close()
