"""Short prefills through the row kernels, the LM head of every prefill and forward_full's way out, against the token-by-token
path (prefill mode 1), which other tests hold against the float64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


def device(pkg, **kw):
    hp = pkg.config(3, transformers=2, maxL=320, queryGating=1, qkRmsNorm=1, **kw)
    pkg.set_layer_pattern(hp, 1)
    model = pkg.Model.generate(hp, 5)
    model.randomize_gains(5)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    return dev


@pytest.mark.parametrize("bf16,hd", [(0, 64), (0, 128), (1, 64), (1, 128)])
@pytest.mark.parametrize("lens", [[2], [1, 1], [15], [16], [5, 1, 27], [33], [1, 63], [40, 25], [1] * 65])
def test_short_prefill_against_steps(pkg, bf16, hd, lens):
    dev = device(pkg, dim=256, attnHeads=256 // hd, headDim=hd, ffnDim=704, vocabSize=1000, gdnHeads=256 // hd, gdnDk=hd, gdnDv=hd,
                 pleDim=64, maxSeqs=len(lens), weightDtype=bf16)
    rng = np.random.default_rng(sum(lens))
    calls = [[rng.integers(0, 1000, n).astype(np.int32) for n in ls] for ls in (lens, lens[::-1])]  # and once more behind the first call
    seqs = list(range(len(lens)))
    out = {}
    for mode in (1, 0):
        dev.reset()
        dev.set_prefill_mode(mode)
        out[mode] = []
        for ids in calls:
            dev.prefill_batch(seqs, ids)
            lg = np.stack([dev.logits(s) for s in seqs])
            assert [dev.greedy_token(s) for s in seqs] == list(lg.argmax(1))
            out[mode].append(lg)
    precise = not bf16 or sum(lens) < 16
    for a, b in zip(out[0], out[1]):
        assert rel(a, b) < (1e-5 if precise else 3e-3)
    dev.close()


@pytest.mark.parametrize("bf16,vocab,n", [(0, 1000, 2), (0, 501, 64), (1, 777, 15), (1, 777, 32), (0, 20001, 60), (0, 20001, 300)])
def test_forward_full_against_steps(pkg, bf16, vocab, n):
    dev = device(pkg, dim=128, attnHeads=2, headDim=64, ffnDim=192, vocabSize=vocab, gdnHeads=2, pleDim=64, maxSeqs=1, weightDtype=bf16)
    ids = np.random.default_rng(n).integers(0, vocab, n).astype(np.int32)
    out = {}
    for mode in (1, 0):
        dev.reset()
        dev.set_prefill_mode(mode)
        out[mode] = dev.forward_full(0, ids)
    tol = 1e-5 if not bf16 or n < 16 else 3e-3
    assert rel(out[0][0], out[1][0]) < tol and rel(out[0][1], out[1][1]) < tol
    assert np.allclose(out[0][1].sum(1), 1, atol=1e-4)
    assert abs(out[0][2] - out[1][2]) < 1e-3
    dev.close()


@pytest.mark.parametrize("lens", [[34], [47], [64], [20, 31], [17, 1, 40]])
def test_tiles_of_33_to_64_halves_against_steps(pkg, lens):
    """Models of halves multiply 33 to 64 rows as one row of 64 x 64 tiles, K split or not, whose last rows are past the end.  Bound: that of the calls above (three
    roundings to half, 2^-11, on the way through each of two layers)."""
    dev = device(pkg, dim=512, attnHeads=8, headDim=64, ffnDim=1472, vocabSize=1000, gdnHeads=8, gdnDk=64, gdnDv=64, pleDim=64, maxSeqs=len(lens), weightDtype=1)
    rng = np.random.default_rng(sum(lens))
    ids = [rng.integers(0, 1000, n).astype(np.int32) for n in lens]
    seqs, out = list(range(len(lens))), []
    for mode in (1, 0):
        dev.reset()
        dev.set_prefill_mode(mode)
        dev.prefill_batch(seqs, ids)
        out.append(np.stack([dev.logits(s) for s in seqs]))
    assert rel(out[1], out[0]) < 3e-3
    dev.close()


@pytest.mark.parametrize("bf16,hd,lens", [(1, 64, [70, 20]), (1, 128, [64, 63, 1]), (1, 64, [150]), (0, 64, [1, 30, 20]), (1, 128, [3, 20])])
def test_embedding_columns_of_mixed_segments_against_steps(pkg, bf16, hd, lens):
    """The per-layer embedding's columns come from workgroups beside the heads': chunked segments (64 tokens and more), recurrent ones and the row kernels.  Bounds: as above."""
    dev = device(pkg, dim=256, attnHeads=256 // hd, headDim=hd, ffnDim=704, vocabSize=1000, gdnHeads=256 // hd, gdnDk=hd, gdnDv=hd, pleDim=128, maxSeqs=len(lens), weightDtype=bf16)
    rng = np.random.default_rng(sum(lens))
    ids = [rng.integers(0, 1000, n).astype(np.int32) for n in lens]
    seqs, out = list(range(len(lens))), []
    for mode in (1, 0):
        dev.reset()
        dev.set_prefill_mode(mode)
        dev.prefill_batch(seqs, ids)
        out.append(np.stack([dev.logits(s) for s in seqs]))
    assert rel(out[1], out[0]) < (3e-3 if bf16 else 1e-5)
    dev.close()
