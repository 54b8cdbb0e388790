"""The row step (csrc/kernels_rows.hip: decode of up to 64 sequences) at the edges of its token blocks, chunks and tiles, against
the GEMV kernels (prefill mode 1), which other tests hold against the float64 oracle: both are fp32 sums of the same products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


# d, ffn, vocab: fewer chunks of K than waves; CNT 1 and 3 with a ragged last tile of vocabulary rows; the streaming form; bf16
@pytest.mark.parametrize("bf16,d,ffn,vocab", [(0, 64, 96, 1000), (0, 256, 704, 4096), (0, 768, 2048, 501), (1, 128, 192, 777), (1, 1024, 2816, 2048), (1, 2048, 5632, 512)])
@pytest.mark.parametrize("nseq", [1, 2, 5, 8, 9, 16, 17, 33, 64])
def test_rows_against_gemv(pkg, bf16, d, ffn, vocab, nseq):
    hp = pkg.config(3, dim=d, attnHeads=d // 64, headDim=64, ffnDim=ffn, transformers=2, vocabSize=vocab, gdnHeads=d // 64, pleDim=64,
                    maxL=24, maxSeqs=nseq, weightDtype=bf16)
    pkg.set_layer_pattern(hp, 1)
    model = pkg.Model.generate(hp, 5)
    model.randomize_gains(5)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    dev.set_persistent(0)
    rng = np.random.default_rng(nseq)
    feed = rng.integers(0, vocab, (3, nseq)).astype(np.int32)
    out = {}
    for mode in (1, 0):
        dev.reset()
        dev.set_prefill_mode(1)
        dev.prefill_batch(list(range(nseq)), [feed[0, s:s + 1] for s in range(nseq)])
        dev.set_prefill_mode(mode)
        picks = [dev.decode_step(f) for f in feed[1:]]
        run = dev.decode_loop(picks[-1], 4)  # steps that embed the next one's tokens
        out[mode] = (np.stack(picks), run, np.stack([dev.logits(s) for s in range(nseq)]))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    assert rel(out[0][2], out[1][2]) < 3e-6
    dev.close()
