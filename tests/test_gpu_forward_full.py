"""mlh_forward_full's result buffers from call to call, resets of single sequences, and the bf16 prefill against the float64
oracle with bounds that follow from its roundings."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


def hybrid(pkg, **kw):
    args = dict(dim=256, attnHeads=4, headDim=64, ffnDim=704, transformers=4, vocabSize=1000, gdnHeads=4, pleDim=64, maxL=400)
    args.update(kw)
    hp = pkg.config(3, **args)
    pkg.set_layer_pattern(hp, 1)
    return hp


def test_forward_full_results_larger_and_smaller_than_what_is_kept(pkg):
    """Results of 550 MB (more than the 512 that stay with the context) between smaller calls with and without probabilities, each
    laid out anew: against prefill mode 1, which other tests hold against the float64 oracle."""
    V, n = 32768, 2100
    hp = hybrid(pkg, dim=64, attnHeads=1, ffnDim=96, transformers=2, vocabSize=V, gdnHeads=1, maxL=n + 50, maxSeqs=1)
    model = pkg.Model.generate(hp, 5).randomize_gains(5)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    ids = pkg.random_tokens(5, 0, V, n + 50)
    dev.set_prefill_mode(1)
    lg, pr, nll = dev.forward_full(0, ids[:n])
    dev.set_prefill_mode(0)
    for m, probs in ((300, True), (450, False), (n, True), (40, True), (700, False), (n, False), (300, True)):
        dev.reset()
        got = dev.forward_full(0, ids[:m], want_probs=probs)
        assert rel(got[0], lg[:m]) < 1e-5
        if probs:
            assert rel(got[1], pr[:m]) < 1e-5
        want = -np.log(np.maximum(pr[np.arange(m - 1), ids[1:m]], 1e-4)).mean()
        assert abs(got[2] - want) < 1e-5 * want
    assert abs(nll - -np.log(np.maximum(pr[np.arange(n - 1), ids[1:n]], 1e-4)).mean()) < 1e-4
    dev.close()


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("dk", [64, 128])
def test_reset_of_some_sequences(pkg, bf16, dk):
    """Resets touch only sequences in use: those emptied start anew, the others go on from their KV rows and GDN states."""
    n = 5
    hp = hybrid(pkg, attnHeads=256 // dk, headDim=dk, gdnHeads=256 // dk, gdnDk=dk, gdnDv=dk, maxSeqs=n, weightDtype=bf16)
    model = pkg.Model.generate(hp, 5).randomize_gains(5)
    first = [pkg.random_tokens(5, s, hp.vocabSize, 9 + 30 * s) for s in range(n)]
    second = [pkg.random_tokens(6, s, hp.vocabSize, 7 + 5 * s) for s in range(n)]

    def run(steps):
        dev = pkg.Device(hp, 0)
        dev.upload(model)
        out = steps(dev)
        dev.close()
        return out

    def mixed(dev):
        dev.prefill_batch(list(range(n)), first)
        dev.decode_loop([1] * n, 3)
        for s in (1, 3, 3):  # (3 is clean the second time)
            dev.reset(s)
        assert [dev.seq_len(s) for s in range(n)] == [len(first[s]) + 3 if s not in (1, 3) else 0 for s in range(n)]
        dev.prefill_batch([3, 1], [second[3], second[1]])
        dev.decode_loop([2] * n, 3)
        return [dev.logits(s) for s in range(n)]

    def alone(s):
        def steps(dev):
            if s not in (1, 3):
                dev.prefill_batch(list(range(n)), first)
                dev.decode_loop([1] * n, 3)
            else:
                dev.prefill_batch([3, 1], [second[3], second[1]])
            dev.decode_loop([2] * n, 3)
            return dev.logits(s)
        return run(steps)

    got = run(mixed)
    for s in range(n):
        assert np.array_equal(got[s], alone(s))


@pytest.mark.parametrize("kind", ["attn64", "attn128", "hybrid64", "hybrid128"])
@pytest.mark.parametrize("n", [12, 200, 390])
def test_bf16_prefill_against_oracle(pkg, orc, kind, n):
    """Logits of every position.  Up to 15 tokens activations stay fp32: 1e-5.  Longer prompts round the inputs of a layer's products
    to halves: two normed rows, the mixing output and the FFN units, and inside the mixing four operands (q, k, v and the
    probabilities or chunk matrices).  Eight roundings a layer, each with an error of at most 2^-11 / sqrt(3) of its row (rms) and
    independent of the others, move the residual rows by at most sqrt(8 layers) 2^-11 / sqrt(3)."""
    hd = int(kind[-3:]) if kind.endswith("128") else 64
    hp = hybrid(pkg, attnHeads=256 // hd, headDim=hd, gdnHeads=256 // hd, gdnDk=hd, gdnDv=hd, maxSeqs=1, weightDtype=1)
    pkg.set_layer_pattern(hp, 1 if kind.startswith("hybrid") else 0)
    model = pkg.Model.generate(hp, 5).randomize_gains(5)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    ids = pkg.random_tokens(5, 0, hp.vocabSize, n)
    want = orc.forward_full(orc.Weights.from_model(model, bf16=True), ids, "f64", last_only=False)["logits"]
    got = dev.forward_full(0, ids, want_probs=False)[0]
    err = rel(got, want)
    print(f"{kind} {n}: {err:.2e}")
    assert err < (1e-5 if n < 16 else np.sqrt(8 * hp.transformers) * 2.0 ** -11 / np.sqrt(3))
    dev.reset()
    dev.prefill(0, ids)
    last = rel(dev.logits(0), want[-1])
    assert last < (1e-5 if n < 16 else 2 * np.sqrt(8 * hp.transformers) * 2.0 ** -11 / np.sqrt(3))  # (a single row: up to twice the rms)
    dev.close()


@pytest.mark.parametrize("vocab", [999, 1024, 8192, 8193, 20480, 20481, 32768, 32770])
def test_probabilities_of_rows_of_every_length(pkg, vocab):
    """Probabilities and loss against float64 from the same call's logits.  Bound: a logit's difference and its exponential are right to 2^-23 (1 + |x|) and
    2^-22, a sum of positive terms to 2^-24 times the longest chain of additions (33 in a thread, 22 across them)."""
    hp = hybrid(pkg, dim=64, attnHeads=1, ffnDim=96, transformers=2, vocabSize=vocab, gdnHeads=1, maxL=80, maxSeqs=1)
    dev = pkg.Device(hp, 0)
    dev.upload(pkg.Model.generate(hp, 5).randomize_gains(5))
    ids = pkg.random_tokens(7, 0, vocab, 70)
    logits, probs, nll = dev.forward_full(0, ids)
    x = logits.astype(np.float64)
    x -= x.max(axis=1, keepdims=True)
    want = np.exp(x) / np.exp(x).sum(axis=1, keepdims=True)
    bound = 2.0 ** -23 * (1 + np.abs(x)) + 2.0 ** -21 + 60 * 2.0 ** -24
    assert np.all(np.abs(probs - want) <= bound * want + 1e-37)
    loss = -np.log(np.maximum(want[np.arange(69), ids[1:]], 1e-4)).mean()
    assert abs(nll - loss) <= 1e-5 * loss
    dev.close()


@pytest.mark.parametrize("head", [64, 128])
def test_attention_by_eight_and_by_four_waves(pkg, head):
    """Up to one workgroup a compute unit eight waves share the keys of 16 queries, beyond it four: either side of the line and lengths of less than a tile
    per wave, against prefill mode 1."""
    heads = 512 // head
    n = 16 * 256 // heads + 1  # at 256 units: the first length beyond it
    hp = pkg.config(2, dim=512, attnHeads=heads, headDim=head, ffnDim=128, transformers=2, vocabSize=300, maxL=n + 8, maxSeqs=1)
    dev = pkg.Device(hp, 0)
    dev.upload(pkg.Model.generate(hp, 5).randomize_gains(5))
    ids = pkg.random_tokens(9, 0, 300, n)
    dev.set_prefill_mode(1)
    want = dev.forward_full(0, ids)[0]
    dev.set_prefill_mode(0)
    for m in (2, 17, 66, 130, n - 1, n):
        dev.reset()
        assert rel(dev.forward_full(0, ids[:m])[0], want[:m]) < 2e-5
    dev.close()
