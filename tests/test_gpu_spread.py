"""fp32 prefills of models whose weights, gains or tables spread over many octaves: halves do not reach that far (csrc/h2.h), and such models multiply planes; models
just inside the rule stay with pairs.  Against the float64 oracle.

Bound: beside what the same context is off token by token (fp32 products), the accumulator of a product of planes rounds 6 K / 32 times, 2^-24 of a partial sum at most and
evenly spread, which is 2^-24 sqrt(K / 16) of the product's norm (rms); four products a layer and the LM head add up in squares; twice that."""
import numpy as np
import pytest

from test_gpu_ranks import config

pytestmark = pytest.mark.gpu
TOKENS = 130


def bound(hp):
    return 2 * 2.0 ** -24 * np.sqrt(hp.dim / 16) * np.sqrt(4 * hp.transformers + 1)


def build(pkg, orc, change, heads=4, layers=4):
    hp = config(pkg, heads=heads, hd=64, ffn=512, layers=layers, vocab=700, ple=64, maxSeqs=2, maxL=200)
    model = pkg.Model.generate(hp, 11).randomize_gains(11)
    change(pkg, model, hp)
    return hp, model, orc.Weights.from_model(model)


def plain(pkg, model, hp):
    pass


def unit_off(pkg, model, hp):
    """A unit whose gate and up rows are 2^33 above the others', and whose gate is far below zero for every token: the unit is 0, its bound is not."""
    model.tensor(0, pkg.T_TOKEN_EMBEDDINGS)[:, 0] = 1.0
    for layer in range(hp.transformers):
        for tid, size in ((pkg.T_FFN_1A, -2.0 ** 14), (pkg.T_FFN_1B, 2.0 ** 16)):
            row = model.tensor(layer, tid)[7]
            row[:] = 0
            row[0] = size


def gains(octaves):
    def change(pkg, model, hp):
        """Gains over 2 x `octaves` octaves, their inverses in the columns that they meet."""
        rng = np.random.default_rng(3)
        for layer in range(hp.transformers):
            for gain, tids in ((pkg.T_RMS_GAMMA, (pkg.T_QUERY, pkg.T_KEY, pkg.T_VALUE, pkg.T_GATED_QUERY, pkg.T_PLE_GATE, pkg.T_GDN_ALPHA_W, pkg.T_GDN_BETA_W)),
                               (pkg.T_RMS_GAMMA2, (pkg.T_FFN_1A, pkg.T_FFN_1B))):
                by = np.exp2(rng.integers(-octaves, octaves + 1, size=hp.dim)).astype(np.float32)
                model.tensor(layer, gain)[:] *= by.reshape(model.tensor(layer, gain).shape)
                for tid in tids:
                    t = model.tensor(layer, tid)
                    if t is not None:
                        t /= by[None, :]
    return change


def column(pkg, model, hp):
    """A residual column 2^9 above the others, from the embeddings on, that no product but the residual's own reads."""
    model.tensor(0, pkg.T_TOKEN_EMBEDDINGS)[:, 3] = 20.0
    model.tensor(0, pkg.T_FINAL_RMS_GAMMA).reshape(-1)[3] = 0
    for layer in range(hp.transformers):
        for tid in (pkg.T_QUERY, pkg.T_KEY, pkg.T_VALUE, pkg.T_PLE_GATE, pkg.T_GDN_ALPHA_W, pkg.T_GDN_BETA_W, pkg.T_FFN_1A, pkg.T_FFN_1B):
            if model.tensor(layer, tid) is not None:
                model.tensor(layer, tid)[:, 3] = 0


def table(pkg, model, hp):
    """Per-layer embeddings 2^20 above the values beside them, brought back by the projection's columns."""
    for layer in range(hp.transformers):
        model.tensor(layer, pkg.T_PLE_TABLE)[:] *= 2.0 ** 24
        model.tensor(layer, pkg.T_PLE_UP)[:] *= 2.0 ** -24


CASES = {"plain": (plain, "PREFILL_PAIRS"), "gains inside": (gains(4), "PREFILL_PAIRS"), "unit off": (unit_off, "PREFILL_PLANES"), "gains": (gains(16), "PREFILL_PLANES"),
         "column": (column, "PREFILL_PLANES"), "table": (table, "PREFILL_PLANES")}


@pytest.mark.parametrize("case,heads,layers", [(c, 4, 4) for c in CASES] + [("gains", 18, 2), ("gains", 34, 2), ("plain", 34, 2)])  # rows of up to 1024, 2048 and more
def test_distance_from_float64(pkg, orc, case, heads, layers):
    change, route = CASES[case]
    hp, model, w = build(pkg, orc, change, heads, layers)
    ids = pkg.random_tokens(5, 0, hp.vocabSize, TOKENS)
    dec = orc.Decoder(w, "f64")
    want = np.array([dec.step(int(t))[1] for t in ids])
    dec.close()
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    assert dev.prefill_route(TOKENS) == getattr(pkg, route) and dev.prefill_route(64) == pkg.PREFILL_ROWS and dev.prefill_route(1) == pkg.PREFILL_BY_TOKEN
    err = {}
    for mode in (0, 1):
        dev.set_prefill_mode(mode)
        dev.reset()
        got = dev.forward_full(0, ids, want_probs=False)[0]
        err[mode] = float(np.linalg.norm(got - want) / np.linalg.norm(want))
    print(f"{case}: prefill {err[0]:.2e}, token by token {err[1]:.2e}")
    assert err[0] <= err[1] + bound(hp)
    # prompts of two sequences in one call, and a second call behind cached rows
    dev.set_prefill_mode(0)
    dev.reset()
    dev.prefill_batch([0, 1], [ids[:40], ids[:50]])
    dev.prefill_batch([1, 0], [ids[50:], ids[40:]])
    for s in range(2):
        assert np.linalg.norm(dev.logits(s) - want[-1]) <= 2 * (err[1] + bound(hp)) * np.linalg.norm(want[-1])  # (one row: twice the rms of all)
    dev.close()


def test_a_finalize_changes_the_form(pkg, orc):
    """Work buffers of one form are not used by the other."""
    hp, even, w = build(pkg, orc, plain)
    _, spread, ws = build(pkg, orc, gains(16))
    ids = pkg.random_tokens(5, 0, hp.vocabSize, TOKENS)
    dev = pkg.Device(hp, 0)
    for model, weights, route in ((even, w, pkg.PREFILL_PAIRS), (spread, ws, pkg.PREFILL_PLANES), (even, w, pkg.PREFILL_PAIRS)):
        dev.upload(model)
        assert dev.prefill_route(TOKENS) == route
        dec = orc.Decoder(weights, "f64")
        for t in ids:
            _, want = dec.step(int(t))
        dec.close()
        dev.reset()
        dev.prefill(0, ids)
        assert np.linalg.norm(dev.logits(0) - want) <= 4 * bound(hp) * np.linalg.norm(want)
    dev.close()
