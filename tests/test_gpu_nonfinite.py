"""Infinite, NaN and the largest finite values in weights, gains and operands: every path gives what fp32 arithmetic gives (the
float64 oracle, or float64 NumPy for the bare products), not the NaN of a product of planes."""
import numpy as np
import pytest

from test_gpu_gemm_tiles import F16, P3, selftest

pytestmark = pytest.mark.gpu
INF = np.inf
TOP = np.float32(3.4e38)  # the bf16 nearest to it is infinite ...
EDGE = np.uint32(0x7f7f8000).view(np.float32)  # ... from here on
ODD = [77, 78, 79]        # vocabulary rows that the cases below change; never fed


def config(pkg, kind, bf16):
    if kind == "attn":  # what the XCD-rank kernel takes
        return pkg.config(2, dim=256, attnHeads=4, headDim=64, ffnDim=704, transformers=2, vocabSize=1000, maxL=160, maxSeqs=5, weightDtype=bf16)
    if kind == "flags":
        return pkg.config(2, dim=256, attnHeads=4, headDim=64, ffnDim=704, transformers=2, vocabSize=1000, maxL=160, maxSeqs=5, weightDtype=bf16,
                          qkRmsNorm=1, queryGating=1)
    hp = pkg.config(3, dim=256, attnHeads=4, headDim=64, ffnDim=704, transformers=4, vocabSize=1000, gdnHeads=6 if kind == "heads6" else 4, pleDim=64,
                    maxL=160, maxSeqs=5, weightDtype=bf16)
    pkg.set_layer_pattern(hp, 1)
    return hp


def model(pkg, hp, case):
    m = pkg.Model.generate(hp, 5).randomize_gains(5)
    E, gF = m.tensor(0, pkg.T_TOKEN_EMBEDDINGS), m.tensor(0, pkg.T_FINAL_RMS_GAMMA)
    if case == "head":  # logits of +-inf, and one of about 1e37
        gF *= np.float32(0.1)
        E[77, 3], E[78, 5], E[79, 7] = INF, -INF, TOP
    elif case == "nan":
        E[77, 3] = np.nan
    elif case == "edge":  # the largest weight that the planes hold
        gF *= np.float32(0.1)
        E[79, 7] = np.nextafter(EDGE, np.float32(0))
    elif case == "gain":  # infinite activations in front of finite weights
        gF[3] = INF
    elif case == "large gain":
        gF[3], gF[4] = 2.0 ** 59.9, 2.0 ** 60
    elif case == "gate":  # decays of 0 and 1, a write strength of 0 or 1
        for layer in range(hp.transformers):
            wa, wb = m.tensor(layer, pkg.T_GDN_ALPHA_W), m.tensor(layer, pkg.T_GDN_BETA_W)
            if wa is not None:
                wa[0, 3], wa[1, 3], wb[2, 3], wb[3, 3] = INF, -INF, INF, 3e38
    elif case == "embedding":  # of a token that the prompts hold
        for layer in range(hp.transformers):
            m.tensor(layer, pkg.T_PLE_TABLE)[7, 5] = INF
    elif case == "bias":  # decays of 0 and 1, write strengths of 1 and 0
        for layer in range(hp.transformers):
            ba, bb = m.tensor(layer, pkg.T_GDN_ALPHA_B), m.tensor(layer, pkg.T_GDN_BETA_B)
            if ba is not None:
                ba[0], ba[1], bb[2], bb[3] = INF, -INF, INF, -INF
    elif case == "large bias":  # sums of 64 logarithms of such a decay would overflow
        for layer in range(hp.transformers):
            ba = m.tensor(layer, pkg.T_GDN_ALPHA_B)
            if ba is not None:
                ba[-1] = 3e38
    elif case == "query gain":
        for layer in range(hp.transformers):
            m.tensor(layer, pkg.T_QUERY_RMS_GAMMA)[9] = 2.0 ** 62
    return m


def same(got, want, tol):
    got, want = np.asarray(got, np.float64), np.asarray(want, np.float64)
    with np.errstate(over="ignore"):
        want = want.astype(np.float32).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.where(np.isinf(got), np.sign(got), 0), np.where(np.isinf(want), np.sign(want), 0))
    odd = np.zeros(got.shape, bool)
    odd[..., ODD] = True
    fine = np.isfinite(want)
    a, b = got[fine & ~odd], want[fine & ~odd]
    assert b.size == 0 or np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
    a, b = got[fine & odd], want[fine & odd]  # (single values: the input's error over one of its elements)
    assert np.all(np.abs(a - b) <= 100 * tol * np.abs(b) + tol)


@pytest.mark.parametrize("kind,case,bf16", [(kind, case, bf16) for bf16 in (0, 1) for kind, case in (
    ("attn", "head"), ("attn", "gain"), ("hybrid", "head"), ("hybrid", "nan"), ("hybrid", "gain"), ("hybrid", "large gain"), ("hybrid", "gate"))]
    + [("hybrid", "edge", 0)])
def test_paths_against_oracle(pkg, orc, kind, case, bf16):
    hp = config(pkg, kind, bf16)
    m = model(pkg, hp, case)
    dev = pkg.Device(hp, 0)
    dev.upload(m)
    w = orc.Weights.from_model(m, bf16=bool(bf16))
    ids = np.random.default_rng(3).integers(0, 70, 120).astype(np.int32)

    def oracle(tokens):
        dec = orc.Decoder(w, "f64")
        out = np.stack([dec.step(int(t))[1] for t in tokens])
        dec.close()
        return out

    want = oracle(ids)
    for n in (20, 100):  # where the row kernels, the tiles would be
        dev.reset()
        same(dev.forward_full(0, ids[:n], want_probs=False)[0], want[:n], 1e-5)
        dev.reset()
        dev.prefill_batch(list(range(5)), [ids[:n]] * 5)
        for s in range(5):
            same(dev.logits(s), want[n - 1], 1e-5)
        for i in range(n, n + 3):
            dev.decode_step([ids[i]] * 5)
            for s in (0, 4):
                same(dev.logits(s), want[i], 1e-5)
    for mode in (3, 1, 0):
        dev.set_persistent(mode)
        dev.reset()
        dev.prefill(0, ids[:9])
        same(dev.logits(0), want[8], 1e-5)
        for i in range(9, 12):
            pick = dev.decode_step([ids[i]])[0]
            lg = dev.logits(0)
            same(lg, want[i], 1e-5)
            if not np.isnan(want[i]).any() and np.sum(want[i] == want[i].max()) == 1:
                assert pick == want[i].argmax()
    dev.close()


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("kind,case", [("hybrid", "embedding"), ("hybrid", "bias"), ("heads6", "large bias"), ("flags", "query gain")])
def test_tables_gains_and_biases_against_oracle(pkg, orc, kind, case, bf16):
    """As above, of the parameters that are no operands of a product themselves (heads6: the last bias lies behind the whole 16-byte pieces)."""
    test_paths_against_oracle(pkg, orc, kind, case, bf16)


def test_finalize_with_and_without_operands(pkg):
    """A captured step of the row kernels, then weights that they are not given, and back."""
    hp = config(pkg, "hybrid", 0)
    plain, odd = model(pkg, hp, ""), model(pkg, hp, "gate")

    def decode(dev):
        dev.reset()
        dev.prefill_batch([0, 1], [np.arange(30, dtype=np.int32), np.arange(40, 60, dtype=np.int32)])
        out = [dev.decode_loop([1, 2], 5)]
        dev.synchronize()
        out.append(dev.decode_loop(out[-1][-1], 5))
        return np.concatenate(out), np.stack([dev.logits(s) for s in (0, 1)])

    def device(m):
        dev = pkg.Device(hp, 0)
        dev.set_graph(2)
        dev.upload(m)
        return dev

    want = []
    for m in (plain, odd):
        dev = device(m)
        want.append(decode(dev))
        dev.close()
    dev = device(plain)
    for m, w in ((plain, want[0]), (odd, want[1]), (plain, want[0])):
        dev.upload(m)
        for got, ref in zip(decode(dev), w):
            assert np.array_equal(got, ref)
    dev.close()


@pytest.mark.parametrize("m,n,k", [(3, 5, 32), (70, 66, 96), (130, 257, 1024)])
def test_planes(pkg, m, n, k):
    """Both operands with infinities of either sign, NaN, zeros against them and the largest finite values."""
    rng = np.random.default_rng(m)
    fmax = np.finfo(np.float32).max
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((n, k)).astype(np.float32)
    a[0, 1], a[1, 2], a[2, 3] = INF, -INF, np.nan
    b[0, 1], b[1, 2], b[2, 1], b[3, 4] = 0, INF, -INF, INF  # inf * 0; -inf * inf, inf * -inf; an infinity against finite values
    with np.errstate(invalid="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64).T
    got = selftest(pkg, P3, a, b).astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want[0, 0]) and want[1, 1] == -INF and want[0, 2] == -INF
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf]) and inf.sum() > 3 and np.all(np.isfinite(got[~inf & ~np.isnan(want)]))
    # one huge element per row against one of b's: what it adds up to fits, plane by plane too
    a = np.zeros((m, k), np.float32)
    b = np.zeros((n, k), np.float32)
    huge = np.array([fmax, -fmax, EDGE, -EDGE, TOP, np.nextafter(EDGE, np.float32(0)), fmax / 2], np.float32)
    a[:, 5] = huge[np.arange(m) % huge.size]
    b[:, 5] = np.array([1, -0.5, 2.0 ** -100, 0.7, 3e-39], np.float32)[np.arange(n) % 5]
    want = a.astype(np.float64) @ b.astype(np.float64).T
    got = selftest(pkg, P3, a, b)
    assert np.all(np.isfinite(got))
    ok = b[:, 5] != np.float32(3e-39)  # (a denormal factor: planes below the bf16 denormals are lost)
    assert np.max(np.abs(got - want)[:, ok] / np.abs(want)[:, ok]) <= 2.0 ** -22


@pytest.mark.parametrize("m,n,k", [(40, 320, 256), (300, 512, 256), (1100, 17000, 192)])  # the three kernels of halves
def test_swiglu_to_halves(pkg, m, n, k):
    """silu(gate) * up on its way into halves: NaN and infinities stay, finite values beyond the halves saturate, and a gate of minus a
    lot gives 0 whatever the other factor is."""
    rng = np.random.default_rng(n)
    a = rng.standard_normal((m, k)).astype(np.float16).astype(np.float32)
    b = (rng.standard_normal((n, k)) / np.sqrt(k)).astype(np.float16).astype(np.float32)
    a[1, 2], a[2, 3], a[3, 4] = np.nan, INF, -INF
    a[4], a[5], a[6] = 0, 0, 0
    a[4, 5], a[5, 6], a[6, 7] = 60000, 300, -60000
    b[0:8, 2:8] = np.array([1, 2, -1, 3, 0.5, -2, -4, -3], np.float32)[:, None]  # gate, up of units 0 .. 3
    b[8:, 2:8] = np.where(b[8:, 2:8] == 0, 1, b[8:, 2:8])  # (no 0 against an infinity)
    got = selftest(pkg, F16, a, b, swiglu=True).astype(np.float64)
    with np.errstate(all="ignore"):
        p = a.astype(np.float64) @ b.astype(np.float64).T
        want = p[:, 0::2] / (1 + np.exp(-p[:, 0::2])) * p[:, 1::2]
    assert np.isnan(want[1]).all() and np.isinf(want[2, 0]) and np.isnan(want[3, 0]) and want[4, 0] > 65504 and want[6, 1] == -1.08e10
    want = np.where(np.isfinite(want), np.clip(want, -65504, 65504), want)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    inf = np.isinf(want)
    assert np.array_equal(got[inf], want[inf])
    ok = np.isfinite(want)
    # one rounding to halves, and the factors' fp32 sums (values up to 65504 come from factors of up to 3e5)
    assert np.all(np.abs(got - want)[ok] <= 2.0 ** -11 * np.abs(want)[ok] + 2e-6 * np.sqrt(k))


@pytest.mark.parametrize("kind", ["attn", "hybrid"])
@pytest.mark.parametrize("n", [40, 90])  # tiled products; also segments in chunks
def test_an_overflow_in_a_long_prompt_of_halves(pkg, kind, n):
    """Finite weights and one token whose residual row overflows in the layer applied first: the next layer makes NaN of its key, value and
    state update, and so are the logits of the tokens behind it, as they are token by token."""
    hp = config(pkg, kind, 1)
    m = model(pkg, hp, "")
    top = hp.transformers - 1
    E, g2 = m.tensor(0, pkg.T_TOKEN_EMBEDDINGS), m.tensor(top, pkg.T_RMS_GAMMA2)
    E[:, 9], E[69, 9], g2[9] = -0.5, 0.5, 1.0
    gate, up = m.tensor(top, pkg.T_FFN_1A), m.tensor(top, pkg.T_FFN_1B)
    gate[0], up[0] = 0, 0
    gate[0, 9] = up[0, 9] = 1000  # unit 0: silu(1000 x) 1000 x of the ninth normed column, x about 13 for token 69 and -13 for the others
    m.tensor(top, pkg.T_FFN_2)[11, 0] = 3e38
    dev = pkg.Device(hp, 0)
    dev.upload(m)
    assert dev.operand_bytes() > 0
    ids = np.random.default_rng(3).integers(0, 60, n).astype(np.int32)
    for odd in (False, True):
        ids[3] = 69 if odd else 7
        seen = {}
        for mode in (0, 1):
            dev.set_prefill_mode(mode)
            dev.reset()
            dev.prefill(0, ids)
            seen[mode] = np.isnan(dev.logits(0))
        assert np.all(seen[1] == odd) and np.all(seen[0] == odd)
    dev.close()
