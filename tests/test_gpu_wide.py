"""Decode of 6 to 64 sequences in one launch (kernels_wide.hip) against the CPU oracle: the smallest and largest batches of every number of
token blocks, heads of which a second one has 1, 2, 4 or no sharers, flags, layer mixes, per-layer embeddings, ragged lengths on shuffled pages,
vocabularies that end inside a tile, and the way out.

Bounds: as in the other decode tests (1e-3 relative, ids by a gap of 2e-5)."""
import numpy as np
import pytest

from conftest import assert_logits_close, check_greedy_against_oracle
from test_gpu_ranks import config, start

pytestmark = pytest.mark.gpu

RTOL = 1e-3
GAP_TOL = 2e-5

CASES = {
    # name: (hyper-parameters, sequences, prompt lengths from .. to, steps)
    "hybrid6": (dict(heads=12, hd=64, ffn=1024, layers=4, vocab=300, ple=64), 6, 2, 50, 4),
    "attn_flags7": (dict(heads=8, hd=64, ffn=768, layers=2, vocab=520, ple=0, gdn=False, flags=True), 7, 5, 120, 3),
    "attn_flags9": (dict(heads=8, hd=64, ffn=768, layers=2, vocab=520, ple=0, gdn=False, flags=True), 9, 5, 120, 3),
    "hybrid16": (dict(heads=10, hd=64, ffn=256, layers=2, vocab=4999, ple=32), 16, 2, 40, 3),
    "hybrid17": (dict(heads=12, hd=64, ffn=2048, layers=4, vocab=1003, ple=64), 17, 1, 90, 4),
    "hybrid32": (dict(heads=8, hd=64, ffn=256, layers=4, vocab=4111, ple=128), 32, 2, 60, 3),
    "hybrid33": (dict(heads=10, hd=64, ffn=512, layers=2, vocab=700, ple=32), 33, 2, 40, 3),
    "hybrid48": (dict(heads=12, hd=64, ffn=768, layers=2, vocab=520, ple=0), 48, 2, 30, 2),
    "hybrid64": (dict(heads=12, hd=64, ffn=512, layers=2, vocab=1000, ple=64), 64, 1, 70, 3),
    "gated12_17": (dict(heads=12, hd=64, ffn=512, layers=2, vocab=600, ple=0, gdn=False, flags=True), 17, 3, 90, 3),  # 32 tiles of the first phase: all there are
    "gated12_64": (dict(heads=12, hd=64, ffn=512, layers=2, vocab=600, ple=0, gdn=False, flags=True), 64, 1, 70, 2),
    "gated10_50": (dict(heads=10, hd=64, ffn=1280, layers=2, vocab=600, ple=0, gdn=False, flags=True), 50, 1, 70, 2),
    "attn_flags49": (dict(heads=8, hd=64, ffn=768, layers=2, vocab=520, ple=32, gdn=False, flags=True), 49, 3, 200, 2),
}


@pytest.mark.parametrize("case", list(CASES))
def test_batches_against_the_oracle(pkg, orc, case):
    shape, n, lo, hi, steps = CASES[case]
    hp = config(pkg, maxSeqs=n, maxL=256, **shape)
    dev, w, prompts = start(pkg, orc, hp, n, lo, hi, 60 + n)
    assert dev.decode_route(n) == (pkg.DECODE_RANKS if case == "attn_flags7" else pkg.DECODE_WIDE)  # (8 heads of attention only: from 9 on)
    first = [dev.greedy_token(s) for s in range(n)]
    a = dev.decode_loop(first, steps)                # a run of steps in one launch
    b = dev.decode_loop([int(t) for t in a[-1]], 1)  # and a step of its own: cache, states, positions carried over
    assert dev.persistent_fallbacks() == 0
    got = np.concatenate([np.array([first]), a, b])
    for s in sorted(s for s in {0, 1, 15, 16, n // 4, n // 2 - 1, n // 2, n - 2, n - 1} if s < n):
        dec = orc.Decoder(w, "f64")
        check_greedy_against_oracle(dec, prompts[s], got[:, s].tolist(), GAP_TOL, what=f"{case} sequence {s}")
        dec.reset()
        for t in list(prompts[s]) + got[:-1, s].tolist():
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"{case} sequence {s}")
        assert dev.seq_len(s) == len(prompts[s]) + steps + 1
        dec.close()
    dev.close()


@pytest.mark.parametrize("n", [6, 17, 40, 64])
def test_every_sequence_against_the_row_kernels(pkg, orc, n):
    """All logits over the same tokens in both, two orders of fp32 sums apart, and no further from the float64 oracle than theirs (a factor
    of two of rounding noise)."""
    hp = config(pkg, heads=12, hd=64, ffn=1024, layers=8, vocab=1024, ple=64, maxSeqs=64, maxL=256)
    out, feed = {}, np.random.default_rng(4).integers(0, hp.vocabSize, size=(5, n))
    for mode in (3, 0):
        dev, w, prompts = start(pkg, orc, hp, n, 3, 60, 71)
        dev.set_persistent(mode)
        assert dev.decode_route(n) == (pkg.DECODE_WIDE if mode == 3 else pkg.DECODE_ROWS)
        for row in feed:
            dev.decode_step([int(t) for t in row])
        assert dev.persistent_fallbacks() == 0
        out[mode] = np.stack([dev.logits(s) for s in range(n)])
        dev.close()
    for s in range(n):
        assert_logits_close(out[3][s], out[0][s], 1e-4, f"sequence {s}")
    err = {3: [], 0: []}
    for s in range(0, n, 5):
        dec = orc.Decoder(w, "f64")
        for t in list(prompts[s]) + feed[:, s].tolist():
            _, lg = dec.step(int(t))
        dec.close()
        for mode in err:
            err[mode].append(np.linalg.norm(out[mode][s] - lg) / np.linalg.norm(lg))
    rms = {mode: float(np.sqrt(np.mean(np.square(e)))) for mode, e in err.items()}
    print(f"distance from float64: one launch {rms[3]:.2e}, row kernels {rms[0]:.2e}")
    assert rms[3] <= 2 * rms[0]


@pytest.mark.parametrize("where", ["meeting", "mid-run"])
def test_gives_up_and_falls_back(pkg, orc, where):
    """A launch that gives up (places taken from the host; a workgroup that leaves at step 2) is redone as row kernels from the states
    before it, also where an earlier launch has left those in their second place; the kernel comes back once it is asked for."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64, maxSeqs=20, maxL=128)
    ids, logits = {}, {}
    for inject in (False, True):
        dev, w, prompts = start(pkg, orc, hp, 20, 3, 30, 83)
        nxt = [dev.greedy_token(s) for s in range(20)]
        out = []
        for k in range(3):
            if inject and k == 1:
                dev.debug_inject_abort(1) if where == "meeting" else dev.debug_inject_abort_at_step(2)
            if inject and k == 2:
                assert dev.get_persistent() == 0 and dev.persistent_fallbacks() == 1
                assert dev.decode_route(20) == pkg.DECODE_ROWS
                dev.set_persistent(3)
            assert dev.decode_route(20) == pkg.DECODE_WIDE
            out.append(dev.decode_loop(nxt, 4))
            nxt = [int(t) for t in out[-1][-1]]
        assert dev.persistent_fallbacks() == int(inject)
        ids[inject] = np.concatenate(out)
        logits[inject] = np.stack([dev.logits(s) for s in range(20)])
        dev.close()
    assert (ids[True] == ids[False]).mean() > 0.99  # (two orders of fp32 sums: a tie may part)
    for s in range(20):
        if (ids[True][:, s] == ids[False][:, s]).all():
            assert_logits_close(logits[True][s], logits[False][s], 1e-4, f"sequence {s}")


def test_batches_of_changing_size_share_the_exchange_memory(pkg, orc):
    """Calls of 40, 17, 64, 5, 9, 33 and 64 sequences in turn on one context, with a tag count that wraps on the way: every size lays the data
    out over what the others left, and the kernel of few sequences works on the same states."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64, maxSeqs=64, maxL=128)
    dev, w, prompts = start(pkg, orc, hp, 64, 2, 40, 91)
    hist = [list(p) for p in prompts]
    nxt = [dev.greedy_token(s) for s in range(64)]
    for n in (40, 17, 64, 5, 9, 33, 64):
        if n == 5:
            dev.debug_set_xcd_tag(0xFFFFFFF0)
        assert dev.decode_route(n) == (pkg.DECODE_RANKS if n == 5 else pkg.DECODE_WIDE)
        out = dev.decode_loop(nxt[:n], 2)
        for s in range(n):
            hist[s] += [nxt[s], int(out[0, s])]
            nxt[s] = int(out[1, s])
    assert dev.persistent_fallbacks() == 0
    for s in (0, 4, 5, 8, 9, 16, 17, 32, 39, 40, 63):
        dec = orc.Decoder(w, "f64")
        for t in hist[s]:
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"sequence {s}")
        assert dev.seq_len(s) == len(hist[s])
        dec.close()
    dev.close()


@pytest.mark.parametrize("heads,ffn", [(8, 2048), (8, 1280), (10, 2048), (10, 1280)])
def test_widths_whose_waves_have_fewer_chunks(pkg, orc, heads, ffn):
    """Widths 512 and 640, where waves have two chunks of a product and not three, over borders of token blocks in both directions: what a launch of another
    size has left in the exchange memory (fp32 sums where this one has planes) is multiplied nowhere."""
    hp = config(pkg, heads=heads, hd=64, ffn=ffn, layers=2, vocab=600, ple=64, maxSeqs=64, maxL=96)
    dev, w, prompts = start(pkg, orc, hp, 64, 2, 24, 97)
    hist = [list(p) for p in prompts]
    nxt = [dev.greedy_token(s) for s in range(64)]
    for n in (20, 10, 40, 10, 64, 20, 48, 9, 33):
        assert dev.decode_route(n) == pkg.DECODE_WIDE
        out = dev.decode_loop(nxt[:n], 2)
        for s in range(n):
            hist[s] += [nxt[s], int(out[0, s])]
            nxt[s] = int(out[1, s])
            assert np.isfinite(dev.logits(s)).all(), f"{n} sequences, sequence {s}"
    assert dev.persistent_fallbacks() == 0
    for s in range(0, 64, 3):
        dec = orc.Decoder(w, "f64")
        for t in hist[s]:
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"sequence {s}")
        dec.close()
    dev.close()


def test_more_than_64_pages(pkg):
    """A wave holds the first 64 page numbers of its sequence in registers and looks the others up: keys beyond 4096 positions, against the row kernels over the
    same tokens (1e-4: two orders of fp32 sums)."""
    n, hp = 9, config(pkg, heads=8, hd=64, ffn=256, layers=2, vocab=300, ple=0, gdn=False, maxL=4400, maxSeqs=9)
    lens, out = (4200, 33, 4094, 70, 4160, 5, 900, 4095, 64), {}
    for mode in (3, 0):
        dev = pkg.Device(hp, 0)
        dev.upload(pkg.Model.generate(hp, 7).randomize_gains(7))
        dev.set_page_table(np.random.default_rng(7).permutation(n * 69).astype(np.int32))
        dev.prefill_batch(list(range(n)), [pkg.random_tokens(7, s, hp.vocabSize, m) for s, m in enumerate(lens)])
        dev.set_persistent(mode)
        assert dev.decode_route(n) == (pkg.DECODE_WIDE if mode == 3 else pkg.DECODE_ROWS)
        lg = []
        for row in np.random.default_rng(8).integers(0, hp.vocabSize, size=(4, n)):  # sequences 2 and 7 reach their 65th page on the way
            dev.decode_step([int(t) for t in row])
            lg.append([dev.logits(s) for s in range(n)])
        assert dev.persistent_fallbacks() == 0
        out[mode] = np.array(lg)
        dev.close()
    for i in range(4):
        for s in range(n):
            assert_logits_close(out[3][i, s], out[0][i, s], 1e-4, f"step {i} sequence {s}")


def test_states_near_the_end_of_their_offsets(pkg):
    """65 500 sequences of 8 heads: a second place of the states for 64 of them would lie beyond 32-bit offsets, one for 16 does not, so calls of up to 16 stay in
    one launch (both kernels) and more rows run as row kernels; the first and last sequences of a call, and what follows on it, as without."""
    hp = config(pkg, heads=8, hd=64, ffn=256, layers=1, vocab=300, ple=0, maxSeqs=65500, maxL=40)
    hp.layerKinds[0] = pkg.KIND_GDN
    out, feed = {}, np.random.default_rng(4).integers(0, 300, size=(3, 17))
    for mode in (3, 0):
        dev = pkg.Device(hp, 0)
        dev.upload(pkg.Model.generate(hp, 7).randomize_gains(7))
        dev.set_persistent(mode)
        want = [pkg.DECODE_RANKS, pkg.DECODE_WIDE, pkg.DECODE_WIDE, pkg.DECODE_ROWS]
        assert [dev.decode_route(n) for n in (5, 6, 16, 17)] == (want if mode == 3 else [pkg.DECODE_ROWS] * 4)
        dev.prefill_batch(list(range(17)), [pkg.random_tokens(7, s, 300, 5 + s % 3) for s in range(17)])
        for n in (16, 17, 5):
            for row in feed:
                dev.decode_step([int(t) for t in row[:n]])
        assert dev.persistent_fallbacks() == 0
        out[mode] = np.stack([dev.logits(s) for s in range(17)])
        dev.close()
    for s in range(17):
        assert_logits_close(out[3][s], out[0][s], 1e-4, f"sequence {s}")


def test_calls_that_the_kernel_does_not_take(pkg, orc):
    """What a caller sees of the route: one and few sequences, sampling, graph replays, prompts token by token, and a first phase of more tiles than workgroups
    (query gating beside per-layer embeddings in models of more than 8 heads)."""
    def context(**kw):
        hp = config(pkg, **{**dict(heads=12, hd=64, ffn=512, layers=2, vocab=300, ple=64, maxSeqs=70, maxL=64), **kw})
        dev = pkg.Device(hp, 0)
        dev.upload(pkg.Model.generate(hp, 3))
        return dev

    # from how many sequences on: pairs of a head and a sequence, and the share of attention layers
    for kw, first in ((dict(heads=8), 6), (dict(heads=10), 7), (dict(heads=12), 6), (dict(heads=8, gdn=False), 9), (dict(heads=10, gdn=False), 7), (dict(heads=12, gdn=False), 7)):
        dev = context(**kw)
        assert [dev.decode_route(n) for n in range(2, 17)] == [pkg.DECODE_RANKS] * (first - 2) + [pkg.DECODE_WIDE] * (17 - first), kw
        dev.close()
    dev = context()
    assert [dev.decode_route(n) for n in (0, 1, 2, 5, 16, 17, 64, 65, 70, 71)] == [
        -1, pkg.DECODE_XCD, pkg.DECODE_RANKS, pkg.DECODE_RANKS, pkg.DECODE_WIDE, pkg.DECODE_WIDE, pkg.DECODE_WIDE, pkg.DECODE_GEMV, pkg.DECODE_GEMV, -1]
    dev.set_sampling(0.8, 1)
    assert dev.decode_route(16) == pkg.DECODE_ROWS
    dev.set_sampling(0.0)
    dev.set_graph(4)
    assert dev.decode_route(16) == pkg.DECODE_ROWS
    dev.set_graph(0)
    dev.set_prefill_mode(1)
    assert dev.decode_route(16) == pkg.DECODE_GEMV
    dev.set_prefill_mode(0)
    assert dev.decode_route(16) == pkg.DECODE_WIDE
    dev.close()
    for kw, n16, n17 in ((dict(gdn=False, flags=True), pkg.DECODE_RANKS, pkg.DECODE_ROWS), (dict(half=True), pkg.DECODE_RANKS, pkg.DECODE_ROWS),
                         (dict(gdn=False, flags=True, ple=0), pkg.DECODE_WIDE, pkg.DECODE_WIDE), (dict(gdn=False, flags=True, heads=8), pkg.DECODE_WIDE, pkg.DECODE_WIDE)):
        dev = context(**kw)
        assert (dev.decode_route(16), dev.decode_route(17)) == (n16, n17), kw
        dev.close()
