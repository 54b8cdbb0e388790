"""Decode of several sequences in one launch (kernels_ranks.hip) against the CPU oracle: the smallest and largest batches it takes, head
sizes, weight types, flags, layer mixes, ragged lengths on shuffled pages, vocabularies that end inside a tile, and the way out.

Bounds: as in the other decode tests (1e-3 relative for fp32, ids by a gap of 2e-5).  bf16 weights run the same fp32-precision
arithmetic on the rounded weights, so they are held to the same bound here."""
import numpy as np
import pytest

from conftest import assert_logits_close, check_greedy_against_oracle

pytestmark = pytest.mark.gpu

RTOL = 1e-3
GAP_TOL = 2e-5

CASES = {
    # name: (hyper-parameters, sequences, prompt lengths from .. to, steps)
    "hybrid2": (dict(heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64), 2, 3, 40, 5),
    "ple32": (dict(heads=12, hd=64, ffn=512, layers=4, vocab=700, ple=32), 3, 2, 40, 4),  # the narrowest per-layer embeddings
    "hybrid9": (dict(heads=12, hd=64, ffn=2048, layers=4, vocab=1003, ple=64), 9, 1, 130, 4),
    "hybrid16": (dict(heads=8, hd=64, ffn=256, layers=4, vocab=4111, ple=128), 16, 2, 70, 4),
    "attn_flags5": (dict(heads=9, hd=64, ffn=768, layers=2, vocab=520, ple=0, gdn=False, flags=True, dim_ok=False), 5, 5, 90, 4),
    "gated_ple16": (dict(heads=12, hd=64, ffn=512, layers=2, vocab=600, ple=64, gdn=False, flags=True), 16, 5, 100, 4),  # fp32 rows that kernels_wide.hip refuses
    "attn_flags8": (dict(heads=8, hd=64, ffn=768, layers=2, vocab=520, ple=0, gdn=False, flags=True), 8, 5, 300, 4),
    "half_hd64": (dict(heads=16, hd=64, ffn=1024, layers=4, vocab=800, ple=64, half=True), 16, 2, 50, 4),
    "half_hd128_one": (dict(heads=8, hd=128, ffn=1536, layers=4, vocab=8200, ple=64, half=True), 1, 9, 9, 5),
    "half_hd128": (dict(heads=16, hd=128, ffn=5632, layers=4, vocab=600, ple=64, half=True), 8, 3, 60, 3),
    "half_hd128_flags": (dict(heads=8, hd=128, ffn=512, layers=2, vocab=600, ple=0, gdn=False, flags=True, half=True), 3, 20, 70, 3),
}


def config(pkg, heads, hd, ffn, layers, vocab, ple, gdn=True, flags=False, half=False, maxSeqs=16, maxL=400, dim_ok=True):
    kw = dict(dim=heads * hd, attnHeads=heads, headDim=hd, ffnDim=ffn, transformers=layers, vocabSize=vocab, pleDim=ple, maxSeqs=maxSeqs, maxL=maxL,
              qkRmsNorm=int(flags), queryGating=int(flags), weightDtype=pkg.DTYPE_BF16 if half else pkg.DTYPE_F32)
    if gdn:
        hp = pkg.config(3, gdnHeads=heads, gdnDk=hd, gdnDv=hd, **kw)
        pkg.set_layer_pattern(hp, 1)  # attention and delta-rule layers in turn
    else:
        hp = pkg.config(1, **kw)
    return hp


def start(pkg, orc, hp, n, lo, hi, seed):
    model = pkg.Model.generate(hp, seed).randomize_gains(seed)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    w = orc.Weights.from_model(model, bf16=hp.weightDtype == pkg.DTYPE_BF16)
    rng = np.random.default_rng(seed)
    dev.set_page_table(rng.permutation(hp.maxSeqs * ((hp.maxL + 63) // 64)).astype(np.int32))
    lens = [lo + (hi - lo) * ((7 * s + 3) % n) // max(1, n - 1) for s in range(n)]
    prompts = [pkg.random_tokens(seed, s, hp.vocabSize, m) for s, m in enumerate(lens)]
    for s, p in enumerate(prompts):  # short pieces: the fp32-precision path for bf16 models too
        for i in range(0, len(p), 12):
            dev.prefill(s, p[i:i + 12])
    return dev, w, prompts


@pytest.mark.parametrize("case", list(CASES))
def test_batches_against_the_oracle(pkg, orc, case):
    shape, n, lo, hi, steps = CASES[case]
    hp = config(pkg, **shape)
    dev, w, prompts = start(pkg, orc, hp, n, lo, hi, 60 + len(case))
    covered = dev.single_launch_sequences() >= n
    assert covered == shape.get("dim_ok", True)  # (dim 576: not a multiple of 128, the row kernels)
    assert dev.decode_route(n) == (pkg.DECODE_ROWS if not covered else pkg.DECODE_WIDE if case in ("hybrid9", "hybrid16") else pkg.DECODE_RANKS)
    first = [dev.greedy_token(s) for s in range(n)]
    a = dev.decode_loop(first, steps)           # a run of steps in one launch
    b = dev.decode_loop([int(t) for t in a[-1]], 1)  # and a step of its own: cache, states, positions carried over
    assert dev.persistent_fallbacks() == 0
    got = np.concatenate([np.array([first]), a, b])
    for s in range(n):
        dec = orc.Decoder(w, "f64")
        check_greedy_against_oracle(dec, prompts[s], got[:, s].tolist(), GAP_TOL, what=f"{case} sequence {s}")
        dec.reset()
        for t in list(prompts[s]) + got[:-1, s].tolist():
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"{case} sequence {s}")
        assert dev.seq_len(s) == len(prompts[s]) + steps + 1
        dec.close()
    dev.close()


@pytest.mark.parametrize("half", [False, True], ids=["fp32", "bf16"])
def test_distance_from_float64_is_that_of_the_row_kernels(pkg, orc, half):
    """The same arithmetic precision as the sequence of row kernels: over the same tokens the rms distance of the logits from the float64
    oracle may exceed theirs by the spread of two orders of summation (a factor of two of rounding noise), no more."""
    hp = config(pkg, heads=8 if half else 12, hd=128 if half else 64, ffn=1024, layers=8, vocab=1024, ple=64, half=half)
    err, n = {}, 6 if half else 5
    for mode in (3, 0):
        dev, w, prompts = start(pkg, orc, hp, n, 10, 60, 71)
        dev.set_persistent(mode)
        assert dev.decode_route(n) == (pkg.DECODE_RANKS if mode == 3 else pkg.DECODE_ROWS)
        feed = np.random.default_rng(4).integers(0, hp.vocabSize, size=(6, n))
        for row in feed:
            dev.decode_step([int(t) for t in row])
        e = []
        for s in range(n):
            dec = orc.Decoder(w, "f64")
            for t in list(prompts[s]) + feed[:, s].tolist():
                _, lg = dec.step(int(t))
            e.append(np.linalg.norm(dev.logits(s) - lg) / np.linalg.norm(lg))
            dec.close()
        err[mode] = float(np.sqrt(np.mean(np.square(e))))
        dev.close()
    print(f"distance from float64: one launch {err[3]:.2e}, row kernels {err[0]:.2e}")
    assert err[3] <= 2 * err[0]


def test_gives_up_at_its_meeting_and_falls_back(pkg, orc):
    """A launch whose workgroups do not all find a place (forced from the host: the places start taken) writes nothing; the call runs as the
    row kernels, the context stays in that mode, and the single launch works again once it is asked for."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64)
    ids = {}
    for inject in (0, 1):
        dev, w, prompts = start(pkg, orc, hp, 4, 6, 30, 83)
        first = [dev.greedy_token(s) for s in range(4)]
        out = [np.array([first])]
        for k in range(3):
            if inject and k == 1:
                dev.debug_inject_abort(1)
            if inject and k == 2:
                assert dev.get_persistent() == 0 and dev.persistent_fallbacks() == 1
                dev.set_persistent(3)
            out.append(dev.decode_loop([int(t) for t in out[-1][-1]], 3))
        assert dev.persistent_fallbacks() == inject and dev.get_persistent() == 3
        ids[inject] = np.concatenate(out)
        for s in range(4):
            dec = orc.Decoder(w, "f64")
            check_greedy_against_oracle(dec, prompts[s], ids[inject][:, s].tolist(), GAP_TOL, what=f"inject {inject} sequence {s}")
            dec.close()
        dev.close()


@pytest.mark.parametrize("case,n,steps,at", [("hybrid16", 16, 4, 1), ("hybrid2", 2, 2, 1), ("half_hd128_one", 1, 3, 2), ("half_hd128", 8, 3, 1),
                                             ("attn_flags8", 8, 5, 3)])
def test_gives_up_in_mid_run_and_falls_back(pkg, orc, case, n, steps, at):
    """A launch that is left in mid-run (forced from the host: workgroup 0 gives up when it reaches that step) has written states, K/V rows,
    picks and perhaps positions.  The call puts the sequences back and redoes its steps: bit for bit what a context does that runs them
    as row kernels from the start."""
    hp = config(pkg, **CASES[case][0])
    out = {}
    for inject in (0, 1):
        dev, _, prompts = start(pkg, orc, hp, n, 5, 80, 97)
        got = [dev.decode_loop([dev.greedy_token(s) for s in range(n)], 2)]
        assert dev.persistent_fallbacks() == 0
        if inject:
            dev.debug_inject_abort_at_step(at)
        else:
            dev.set_persistent(0)
        got.append(dev.decode_loop([int(t) for t in got[-1][-1]], steps))
        assert dev.persistent_fallbacks() == inject
        assert [dev.seq_len(s) for s in range(n)] == [len(p) + 2 + steps for p in prompts]
        dev.set_persistent(3)
        got.append(dev.decode_loop([int(t) for t in got[-1][-1]], 2))  # positions, states and rows carried over
        assert dev.persistent_fallbacks() == inject
        out[inject] = np.concatenate(got), np.stack([dev.logits(s) for s in range(n)])
        dev.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_giving_up_costs_the_one_sequence_kernel_nothing(pkg, orc):
    """Once the launch of several sequences has given up, calls that it would take run as row kernels; one sequence stays in its single
    launch (a second forced start shows it: only a single launch takes it)."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64)
    dev, w, prompts = start(pkg, orc, hp, 4, 6, 30, 83)
    assert dev.xcd_decode_supported()
    hist = [list(p) for p in prompts]
    nxt = [dev.greedy_token(s) for s in range(4)]
    for n, arm, mode, fallbacks in ((4, 1, 0, 1), (1, 0, 3, 1), (4, 1, 0, 1), (1, 0, 0, 2), (4, 0, 0, 2)):
        if arm:
            dev.debug_inject_abort(1)
        out = dev.decode_loop(nxt[:n], 2)
        assert (dev.get_persistent(), dev.persistent_fallbacks()) == (mode, fallbacks)
        for s in range(n):
            hist[s] += [nxt[s], int(out[0, s])]
            nxt[s] = int(out[1, s])
    for s in range(4):
        dec = orc.Decoder(w, "f64")
        for t in hist[s]:
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"sequence {s}")
        dec.close()
    dev.close()


def test_tags_are_cleared_before_they_wrap(pkg, orc):
    """The 32-bit tags of the exchange words are a running count of layer passes.  With the count set just below 2^32 a launch whose tags
    do not fit starts from cleared words and count 0; one whose tags just fit runs up to the last; both agree with the oracle."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64)
    dev, w, prompts = start(pkg, orc, hp, 3, 6, 40, 101)
    hist = [list(p) for p in prompts]
    nxt = [dev.greedy_token(s) for s in range(3)]
    top, passes = 0xFFFFFFFF, hp.transformers + 1  # a launch of n steps takes n * passes + 1 tags; below `top` they fit
    for n, tag in ((3, None), (4, top - 4 * passes - 1), (2, None), (5, top - 5 * passes - 2), (1, None), (3, top - 1), (2, None)):
        if tag is not None:
            dev.debug_set_xcd_tag(tag)
        out = dev.decode_loop(nxt, n)
        for s in range(3):
            hist[s] += [nxt[s]] + [int(t) for t in out[:-1, s]]
            nxt[s] = int(out[-1, s])
    assert dev.get_persistent() == 3 and dev.persistent_fallbacks() == 0
    for s in range(3):
        dec = orc.Decoder(w, "f64")
        check_greedy_against_oracle(dec, prompts[s], hist[s][len(prompts[s]):] + [nxt[s]], GAP_TOL, what=f"sequence {s}")
        dec.reset()
        for t in hist[s]:
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"sequence {s}")
        dec.close()
    dev.close()


def test_more_than_64_pages(pkg):
    """A wave holds the first 64 page numbers of its sequence in registers and looks the others up: keys beyond 4096 positions, against the
    row kernels over the same tokens (1e-4: two orders of fp32 sums; one of 66 pages in another's place moves a logit by some 1e-2)."""
    hp = config(pkg, heads=8, hd=64, ffn=256, layers=2, vocab=300, ple=0, gdn=False, maxL=4400, maxSeqs=3)
    out = {}
    for mode in (3, 0):
        model = pkg.Model.generate(hp, 7).randomize_gains(7)
        dev = pkg.Device(hp, 0)
        dev.upload(model)
        dev.set_page_table(np.random.default_rng(7).permutation(3 * 69).astype(np.int32))
        dev.prefill_batch([0, 1, 2], [pkg.random_tokens(7, s, hp.vocabSize, n) for s, n in enumerate((4200, 33, 4094))])
        dev.set_persistent(mode)
        assert dev.single_launch_sequences() >= 3
        lg = []
        for row in np.random.default_rng(8).integers(0, hp.vocabSize, size=(4, 3)):  # sequence 2 reaches its 65th page on the way
            dev.decode_step([int(t) for t in row])
            lg.append([dev.logits(s) for s in range(3)])
        assert dev.persistent_fallbacks() == 0
        out[mode] = np.array(lg)
        dev.close()
    for i in range(4):
        for s in range(3):
            assert_logits_close(out[3][i, s], out[0][i, s], 1e-4, f"step {i} sequence {s}")


def test_other_kernels_go_on_where_it_left_the_states(pkg, orc):
    """After a launch the delta-rule states may be in their second place: prompts that continue a sequence, a teacher-forced forward, a new
    prompt after a reset, row kernels, the one-sequence launch and kernels without copies of the matrices all find them."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64, maxSeqs=18, maxL=200)
    dev, w, prompts = start(pkg, orc, hp, 17, 4, 40, 107)
    hist = [list(p) for p in prompts]
    nxt = [dev.greedy_token(s) for s in range(17)]

    def decode(n, steps):
        out = dev.decode_loop(nxt[:n], steps)
        for s in range(n):
            hist[s] += [nxt[s]] + [int(t) for t in out[:-1, s]]
            nxt[s] = int(out[-1, s])

    def prompt(seqs, n):
        more = [pkg.random_tokens(n, s, hp.vocabSize, n + s) for s in seqs]
        dev.prefill_batch(seqs, more)
        for s, ids in zip(seqs, more):
            hist[s] += list(ids)
            nxt[s] = dev.greedy_token(s)

    assert dev.single_launch_sequences() == 16
    assert [dev.decode_route(m) for m in (1, 5, 17)] == [pkg.DECODE_XCD, pkg.DECODE_RANKS, pkg.DECODE_WIDE]
    decode(5, 2)               # 0 .. 4 in the second place
    prompt([0, 2], 7)          # row kernels
    prompt([16, 1], 40)        # tiled products
    lg, _, _ = dev.forward_full(3, np.arange(9, dtype=np.int32), want_probs=False)
    hist[3] += list(range(9))
    nxt[3] = dev.greedy_token(3)
    assert nxt[3] == int(np.argmax(lg[-1]))
    dev.reset(4)
    hist[4] = []
    prompt([4], 11)
    decode(4, 3)
    decode(17, 2)              # one launch for more rows
    decode(4, 1)
    dev.set_persistent(0)
    decode(17, 2)              # row kernels
    dev.set_persistent(3)
    decode(3, 1)
    decode(1, 2)               # one sequence
    decode(2, 1)
    dev.limit_operands(0)
    dev.finalize()
    assert dev.single_launch_sequences() <= 1
    decode(3, 2)
    for s in range(17):
        dec = orc.Decoder(w, "f64")
        for t in hist[s]:
            _, want = dec.step(int(t))
        assert dev.seq_len(s) == len(hist[s])
        assert_logits_close(dev.logits(s), want, RTOL, f"sequence {s}")
        dec.close()
    assert dev.persistent_fallbacks() == 0
    dev.close()


def test_batches_of_changing_size_share_the_exchange_words(pkg, orc):
    """Calls of 5, 2, 7 and 1 sequences in turn on one context: every size lays the exchange words out differently over what the others left."""
    hp = config(pkg, heads=12, hd=64, ffn=512, layers=4, vocab=1000, ple=64)
    dev, w, prompts = start(pkg, orc, hp, 7, 4, 50, 91)
    hist = [list(p) for p in prompts]
    nxt = [dev.greedy_token(s) for s in range(7)]
    for n in (5, 2, 7, 1, 3, 7):
        out = dev.decode_loop(nxt[:n], 2)
        for s in range(n):
            hist[s] += [nxt[s], int(out[0, s])]
            nxt[s] = int(out[1, s])
    for s in range(7):
        dec = orc.Decoder(w, "f64")
        for t in hist[s]:
            _, lg = dec.step(int(t))
        assert_logits_close(dev.logits(s), lg, RTOL, f"sequence {s}")
        assert dev.seq_len(s) == len(hist[s])
        dec.close()
    dev.close()
