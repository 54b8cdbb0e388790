"""mlh_profile_decode runs the step that a decode call runs, row kernels or GEMVs, and counts its parts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("nseq", [1, 5, 20])
def test_profile_decode_is_the_decode_step(pkg, bf16, nseq):
    hp = pkg.config(3, dim=256, attnHeads=4, headDim=64, ffnDim=704, transformers=4, vocabSize=1000, gdnHeads=4, pleDim=64, maxL=100,
                    maxSeqs=nseq, weightDtype=bf16)
    pkg.set_layer_pattern(hp, 1)
    model = pkg.Model.generate(hp, 5).randomize_gains(5)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    dev.set_persistent(0)
    prompts = [pkg.random_tokens(5, s, hp.vocabSize, 9 + s) for s in range(nseq)]
    for mode in (0, 1):
        dev.set_prefill_mode(mode)
        out = []
        for profile in (True, False):
            dev.reset()
            dev.prefill_batch(list(range(nseq)), prompts)
            if profile:
                parts = dev.profile_decode([1] * nseq, 4)
                assert {k: n for k, (us, n) in parts.items()} == {"k_embed": 1, "k_phaseA": 4, "k_attn": 2, "k_gdn": 2, "k_oproj": 4, "k_ffn13": 4,
                                                                  "k_down": 4, "k_lmhead": 1, "k_finish": 1}
                assert all(us > 0 for us, n in parts.values())
            else:
                dev.decode_loop([1] * nseq, 4)
            assert [dev.seq_len(s) for s in range(nseq)] == [len(p) + 4 for p in prompts]
            out.append(np.stack([dev.logits(s) for s in range(nseq)]))
        assert np.array_equal(out[0], out[1])
    dev.close()
