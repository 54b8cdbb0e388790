"""The XCD-rank decode kernel (csrc/kernels_xcd.hip) where its fixed-width reads change: numbers of 32-key tiles around the rounds of
the softmax combine, widths of the exchanged rows, XCDs without heads, the form for wide models; against the kernel sequence."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


# dim, head size, ffn, gating, bf16: 4 heads (four XCDs have none); 8 heads of 64; 12 heads; the widest rows of either type
@pytest.mark.parametrize("d,hd,ffn,gate,bf16", [(256, 64, 704, 0, 0), (512, 64, 1408, 1, 0), (768, 64, 2048, 1, 0), (1024, 128, 2816, 0, 0), (2048, 64, 5632, 1, 1)])
@pytest.mark.parametrize("n", [2, 126, 254, 382, 766, 1022])
def test_xcd_against_kernel_sequence(pkg, d, hd, ffn, gate, bf16, n):
    hp = pkg.config(2, dim=d, attnHeads=d // hd, headDim=hd, ffnDim=ffn, transformers=2, vocabSize=1000, queryGating=gate, qkRmsNorm=1,
                    maxL=1040, maxSeqs=1, weightDtype=bf16)
    model = pkg.Model.generate(hp, 5)
    dev = pkg.Device(hp, 0)
    dev.upload(model)
    assert dev.xcd_decode_supported()
    ids = np.random.default_rng(n).integers(0, 1000, n).astype(np.int32)
    out = {}
    for mode in (0, 3):
        dev.set_persistent(mode)
        dev.reset()
        dev.prefill(0, ids)
        picks = dev.decode_loop([7], 4)  # the new key is the last of a tile, then the first of the next
        out[mode] = (picks, dev.logits(0))
        assert dev.get_persistent() == mode if hasattr(dev, "get_persistent") else True
    assert np.array_equal(out[0][0], out[3][0])
    assert rel(out[3][1], out[0][1]) < 1e-5
    dev.close()
