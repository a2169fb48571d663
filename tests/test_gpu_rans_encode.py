"""rans_ilv encoder: the payload equals the format specification's (oracle)
for planes on both sides of the lines between the coded and the packed or
stored form, which the encoder decides for some of them without sizing them."""
import numpy as np
import pytest

import oracle as O
from ptwm_amd import api, ids

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BLOCK = 16384


def encode(t, out):
    return api.plane_codec_encode_cuda(ids.PLANE_CODEC_LABEL, ids.RANS_CODEC_LABEL, b"", t, out, 0)


# the block overhead of 264 bytes puts the lines near log2(k) = 0.984 * 8 and
# 0.968 * 4 bits for k equally likely symbols, less what the rounded
# frequencies cost
@pytest.mark.parametrize("n", [300, BLOCK, 5 * BLOCK + 777])
@pytest.mark.parametrize("k", [2, 10, 11, 12, 13, 14, 15, 16, 17, 180, 200, 210, 216, 222, 228, 232, 236, 240, 256])
def test_forms_near_the_line(n, k):
    rng = np.random.default_rng(1000 * k + n)
    for src in (rng.integers(0, k, n), np.minimum(rng.integers(0, k, n), rng.integers(0, 2 * k, n))):
        src = src.astype(np.uint8)
        out = torch.full((n + 64,), 7, dtype=torch.uint8, device="cuda:0")
        used = encode(torch.from_numpy(src.copy()).cuda(), out)
        assert out[:used].cpu().numpy().tobytes() == O.rans_ilv_encode(src.tobytes())
