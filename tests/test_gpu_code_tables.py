"""The encoders' entropy tables, built on the device:
payload bytes equal the oracle encoder's (header, code lengths, streams) on
histograms where the construction can go wrong: one and two symbols, ties
everywhere, Fibonacci counts (depths past the length limit, several symbols
lengthened to fit), 256 used symbols, symbol 255 alone at the end, nibble
alphabets (the 6-bit limit of huff_ilv), rANS rounding up and down, and planes
that the frequency normalisation refuses."""
import numpy as np
import pytest

import oracle as O
from ptwm_amd import api, ids

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def spread(counts, seed):
    """A plane with counts[s] of symbol s, shuffled."""
    plane = np.repeat(np.arange(len(counts), dtype=np.uint8), counts)
    np.random.default_rng(seed).shuffle(plane)
    return plane


def fibonacci(n):
    f = [1, 1]
    while len(f) < n:
        f.append(f[-1] + f[-2])
    return f


def planes():
    out = {
        "one": spread([0] * 9 + [5000], 1),
        "last": spread([900] + [0] * 254 + [70], 2),
        "two": spread([3, 4000], 3),
        "ties": spread([37] * 100, 4),
        "all": spread([20] * 256, 5),
        "fibonacci": spread(fibonacci(24), 6),
        "fibonacci reversed": spread(fibonacci(22)[::-1], 7),
        "two fibonacci": spread(fibonacci(18) + fibonacci(18), 8),
        "nibble fibonacci": spread(fibonacci(16), 9),
        "nibble ties": spread([100, 100, 100, 1, 1, 1, 1, 1, 1], 10),
        "long tail": spread([60000] + [1] * 255, 11),
        "rounding": spread([1000 // (k + 1) for k in range(200)], 12),
        "refused": spread([353] * 56 + [1] * 200, 14),
    }
    rng = np.random.default_rng(13)
    for k in range(20):
        n = int(rng.integers(2, 257))
        out[f"random {k}"] = spread((rng.pareto(0.7, n) * 3).astype(int).clip(0, 9000) + (rng.random(n) < 0.5), 20 + k)
    return {k: v for k, v in out.items() if len(v)}


PLANES = planes()


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


@pytest.mark.parametrize("name", list(PLANES))
def test_payloads(name):
    plane = PLANES[name]
    src = dev(plane)
    out = torch.zeros(2 * len(plane) + 4096, dtype=torch.uint8, device="cuda:0")
    for label, want in (("huffman", O.codec_encode(O.CODEC_HUFFMAN, plane.tobytes())),
                        ("rans", O.codec_encode(O.CODEC_RANS, plane.tobytes())),
                        (ids.PLANE_CODEC_LABEL, O.ilv_encode(plane.tobytes())),
                        (ids.RANS_CODEC_LABEL, O.rans_ilv_encode(plane.tobytes()))):
        print(name, label, len(plane), flush=True)
        n = api.plane_codec_encode_cuda(ids.PLANE_CODEC_LABEL, label, b"", src, out, 0)
        assert out[:n].cpu().numpy().tobytes() == want


def test_many_tables_in_one_call():
    """One tensor in small chunks: a table per chunk, four histogram rows each."""
    data = np.concatenate(list(PLANES.values()))
    src = dev(data)
    out = torch.zeros(2 * len(data) + (1 << 20), dtype=torch.uint8, device="cuda:0")
    for codec in (O.CODEC_HUFFMAN, O.CODEC_RANS):
        used, st = api.encode_tensor_ref_cuda(6, [codec], 777, src, out, 0)
        want, _ = O.encode_plane_chunked(codec, data.tobytes(), 777)
        assert out[:used].cpu().numpy().tobytes() == want


@pytest.mark.parametrize("n", [16, 17, 22, 30, 31, 32, 33, 44, 57, 60, 61, 88, 113, 120, 121, 225, 240, 255])
def test_flat_alphabets(n):
    """Alphabets of n equal counts: all pairs of a level are alike, so that the merge goes through rounds and leaves
    between 2 and 16 nodes of one queue to the serial steps."""
    plane = spread([37] * n, n)
    src = dev(plane)
    out = torch.zeros(2 * len(plane) + 4096, dtype=torch.uint8, device="cuda:0")
    for label, want in (("huffman", O.codec_encode(O.CODEC_HUFFMAN, plane.tobytes())),
                        (ids.PLANE_CODEC_LABEL, O.ilv_encode(plane.tobytes()))):
        print(n, label, flush=True)
        used = api.plane_codec_encode_cuda(ids.PLANE_CODEC_LABEL, label, b"", src, out, 0)
        assert out[:used].cpu().numpy().tobytes() == want
