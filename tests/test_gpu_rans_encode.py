"""rans_ilv encoder: blocks whose words the first pass keeps, and those past them.

The payload equals the format specification's (oracle) for blocks of even and
odd word counts, partial blocks and blocks with hardly a word; and of a plane
of more blocks than are kept (32768), blocks on both sides of the line decode
to their symbols in the specification's decoder and the whole plane on the
device.  The payload equals the specification's too on both sides of the lines
between the coded and the packed or stored form, which the encoder decides for
some planes without sizing them.
"""
import numpy as np
import pytest

import oracle as O
from ptwm_amd import api, ids, plan

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

BLOCK = 16384
KEPT = 32768


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


def symbols(n, p, seed):
    return np.random.default_rng(seed).geometric(p, n).clip(1, 255).astype(np.uint8) - 1


@pytest.mark.parametrize("n", [1, 64, 1023, BLOCK - 1, BLOCK, BLOCK + 1, 3 * BLOCK - 17, 40 * BLOCK + 5])
@pytest.mark.parametrize("p", [0.9999, 0.8, 0.15])
def test_payload(n, p):
    src = symbols(n, p, n)
    d = torch.from_numpy(src.copy()).cuda()
    out = torch.full((n + 64,), 7, dtype=torch.uint8, device="cuda:0")
    used = encode(d, out)
    got = out.cpu().numpy().tobytes()
    assert got[:used] == O.rans_ilv_encode(src.tobytes())
    assert got[used:] == b"\7" * (n + 64 - used)


def test_blocks_past_the_kept_ones():
    n = (KEPT + 3) * BLOCK + 1001
    g = torch.Generator(device="cuda:0").manual_seed(8)
    d = (torch.randn(n, generator=g, device="cuda:0") * 2).abs().to(torch.uint8)
    out = torch.zeros(n + 4096, dtype=torch.uint8, device="cuda:0")
    used, state = api.encode_tensor_cuda(plan.CHAIN_PASSTHROUGH, d, out, 0, codec="rans_ilv")
    p = plan.decode_plan(state)[0].planes[0]
    assert p.codec == ids.CODEC_RANS_ILV and p.payload_len < n // 2
    back = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL, state, out[:used],
                                              back, 0)
    assert torch.equal(back, d)
    # the blocks around the line, as a payload of their own: its header and
    # table entries for them
    max_sym = int(out[5])
    head = (5 + 1 + 2 * (max_sym + 1) + 3) // 4 * 4
    n_blocks = -(-n // BLOCK)
    base = p.payload_offset
    table = out[base + head:base + head + 4 * (n_blocks + 1)].cpu().numpy().view(np.uint32)
    lo, hi = KEPT - 2, KEPT + 2
    data = base + head + 4 * (n_blocks + 1)
    h = bytearray(out[base:base + head].cpu().numpy().tobytes())
    h[1:5] = np.uint32((hi - lo) * BLOCK).tobytes()
    part = bytes(h) + (table[lo:hi + 1] - table[lo]).astype(np.uint32).tobytes() + \
        out[data + int(table[lo]):data + int(table[hi])].cpu().numpy().tobytes()
    assert O.rans_ilv_decode(part, (hi - lo) * BLOCK) == d[lo * BLOCK:hi * BLOCK].cpu().numpy().tobytes()


def test_kept_words_are_given_back():
    """A call that needs more scratch than the card has left gets what the kept words of an earlier call hold, and
    encodes its blocks twice.  Both tensors are larger than any that another test encodes, so that their planes'
    scratch is allocated here; some 300 MiB stay free throughout."""
    mib = 1 << 20
    n, before = 6 << 30, 9 << 29
    a = (torch.randn(32 * mib, device="cuda:0") * 0.02).to(torch.bfloat16).view(torch.uint8).repeat(n // (64 * mib))
    out = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    back = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    torch.cuda.empty_cache()
    api.encode_tensor_cuda(plan.CHAIN_IEEE16_SPLIT2, a[:before], out, 0, codec="rans_ilv")  # keeps all it may
    free = torch.cuda.mem_get_info()[0]
    filler = torch.empty(free - (n - before - 700 * mib), dtype=torch.uint8, device="cuda:0")
    print("free", torch.cuda.mem_get_info()[0] // mib, "MiB, needed", (n - before) // mib, flush=True)
    try:
        used, state = api.encode_tensor_cuda(plan.CHAIN_IEEE16_SPLIT2, a, out, 0, codec="rans_ilv")
    finally:
        del filler
        torch.cuda.empty_cache()
    p = plan.decode_plan(state)[0].planes[1]
    assert p.codec == ids.CODEC_RANS_ILV and p.payload_len < n // 4
    api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL, state, out[:used],
                                              back, 0)
    assert torch.equal(back, a)
