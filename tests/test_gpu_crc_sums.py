"""Plane CRCs summed on the device by the fused decode kernels (whole 16 KiB
blocks on the matrix cores, the last one padded with zeros, each block's sum
moved to the plane's end and XORed into the plane's accumulator):

- every chain in both GPU-native codecs, at plane lengths around the 16-byte
  piece, the 1 KiB round, the 16 KiB block and the 256-block step of the block
  weights, several such tensors in one call and each alone; the wanted CRCs
  are the oracle's, a flipped bit of any plane's CRC is refused;
- the mixed nibble-split and passthrough launch;
- a plane past 65536 blocks (the next step of the block weights);
- nibble-chain planes that hold symbols above 15: the merge masks them, the
  CRC covers them as they are (the tensor is decoded through plane scratch).
"""
import numpy as np
import pytest

import oracle as O
from ptwm_amd import api, ids, plan

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

LENGTHS = [1, 15, 17, 1023, 1025, 16383, 16384, 16385, 4 * 16384 + 7 * 1024 + 3, 257 * 16384 + 5]
CHAINS = [1, 2, 3, 4, 5, 6]
CODECS = {"huff_ilv": (ids.CODEC_HUFF_ILV, ids.PLANE_CODEC_LABEL), "rans_ilv": (ids.CODEC_RANS_ILV,
                                                                               ids.RANS_CODEC_LABEL)}


def dev(b):
    return torch.from_numpy(np.frombuffer(bytes(b), np.uint8).copy()).to("cuda:0")


def data(chain, n, seed):
    """Tensor bytes whose planes are n long: skewed, so that planes code."""
    rng = np.random.default_rng(seed)
    size = n * plan.CHAIN_RATIO[chain]
    return np.minimum(rng.geometric(0.15, size) * 3, 255).astype(np.uint8).tobytes()


def encode(items, codec):
    src = [(c, dev(d)) for c, d in items]
    out = torch.zeros(2 * sum(t.numel() for _, t in src) + 65536 * len(src), dtype=torch.uint8, device="cuda:0")
    used, st = api.encode_tensors_cuda(src, out, 0, codec=codec)
    tensors = plan.decode_plan(st)
    for (c, d), t in zip(items, tensors):
        for p, pb in zip(t.planes, O.chain_forward(c, d)):
            p.crc32 = O.crc32(pb)
    return out[:used], tensors


def decode(tensors, blob):
    total = max(t.out_offset + t.out_len for t in tensors)
    out = torch.zeros(total, dtype=torch.uint8, device="cuda:0")
    api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL,
                                              plan.encode_plan(tensors), blob, out, 0)
    return out.cpu().numpy().tobytes()


def check(items, tensors, blob):
    got = decode(tensors, blob)
    for (_, d), t in zip(items, tensors):
        assert got[t.out_offset:t.out_offset + t.out_len] == d


def refused(tensors, blob, p):
    p.crc32 ^= 1 << (p.plane_len % 32)
    with pytest.raises(Exception) as e:
        decode(tensors, blob)
    assert getattr(e.value, "rc", None) == -1
    p.crc32 ^= 1 << (p.plane_len % 32)


@pytest.mark.parametrize("codec", list(CODECS))
@pytest.mark.parametrize("chain", CHAINS)
def test_lengths(chain, codec):
    items = [(chain, data(chain, n, 7 * chain + k)) for k, n in enumerate(LENGTHS)]
    blob, tensors = encode(items, codec)
    check(items, tensors, blob)
    for t in tensors:
        for p in t.planes:
            refused(tensors, blob, p)
    for k, t in enumerate(tensors):
        print("alone", chain, codec, LENGTHS[k], flush=True)
        got = decode([t], blob)
        assert got[t.out_offset:t.out_offset + t.out_len] == items[k][1]
        refused([t], blob, t.planes[-1])


def test_mixed_launch():
    items = [(5, data(5, 70_001, 1)), (6, data(6, 4379, 2)), (5, data(5, 16384, 3)), (6, data(6, 33_000, 4))]
    blob, tensors = encode(items, "huff_ilv")
    check(items, tensors, blob)
    for t in tensors:
        for p in t.planes:
            refused(tensors, blob, p)


def test_past_65536_blocks():
    n = 65536 * 16384 + 3 * 16384 + 77
    g = torch.Generator(device="cuda:0").manual_seed(9)
    src = torch.randint(100, 104, (n,), generator=g, device="cuda:0", dtype=torch.uint8)
    out = torch.zeros(n // 2, dtype=torch.uint8, device="cuda:0")
    used, st = api.encode_tensors_cuda([(6, src)], out, 0)
    tensors = plan.decode_plan(st)
    tensors[0].planes[0].crc32 = O.crc32(src.cpu().numpy())
    back = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL,
                                              plan.encode_plan(tensors), out[:used], back, 0)
    assert torch.equal(back, src)
    tensors[0].planes[0].crc32 ^= 2
    with pytest.raises(Exception) as e:
        api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL,
                                                  plan.encode_plan(tensors), out[:used], back, 0)
    assert getattr(e.value, "rc", None) == -1


@pytest.mark.parametrize("codec", list(CODECS))
@pytest.mark.parametrize("blocks", [8191, 8193])
def test_many_blocks_without_sums(codec, blocks):
    """Tensors with plane CRCs beside one without: in its launch up to 8192 of its blocks, else in one of their own."""
    n = blocks * 16384 - 77
    g = torch.Generator(device="cuda:0").manual_seed(blocks)
    plain = torch.randint(100, 104, (n,), generator=g, device="cuda:0", dtype=torch.uint8)
    items = [(6, data(6, 20_001, 1)), (6, data(6, 33_000, 2))]
    src = [(6, dev(items[0][1])), (6, plain), (6, dev(items[1][1]))]
    out = torch.zeros(n // 2, dtype=torch.uint8, device="cuda:0")
    used, st = api.encode_tensors_cuda(src, out, 0, codec=codec)
    tensors = plan.decode_plan(st)
    for k in (0, 2):
        tensors[k].planes[0].crc32 = O.crc32(items[k // 2][1])
    plain_plan = plan.encode_plan([tensors[1]])
    total = tensors[2].out_offset + tensors[2].out_len
    for wrong in (False, True):
        back = torch.zeros(total, dtype=torch.uint8, device="cuda:0")
        if wrong:
            tensors[2].planes[0].crc32 ^= 4
        # has_crc is a tensor's own flag: each tensor encoded by itself, then joined
        parts = [plan.encode_plan([tensors[0]]), plain_plan, plan.encode_plan([tensors[2]])]
        joined = parts[0][:8] + (3).to_bytes(4, "little") + b"".join(p[12:] for p in parts)
        print(codec, blocks, wrong, flush=True)
        if wrong:
            with pytest.raises(Exception) as e:
                api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL, joined,
                                                          out[:used], back, 0)
            assert getattr(e.value, "rc", None) == -1
            continue
        api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL, joined,
                                                  out[:used], back, 0)
        for (_, s), t in zip(src, tensors):
            assert torch.equal(back[t.out_offset:t.out_offset + t.out_len], s)


@pytest.mark.parametrize("stored", [False, True])
@pytest.mark.parametrize("codec", list(CODECS))
@pytest.mark.parametrize("chain", [3, 4, 5])
def test_wide_symbols_in_a_nibble_chain(chain, codec, stored):
    n = 3 * 16384 + 901
    rng = np.random.default_rng(chain)
    planes = [np.minimum(rng.geometric(0.3, n), 15).astype(np.uint8) for _ in range(2)]
    planes[0][n - 5] = 0x31  # one symbol above 15
    wire, label = CODECS[codec]
    blob, pp = b"", []
    for k, pb in enumerate(planes):
        blob += b"\0" * (-len(blob) % 256)
        if k == 0 and stored:
            pay, c = pb.tobytes(), ids.CODEC_IDENTITY
        else:
            buf = torch.zeros(2 * n, dtype=torch.uint8, device="cuda:0")
            used = api.plane_codec_encode_cuda(label, label, b"", dev(pb), buf, 0) if codec == "huff_ilv" else \
                api.plane_codec_encode_cuda(ids.PLANE_CODEC_LABEL, label, b"", dev(pb), buf, 0)
            pay, c = buf[:used].cpu().numpy().tobytes(), wire
        pp.append(plan.PlanePlan(c, len(blob), len(pay), n, crc32=O.crc32(pb.tobytes())))
        blob += pay
    t = plan.TensorPlan(chain, 0, n, pp)
    want = O.chain_inverse(chain, [(pb & 15).tobytes() for pb in planes])
    assert decode([t], dev(blob)) == want
    for p in pp:
        refused([t], dev(blob), p)
