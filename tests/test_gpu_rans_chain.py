"""The reference rANS chains on the device, at the sizes where they can go
wrong, against the oracle byte for byte: segments around the encoder's 32-step
batches at any source alignment, alphabets that shed no byte, one and two per
step, segment counts around a workgroup's sixteen; decode rounds of 256
symbols and their ends, first states above and below the normalised range, and
streams whose bytes run out."""
import numpy as np
import pytest

import oracle as O
from ptwm_amd import api, ids, plan

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

SIZES = [1, 3, 4, 5, 31 * 4, 32 * 4, 33 * 4 + 1, 63 * 4 + 3, 65 * 4 + 2, 257 * 4, 1023 * 4 + 3, 3001 * 4 + 2]


def symbols(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "one":
        return np.full(n, 200, np.uint8)
    if kind == "rare":  # frequencies near 1 and near 2^11: two bytes in some steps, none in most
        return np.where(rng.random(n) < 0.99, 7, rng.integers(0, 256, n)).astype(np.uint8)
    if kind == "flat":  # every frequency 8: a byte in every step
        return rng.integers(0, 256, n).astype(np.uint8)
    return rng.geometric(0.3, n).clip(0, 255).astype(np.uint8)


def device(a, offset=0):
    t = torch.zeros(len(a) + offset + 16, dtype=torch.uint8, device="cuda:0")
    t[offset:offset + len(a)].copy_(torch.from_numpy(np.array(a, np.uint8)))
    return t[offset:offset + len(a)]


def decode(payload, n):
    dst = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    try:
        got = api.plane_codec_decode_cuda(ids.PLANE_CODEC_LABEL, "rans", b"", device(np.frombuffer(payload, np.uint8)),
                                          dst, 0)
    except Exception:  # noqa: BLE001
        return None
    return dst.cpu().numpy().tobytes()[:got]


@pytest.mark.parametrize("kind", ["one", "rare", "flat", "geometric"])
def test_sizes(kind):
    for k, n in enumerate(SIZES):
        plane = symbols(kind, n, n)
        print(kind, n, flush=True)
        out = torch.zeros(2 * n + 4096, dtype=torch.uint8, device="cuda:0")
        used = api.plane_codec_encode_cuda(ids.PLANE_CODEC_LABEL, "rans", b"", device(plane, 5 * k % 37), out, 0)
        want = O.codec_encode(O.CODEC_RANS, plane.tobytes())
        assert out[:used].cpu().numpy().tobytes() == want
        assert decode(want, n) == plane.tobytes()


@pytest.mark.parametrize("chunks", [1, 4, 5, 17])
def test_segment_counts(chunks):
    plane = np.concatenate([symbols("rare" if c % 2 else "geometric", 2100, c) for c in range(chunks)])[:-7]
    out = torch.zeros(2 * len(plane) + (1 << 16), dtype=torch.uint8, device="cuda:0")
    used, _ = api.encode_tensor_ref_cuda(6, [O.CODEC_RANS], 2100, device(plane), out, 0)
    want, _ = O.encode_plane_chunked(O.CODEC_RANS, plane.tobytes(), 2100)
    assert out[:used].cpu().numpy().tobytes() == want


@pytest.mark.parametrize("state", [0, 1, 1 << 11, (1 << 23) - 1, 1 << 23, (1 << 31) - 1, 1 << 31, (1 << 32) - 1])
@pytest.mark.parametrize("kind", ["one", "rare", "geometric"])
def test_first_states(kind, state):
    """Any 32-bit first state and cut or padded streams: accepted or refused as the reference does."""
    plane = symbols(kind, 5000, 11)
    good = O.codec_encode(O.CODEC_RANS, plane.tobytes())
    at = 5 + 1 + 2 * (good[5] + 1)  # the jump table: four lengths, then the streams
    lens = np.frombuffer(good[at:at + 16], "<u4")
    for seg in (0, 3):
        first = at + 16 + int(lens[:seg].sum())
        bad = bytearray(good)
        bad[first:first + 4] = int(state).to_bytes(4, "little")
        for payload in (bytes(bad), bytes(bad[:-1]), bytes(bad) + b"\x5a"):
            print(kind, state, seg, len(payload), flush=True)
            try:
                want = O.codec_decode(O.CODEC_RANS, payload, len(plane))
            except O.OracleError:
                want = None
            assert decode(payload, len(plane)) == want


def test_refused_tables():
    """Chunks whose frequencies cannot be normalised (stored raw) between coded ones, in two calls: the second finds
    the first one's tables in the same rows."""
    rng = np.random.default_rng(3)
    refused = np.repeat(np.arange(256, dtype=np.uint8), [353] * 56 + [1] * 200)
    n = len(refused)
    rng.shuffle(refused)
    assert O.codec_encode(O.CODEC_RANS, refused.tobytes())[0] == 0
    coded = [symbols(k, n, 5) for k in ("rare", "geometric", "one")]
    assert all(O.codec_encode(O.CODEC_RANS, c.tobytes())[0] == 1 for c in coded)
    for order in (coded + [refused], [refused, coded[0], refused, coded[1]], [refused] * 4):
        plane = np.concatenate(order)[:-5]
        out = torch.zeros(2 * len(plane) + (1 << 16), dtype=torch.uint8, device="cuda:0")
        print([len(o) for o in order], flush=True)
        used, _ = api.encode_tensor_ref_cuda(6, [O.CODEC_RANS], n, device(plane), out, 0)
        want, _ = O.encode_plane_chunked(O.CODEC_RANS, plane.tobytes(), n)
        assert out[:used].cpu().numpy().tobytes() == want


def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


@pytest.mark.parametrize("extra", [0, 1, 700])
def test_decode_chunk_counts(extra):
    """Chunks around the line between the decoder's two forms (four per CU), of any alphabet and alignment."""
    chunks, size = 4 * cus() + extra, 2061
    kinds = ["one", "rare", "flat", "geometric"]
    plane = np.concatenate([symbols(kinds[c % 4], size, c) for c in range(chunks)])[:-9]
    payload, entries = O.encode_plane_chunked(O.CODEC_RANS, plane.tobytes(), size)
    n = len(plane)
    st = plan.encode_plan([plan.TensorPlan(plan.CHAIN_PASSTHROUGH, 0, n, [
        plan.PlanePlan(O.CODEC_RANS, 0, len(payload), n, [tuple(map(int, e)) for e in entries])])])
    out = torch.zeros(n, dtype=torch.uint8, device="cuda:0")
    print(chunks, flush=True)
    api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL, st,
                                              device(np.frombuffer(payload, np.uint8)), out, 0)
    assert out.cpu().numpy().tobytes() == plane.tobytes()


@pytest.mark.parametrize("extra", [0, 1])
def test_decode_chunk_counts_beside_huffman(extra):
    """The line for calls that hold other jobs too: two chunks per CU."""
    chunks, size = 2 * cus() + extra, 1283
    planes = [np.concatenate([symbols(k, size, 3 * c) for c in range(chunks)])[:-9] for k in ("geometric", "rare")]
    n, blob, pp = len(planes[0]), b"", []
    for codec, plane in zip((O.CODEC_HUFFMAN, O.CODEC_RANS), planes):
        blob += b"\0" * (-len(blob) % 16)
        payload, entries = O.encode_plane_chunked(codec, plane.tobytes(), size)
        pp.append(plan.PlanePlan(codec, len(blob), len(payload), n, [tuple(map(int, e)) for e in entries]))
        blob += payload
    want = O.chain_inverse(O.CHAIN_IEEE16_SPLIT2, [p.tobytes() for p in planes])
    out = torch.zeros(2 * n, dtype=torch.uint8, device="cuda:0")
    print(chunks, flush=True)
    api.hardware_backend_dispatch_decode_cuda(
        ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL,
        plan.encode_plan([plan.TensorPlan(plan.CHAIN_IEEE16_SPLIT2, 0, 2 * n, pp)]),
        device(np.frombuffer(blob, np.uint8)), out, 0)
    assert out.cpu().numpy().tobytes() == want


@pytest.mark.parametrize("state", [0, (1 << 23) - 1, 1 << 23, (1 << 31) - 1, 1 << 31, (1 << 32) - 1])
@pytest.mark.parametrize("kind", ["one", "rare", "geometric"])
def test_first_states_of_one_among_many(kind, state):
    """As test_first_states, in the form for many chunks: the last of a call's payloads is the altered one."""
    src = symbols(kind, 5000, 11)
    good = O.codec_encode(O.CODEC_RANS, src.tobytes())
    at = 5 + 1 + 2 * (good[5] + 1)
    lens = np.frombuffer(good[at:at + 16], "<u4")
    count, room = 4 * cus() + 1, 5008
    for seg in (0, 3):
        bad = bytearray(good)
        first = at + 16 + int(lens[:seg].sum())
        bad[first:first + 4] = int(state).to_bytes(4, "little")
        for payload in (bytes(bad), bytes(bad[:-1]), bytes(bad) + b"\x5a"):
            tensors = [plan.TensorPlan(plan.CHAIN_PASSTHROUGH, room * k, len(src), [
                plan.PlanePlan(O.CODEC_RANS, 0, len(good), len(src))]) for k in range(count)]
            tensors[-1].planes[0].payload_offset = len(good)
            tensors[-1].planes[0].payload_len = len(payload)
            out = torch.zeros(room * count, dtype=torch.uint8, device="cuda:0")
            print(kind, state, seg, len(payload), flush=True)
            try:
                want = O.codec_decode(O.CODEC_RANS, payload, len(src))
            except O.OracleError:
                want = None
            try:
                api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL,
                                                          plan.encode_plan(tensors),
                                                          device(np.frombuffer(good + payload, np.uint8)), out, 0)
                got = out.view(count, room)[:, :len(src)].cpu().numpy()
            except Exception:  # noqa: BLE001
                got = None
            assert (got is None) == (want is None)
            if want is not None:
                assert (got[:-1] == src).all() and got[-1].tobytes() == want


@pytest.mark.parametrize("share", [31, 32, 33, 64, 65, 1000, 2047])
def test_slots_of_frequent_symbols(share):
    """Frequencies around the line (64 table entries) from which all lanes fill a symbol's slots, in both forms."""
    counts = np.zeros(256, int)
    counts[7] = counts[70] = share if 2 * share < 2048 else 1
    counts[200] = 2048 - counts.sum()
    src = np.repeat(np.arange(256, dtype=np.uint8), counts)
    np.random.default_rng(share).shuffle(src)
    pay = O.codec_encode(O.CODEC_RANS, src.tobytes())
    assert pay[0] == 1
    print(share, flush=True)
    assert decode(pay, len(src)) == src.tobytes()
    count = 4 * cus() + 1
    tensors = [plan.TensorPlan(plan.CHAIN_PASSTHROUGH, 2048 * k, len(src), [
        plan.PlanePlan(O.CODEC_RANS, 0, len(pay), len(src))]) for k in range(count)]
    out = torch.zeros(2048 * count, dtype=torch.uint8, device="cuda:0")
    api.hardware_backend_dispatch_decode_cuda(ids.HARDWARE_BACKEND_LABEL, ids.DECODE_PLAN_LABEL,
                                              plan.encode_plan(tensors), device(np.frombuffer(pay, np.uint8)), out, 0)
    assert (out.view(count, 2048).cpu().numpy() == src).all()
