"""The 16-bit split that also counts its planes: payloads of a tensor's planes
equal the oracle encoder's for each plane alone, at sizes around the vector of
16, a workgroup's pass and the whole grid's, on skewed and on flat planes, and
beside a chain whose planes are counted in a pass of their own."""
import pytest

import oracle as O
from ptwm_amd import api, ids, plan

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

ORACLE = {"huff_ilv": O.ilv_encode, "rans_ilv": O.rans_ilv_encode}


def check(codec, items, used, out, st):
    blob = out[:used].cpu().numpy().tobytes()
    for (chain, src), t in zip(items, plan.decode_plan(st)):
        planes = O.chain_forward(chain, src.cpu().numpy().tobytes())
        for raw, p in zip(planes, t.planes):
            raw = bytes(raw)
            got = blob[p.payload_offset:p.payload_offset + p.payload_len]
            assert got == (raw if p.codec == O.CODEC_IDENTITY else ORACLE[codec](raw))


@pytest.mark.parametrize("codec", list(ORACLE))
@pytest.mark.parametrize("n", [0, 1, 15, 16, 17, 16 * 1024 - 1, 16 * 1024 + 5, 256 * 16 * 1024 + 16 * 7 + 3])
def test_payloads(n, codec):
    g = torch.Generator(device="cuda:0").manual_seed(n + 1)
    a = (torch.randn(n, generator=g, device="cuda:0") * 0.02).to(torch.bfloat16).view(torch.uint8)
    b = torch.randint(0, 256, (2 * n,), generator=g, device="cuda:0", dtype=torch.uint8)
    c = torch.randint(0, 9, (4 * (n % 5000),), generator=g, device="cuda:0", dtype=torch.uint8)
    c16 = plan.CHAIN_IEEE16_SPLIT2
    print(codec, n, flush=True)
    for items in ([(c16, a)], [(c16, b), (plan.CHAIN_IEEE32_SPLIT4, c), (c16, a)]):
        out = torch.zeros(sum(2 * t.numel() for _, t in items) + (1 << 16), dtype=torch.uint8, device="cuda:0")
        if len(items) == 1:
            used, st = api.encode_tensor_cuda(*items[0], out, 0, codec=codec)
        else:
            used, st = api.encode_tensors_cuda(items, out, 0, codec=codec)
        check(codec, items, used, out, st)
