"""GPU parity of the trellis format kernels (decode, pack, unpack): every
state of every codebook against the library's host table, and the shapes at
which the kernels' tiling ends (one tile, a workgroup's tiles and one more or
less), against the CPU oracle, bit for bit."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hb():
    import hip_backend
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    hip_backend.lib()
    return hip_backend


def _bits(shape, seed, offset=0):
    """Random trellis words on the GPU, `offset` int16 elements into their
    allocation."""
    g = torch.Generator().manual_seed(seed)
    n = int(np.prod(shape))
    buf = torch.randint(-32768, 32768, (n + offset,), generator=g, dtype=torch.int16).cuda()
    return buf[offset:].view(shape)


@pytest.mark.parametrize("code", ("mul1", "3inst", "mcg", "1mad"))
def test_decode_every_state(hb, oracle_mod, code):
    """The computed codebook values equal the table's at all 65,536 states."""
    tr = _bits((64, 64, 48), 1)
    states = oracle_mod.unpack(tr.cpu().numpy().reshape(-1, 48), 3)
    assert np.unique(states).size == 65536
    lut = hb.get_lut(code).numpy()
    want = oracle_mod.decode(tr.cpu().numpy(), lut, 3)
    np.testing.assert_array_equal(hb.decode(tr, 3, code=code).cpu().numpy(), want)
    np.testing.assert_array_equal(hb.decode(tr, 3, code=code, dtype=torch.float16).cpu().numpy(),
                                  want.astype(np.float16))


@pytest.mark.parametrize("K", range(2, 8))
@pytest.mark.parametrize("tk,tn,offset", [(1, 1, 0), (3, 15, 1), (2, 16, 0), (5, 17, 1), (1, 33, 0)])
def test_format_edges(hb, oracle_mod, mul1_lut, K, tk, tn, offset):
    """Ragged tile counts, also from words at an odd 16-bit address."""
    tr = _bits((tk, tn, 16 * K), 10 * K + tn, offset)
    host = tr.cpu().numpy()
    st = oracle_mod.unpack(host.reshape(-1, 16 * K), K)
    np.testing.assert_array_equal(hb.unpack(tr, K).cpu().numpy(), st)
    st64 = hb.unpack64(tr, K)
    assert st64.dtype == torch.int64
    np.testing.assert_array_equal(st64.cpu().numpy(), st)
    np.testing.assert_array_equal(hb.decode(tr, K).cpu().numpy(),
                                  oracle_mod.decode(host, mul1_lut, K))
    # symbols are the states' low bits: higher bits are ignored
    for packed in (hb.pack(hb.unpack(tr, K) | (1 << 20), K), hb.pack64(st64 | (1 << 40), K)):
        np.testing.assert_array_equal(packed.cpu().numpy(), host.reshape(-1, 16 * K))
