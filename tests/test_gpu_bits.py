"""Bits that stay: a sampled reply depends on the last bits of the logits
wherever a draw falls next to an edge of the distribution, so a seed gives the
reply it gave before only while the arithmetic behind the cache and the logits
keeps its order of sums. The CRC32s below are those of the kernels that the
replies were first recorded with (one MI355X, 256 compute units: the split
products' K parts follow the count)."""

import zlib

import numpy as np
import pytest

import oracle
import rpgbarengine_amd as eng

pytestmark = pytest.mark.gpu


def _crc(a):
    return zlib.crc32(np.ascontiguousarray(a).tobytes())


# seq, heads, KV heads, pos0: segments below and above the length from which
# the key blocks are converted once (81 queries), every group size, one and
# two query tiles per workgroup
@pytest.mark.parametrize("seq,n_heads,n_kv,pos0,crc", [
    (3, 32, 8, 3990, 2138426575), (24, 32, 8, 1000, 3960973222), (80, 2, 2, 9, 486787970),
    (81, 2, 2, 0, 2980881145), (96, 16, 8, 0, 3239603172), (130, 3, 1, 77, 501665710),
    (203, 32, 8, 1500, 2800405350), (97, 5, 1, 300, 304778863), (90, 6, 1, 40, 1261959375),
    (100, 7, 1, 64, 1158332145), (120, 8, 1, 50, 3911523053), (1040, 16, 8, 13, 4284863714),
    (2050, 8, 8, 5, 2956879740)])
def test_prefill_attention_bits(seq, n_heads, n_kv, pos0, crc):
    """Values with a heavy tail (seventh powers), so that the V scales of the
    key blocks vary; also against the oracle, at 2e-5 of the largest value."""
    rng = np.random.default_rng([seq, n_heads, pos0])
    q = rng.standard_normal((seq, n_heads, 128)).astype(np.float32)
    k = rng.standard_normal((n_kv, pos0 + seq, 128)).astype(np.float32)
    v = (rng.standard_normal((n_kv, pos0 + seq, 128)) ** 7).astype(np.float32)
    got = eng.attention(q, k, v, pos0)
    if seq < 1000:
        assert np.abs(got - oracle.attention(q, k, v, pos0)).max() <= 2e-5 * np.abs(v).max()
    assert _crc(got) == crc
