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
from rpgbarengine_amd import synth

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


# Two layers of the 1.7B width (a gate+up pair of 16.8 M weights), a segment
# per entry: (tokens, logits of every position wanted, CRC of the logits)
SHORT = {
    "q4_k_m": [(20, 0, 1949256523), (41, 0, 3275326450), (64, 0, 432836158), (2, 0, 1009124003),
               (8, 1, 490016019), (40, 1, 3505451445), (64, 1, 3998693554)],
    "q8_0": [(20, 0, 2284655582), (41, 0, 1172620475), (64, 0, 4085952823), (2, 0, 3567769502),
             (8, 1, 1359826666), (40, 1, 1070287797), (64, 1, 3021317139)],
}


@pytest.mark.parametrize("mix", sorted(SHORT))
def test_short_segment_bits(gguf_factory, mix):
    """Segments of up to 64 tokens stay on the few-token matvec, and the logits
    of every position on fp32 inputs, whatever a wider launch would take."""
    model = eng.Model(gguf_factory("tiny", mix, hidden=2048, n_heads=16, ffn=4096), max_pos=1024)
    s = model.session(1024)
    rng = np.random.default_rng(6)
    got = []
    for n, every, _ in SHORT[mix]:
        ids = rng.integers(0, 1024, n, dtype=np.int32)
        got.append(_crc(s.prefill(ids, all_logits=bool(every))))
    assert got == [c for _, _, c in SHORT[mix]]
