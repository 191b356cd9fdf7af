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


# 24 tokens on the few-token matvec, 65 and 95 on the 32-token kernels, the rest
# on the tiled one: K splits of one to four parts
@pytest.mark.parametrize("qtype,k,rows,m,crc", [
    (synth.Q4_K, 2560, 300, 24, 263964610), (synth.Q4_K, 2560, 1000, 65, 514150326),
    (synth.Q4_K, 2560, 1000, 95, 1752270011), (synth.Q4_K, 2560, 1000, 96, 592997306),
    (synth.Q4_K, 9728, 513, 130, 1119775581), (synth.Q4_K, 2560, 6144, 512, 1719389901),
    (synth.Q4_K, 256, 1, 100, 4253233896), (synth.Q4_K, 4096, 2560, 333, 3376873728),
    (synth.Q4_K, 2304, 640, 900, 2955258594), (synth.Q6_K, 2560, 300, 24, 2335545069),
    (synth.Q6_K, 2560, 1000, 65, 2692310153), (synth.Q6_K, 2560, 1000, 95, 795841049),
    (synth.Q6_K, 2560, 1000, 96, 2543986180), (synth.Q6_K, 9728, 513, 130, 3445473103),
    (synth.Q6_K, 2560, 6144, 512, 1992489358), (synth.Q6_K, 256, 1, 100, 605201952),
    (synth.Q6_K, 4096, 2560, 333, 4250083847), (synth.Q6_K, 2304, 640, 900, 3129518966),
])
def test_kquant_product_bits(qtype, k, rows, m, crc):
    """Inputs with a heavy tail (cubed normals)."""
    raw = synth.quantize(qtype, synth.gaussian(71, k + rows + qtype, rows * k, 0.02).reshape(rows, k))
    X = synth.gaussian(72, k + m, m * k, 1.0).reshape(m, k) ** 3
    assert _crc(eng.matmul(qtype, raw, rows, k, X)) == crc


@pytest.mark.parametrize("k,rows,m,fused,crc", [
    (2560, 1000, 70, True, 1717677690), (2560, 2560, 101, False, 451792006), (1024, 2820, 900, True, 3251317571),
    (2560, 9728, 512, True, 3292148604), (512, 2560, 900, True, 2681902950),
])
def test_q4k_gate_up_bits(k, rows, m, fused, crc):
    g = synth.quantize(synth.Q4_K, synth.gaussian(73, k + rows, rows * k, 0.02).reshape(rows, k))
    u = synth.quantize(synth.Q4_K, synth.gaussian(74, k + rows, rows * k, 0.02).reshape(rows, k))
    X = synth.gaussian(75, k + m, m * k, 1.0).reshape(m, k)
    y, one_launch = eng.matmul_swiglu(synth.Q4_K, g, u, rows, k, X)
    assert one_launch == fused and _crc(y) == crc


def test_conversation_bits(gguf_factory):
    """A Q4_K_M conversation of growing and shrinking segments, a sampled
    reply, scores, and two batches of sampled replies."""
    model = eng.Model(gguf_factory("mid", "q4_k_m"), max_pos=2048)
    rng = np.random.default_rng(5)

    def ids(n):
        return rng.integers(0, 32000, n, dtype=np.int32)

    s = model.session(2048)
    turns = [(700, 2611664729), (24, 3362935199), (130, 3519248235), (1, 1733760205), (64, 2136527876),
             (65, 3586634463), (300, 3345292912), (2, 1123258492)]
    assert [(n, _crc(s.prefill(ids(n)))) for n, _ in turns] == turns
    assert _crc(s.generate(24, 0.2, 0, 0.95, 77)) == 3017764523
    s = model.session(1024)
    s.prefill(ids(50))
    scores = [(8, 2850593359), (40, 1962683207), (200, 501750474)]
    assert [(n, _crc(s.prefill(ids(n), all_logits=True))) for n, _ in scores] == scores
    for n, reply, after in [(3, 3979195660, 1440404889), (8, 1401735295, 1483802196)]:
        sessions = [model.session(512) for _ in range(n)]
        for x in sessions:
            x.prefill(ids(100 + n))
        got, _ = eng.generate_batch(sessions, 16, 0.2, 0, 0.95, [9 + i for i in range(n)])
        assert (_crc(got), _crc(np.stack([x.prefill(ids(3)) for x in sessions]))) == (reply, after)


@pytest.mark.parametrize("mix", ["q4_k_m", "q8_0"])
def test_bits_do_not_depend_on_a_sessions_past(gguf_factory, mix):
    """The same turns give the same logits in a session that only ever took
    short segments and in one whose scratch a long segment has grown (8 KV
    heads, to a history whose key images are some 30 MB)."""
    model = eng.Model(gguf_factory("tiny", mix, n_heads=16, n_kv_heads=8), max_pos=4096)
    rng = np.random.default_rng(8)
    turns = [rng.integers(0, 1024, n, dtype=np.int32) for n in [100] * 36 + [70, 33, 128, 2, 81]]
    short, grown = model.session(4096), model.session(4096)
    grown.prefill(rng.integers(0, 1024, 4096, dtype=np.int32))
    grown.set_len(0)
    for t in turns:
        assert np.array_equal(short.prefill(t).view(np.uint32), grown.prefill(t).view(np.uint32))
