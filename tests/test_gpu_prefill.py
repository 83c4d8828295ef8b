"""Prefill chunks through attention and the decoder layer on the GPU against
the oracle's one-token path run over the same tokens in order (a chunk must
give what decoding its tokens one after another gives): full attention with
its KV cache, Gated DeltaNet with its convolution and recurrent state, and a
whole decoder layer, over two consecutive chunks; chunks of 64 tokens and
more take the MFMA projections. Outputs within 1e-3 of their largest value,
caches and states elementwise within 1e-3 of their largest value."""
import numpy as np
import pytest
import torch

import pyoracle as po
from adi_amd import hip
from adi_amd import synthetic as syn
from conftest import max_rel_error

pytestmark = pytest.mark.gpu

HIDDEN = 256
CHUNKS = [(0, 7), (7, 70)]  # (position, count): a short chunk, then one on the MFMA path


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def close(got, want, what):
    assert np.max(np.abs(got - want)) <= 1e-3 * np.max(np.abs(want)), what


@pytest.fixture(scope="module")
def tluts():
    rng = syn.rng_for(60, 0)
    return syn.expert_tlut(rng), syn.ne_tlut(rng)


def test_full_attention_prefill(gpu, oracle, tluts):
    rng = syn.rng_for(61, 0)
    layer = syn.full_attention(rng, HIDDEN, tluts[1])
    d = hip.upload_full_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    held = po.FullAttentionStruct(layer)
    capacity = sum(c for _, c in CHUNKS)
    keys = np.zeros((capacity, 2, 256), np.float32)
    values = np.zeros_like(keys)
    dk = torch.zeros((capacity, 2, 256), dtype=torch.float32, device="cuda")
    dv = torch.zeros_like(dk)
    for position, count in CHUNKS:
        x = syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN))
        want = np.stack([po.full_attention_forward(oracle, held, position + b, x[b], keys, values)
                         for b in range(count)])
        out = torch.empty((count, HIDDEN), dtype=torch.float32, device="cuda")
        hip.full_attention_prefill(gpu, d, position, count, dev(x), out, dk, dv, capacity)
        assert max_rel_error(out.cpu().numpy(), want) <= 1e-3, (position, count)
        end = position + count
        close(dk.cpu().numpy()[:end], keys[:end], "keys")
        close(dv.cpu().numpy()[:end], values[:end], "values")


@pytest.mark.parametrize("position,count", [(1016, 16), (1000, 17), (500, 47), (0, 256), (130, 129), (4000, 20)])
def test_attention_chunk_edges(gpu, oracle, tluts, position, count):
    """The matrix-core attention of a chunk at the edges of its 16-token
    blocks and 32-key tiles, with one and several splits, against the oracle's
    one-token form for the first, last and middle tokens (the caches as the
    chunk left them). Both sides sum in floats; the largest difference seen is
    2.9e-6 of the largest output (20 tokens at 4000), and 1e-5 is about four
    times that. test_attention_chunk_precision holds the pieces to 64 bits."""
    rng = syn.rng_for(66, position + count)
    layer = syn.full_attention(rng, HIDDEN, tluts[1])
    d = hip.upload_full_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    held = po.FullAttentionStruct(layer)
    capacity = position + count
    dk = dev(rng.normal(0.0, 1.0, (capacity, 2, 256)).astype(np.float32))
    dv = dev(rng.normal(0.0, 1.0, (capacity, 2, 256)).astype(np.float32))
    x = syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN))
    out = torch.empty((count, HIDDEN), dtype=torch.float32, device="cuda")
    hip.full_attention_prefill(gpu, d, position, count, dev(x), out, dk, dv, capacity)
    keys, values = dk.cpu().numpy(), dv.cpu().numpy()
    for b in sorted({0, 1, 15, count // 2, count - 1}):
        want = po.full_attention_forward(oracle, held, position + b, x[b], keys.copy(), values.copy())
        assert max_rel_error(out[b].cpu().numpy(), want) <= 1e-5, b


@pytest.mark.parametrize("case", ["token", "key", "value", "large", "query", "unseen"])
def test_attention_chunk_odd_values(gpu, tluts, case):
    """Values the matrix cores' pieces cannot stand for: a NaN token (its row
    and those after it are NaN, those before it are not), an infinity in the
    history's keys or values, finite values beyond f16 and bf16, a query of 2^62,
    and keys of 2^70 in the first, a middle, the last whole and the chunk's own
    tile where the query is 0, so that tiles in floats and on the matrix cores
    take turns at one softmax, give what the vector kernel (chunks of 8 tokens)
    gives."""
    rng = syn.rng_for(67, len(case))
    layer = syn.full_attention(rng, HIDDEN, tluts[1])
    if case == "query":
        layer.query_norm[100] = 0x5E80  # 2^62 in bf16
    elif case == "unseen":
        layer.query_norm[100] = 0xBF80  # -1: times 0
    d = hip.upload_full_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    position, count = 600, 40
    keys = rng.normal(0.0, 1.0, (position + count, 2, 256)).astype(np.float32)
    values = rng.normal(0.0, 1.0, (position + count, 2, 256)).astype(np.float32)
    x = syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN))
    if case == "unseen":
        keys[[5, 300, 575, 599], :, 100] = 2.0 ** 70
        keys[64:96, :, 100] = -2.0 ** 70
    elif case == "query":
        pass
    elif case == "token":
        x[21, 5] = np.nan
    elif case == "key":
        keys[70, 0, 9] = np.inf
    elif case == "value":
        values[333, 1, 200] = -np.inf
    else:
        keys[70, 0, 9] = 3e5
        values[599, 1, 3] = 3.4e38

    def run(step):
        dk, dv = dev(keys), dev(values)
        out = torch.empty((count, HIDDEN), dtype=torch.float32, device="cuda")
        for b in range(0, count, step):
            hip.full_attention_prefill(gpu, d, position + b, step, dev(x[b:b + step]), out[b:b + step], dk, dv,
                                       position + count)
        return out.cpu().numpy()

    got, want = run(count), run(8)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    if case == "token":
        assert np.isfinite(got[:21]).all() and np.isnan(got[21:]).all()
    for a, b in zip(got, want):
        if np.isfinite(b).all():
            assert max_rel_error(a, b) <= 1e-4


def hadamard64(v):
    n, lead, h = v.shape[-1], v.shape[:-1], 1
    while h < n:
        v = v.reshape(*lead, n // (2 * h), 2, h)
        v = np.stack((v[..., 0, :] + v[..., 1, :], v[..., 0, :] - v[..., 1, :]), -2)
        h *= 2
    return v.reshape(*lead, n) / np.sqrt(n)


def ne64(m, x):
    """An NE projection in 64 bits: 16-bit windows of each tile's 64 words, one
    every 8 bits, through the state table."""
    w = np.asarray(m.trellis).astype(np.int64).reshape(-1, 64) & 0xFFFF
    at = np.arange(128) * 8
    pair = (w[:, at // 16] << 16) | w[:, (at // 16 + 1) % 64]
    state = (pair >> (16 - at % 16)) & 0xFFFF
    product = state * (state + 1)
    v = np.asarray(m.tlut, np.float64).astype(np.float16).astype(np.float64).reshape(512, 2)[(product >> 6) & 0x1FF]
    v[..., 0] *= 1.0 - 2.0 * ((product >> 15) & 1)
    dense = v.reshape(m.rows // 16, m.columns // 16, 16, 16).transpose(0, 2, 1, 3).reshape(m.rows, m.columns)
    return hadamard64(hadamard64(x * np.asarray(m.su, np.float64)) @ dense.T * m.weight_scale) * np.asarray(m.sv, np.float64)


def full_attention64(layer, position, x, keys, values, planted=None):
    """A chunk's attention in 64 bits over the history keys[:position],
    values[:position]; `planted` changes (weights, values) before their product."""
    n = len(x)
    positions = np.arange(position, position + n)
    bf16 = lambda bits: (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    angle = (positions.astype(np.float32)[:, None]
             / np.power(1e7, np.arange(32) / 32.0).astype(np.float32)).astype(np.float64)[:, None]

    def norm_rope(v, weight):
        v = v / np.sqrt((v * v).mean(-1, keepdims=True) + 1e-6) * (1.0 + bf16(weight))
        c, s = np.cos(angle), np.sin(angle)
        return np.concatenate((v[..., :32] * c - v[..., 32:64] * s, v[..., 32:64] * c + v[..., :32] * s, v[..., 64:]), -1)

    qg = ne64(layer.query, x).reshape(n, 16, 2, 256)
    q, gate = norm_rope(qg[:, :, 0], layer.query_norm), qg[:, :, 1]
    k = np.concatenate((keys[:position], norm_rope(ne64(layer.key, x).reshape(n, 2, 256), layer.key_norm)))
    v = np.concatenate((values[:position], ne64(layer.value, x).reshape(n, 2, 256)))
    attended = np.empty((n, 16, 256))
    for h in range(16):
        s = q[:, h] @ k[:, h // 8].T / 16.0
        s[np.arange(position + n)[None] > positions[:, None]] = -np.inf
        w = np.exp(s - s.max(1, keepdims=True))
        held = v[:, h // 8]
        if planted is not None:
            w, held = planted(w, held)
        attended[:, h] = w @ held / w.sum(1, keepdims=True)
    return ne64(layer.output, (attended / (1.0 + np.exp(-gate))).reshape(n, -1))


# The query and key scales of the chunk attention's precision test: the query
# norm's weight (a scale of 1 + w), the scale of the history's keys, and a scale
# of dimension 100's keys with the query's norm weight there.
PRECISION = {
    "flat": (-1 + 2.0 ** -4, 1.0, None), "unit": (0.0, 1.0, None), "low keys": (255.0, 2.0 ** -8, None),
    "lower keys": (2.0 ** 13, 2.0 ** -13, None), "lowest keys": (2.0 ** 30, 2.0 ** -30, None),
    "high keys": (-1 + 2.0 ** -8, 2.0 ** 8, None),
    "one dimension": (255.0, 2.0 ** -8, (2.0 ** 8, -1 + 2.0 ** -8))}


def precision_case(tlut, name):
    """Layer, position, tokens and history of a case. The fresh keys are 0 (their
    norm weight is -1), so that scores come from the history's scale alone."""
    weight, scale, dimension = PRECISION[name]
    rng = syn.rng_for(68, sorted(PRECISION).index(name))
    layer = syn.full_attention(rng, HIDDEN, tlut)
    bf16 = lambda v: np.array([v], np.float32).view(np.uint32)[0] >> 16
    layer.query_norm[:] = bf16(weight)
    layer.key_norm[:] = bf16(-1.0)
    position, count = 1000, 64
    keys = rng.normal(0.0, scale, (position + count, 2, 256)).astype(np.float32)
    values = rng.normal(0.0, 1.0, (position + count, 2, 256)).astype(np.float32)
    if dimension is not None:
        keys[:, :, 100] *= dimension[0] / scale
        layer.query_norm[100] = bf16(dimension[1])
    return layer, position, syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN)), keys, values


def two_bf16_pieces(v):
    """v rounded to bf16 plus the rest rounded to bf16."""
    v, out = np.asarray(v, np.float32), 0.0
    for _ in range(2):
        bits = (v - np.float32(out)).view(np.uint32)
        out = out + ((bits + 0x7FFF + ((bits >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)
    return out.astype(np.float64)


@pytest.mark.parametrize("name", list(PRECISION))
def test_attention_chunk_precision(gpu, tluts, name):
    """The layer's error against 64 bits at query and key scales from 2^-30 to
    2^30, and with one dimension's keys 2^16 times the others'. The projections'
    part is about 5e-7 (relative, 2-norm), which the vector kernel shows too; the
    bound is twice the 6.2e-7 seen. Weights or values in two pieces instead of
    three, planted in the 64-bit form, are past it by half, and pieces of
    unscaled keys were 3e-6 to 1e-4 off."""
    bound = 1.25e-6
    layer, position, x, keys, values = precision_case(tluts[1], name)
    want = full_attention64(layer, position, x, keys, values)
    error = lambda got: np.linalg.norm(got - want) / np.linalg.norm(want)
    for planted in (lambda w, v: (two_bf16_pieces(w), v), lambda w, v: (w, two_bf16_pieces(v))):
        assert error(full_attention64(layer, position, x, keys, values, planted)) > 1.5 * bound
    d = hip.upload_full_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    dk, dv = dev(keys), dev(values)
    out = torch.empty((len(x), HIDDEN), dtype=torch.float32, device="cuda")
    hip.full_attention_prefill(gpu, d, position, len(x), dev(x), out, dk, dv, len(keys))
    assert error(out.cpu().numpy()) <= bound


def test_linear_attention_prefill(gpu, oracle, tluts):
    rng = syn.rng_for(62, 0)
    layer = syn.linear_attention(rng, HIDDEN, tluts[1])
    d = hip.upload_linear_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    held = po.LinearAttentionStruct(layer)
    conv = np.zeros(8192 * 3, np.float32)
    rec = np.zeros(32 * 128 * 128, np.float32)
    dconv = torch.zeros(8192 * 3, dtype=torch.float32, device="cuda")
    drec = torch.zeros(32 * 128 * 128, dtype=torch.float32, device="cuda")
    for position, count in CHUNKS + [(77, 2)]:
        x = syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN))
        want = np.stack([po.linear_attention_forward(oracle, held, x[b], conv, rec, isa=16)
                         for b in range(count)])
        out = torch.empty((count, HIDDEN), dtype=torch.float32, device="cuda")
        hip.linear_attention_prefill(gpu, d, count, dev(x), out, dconv, drec)
        assert max_rel_error(out.cpu().numpy(), want) <= 1e-3, (position, count)
        close(dconv.cpu().numpy(), conv, "convolution state")
        close(drec.cpu().numpy(), rec, "recurrent state")


@pytest.mark.parametrize("count", [2, 3, 15, 16, 17, 33, 64, 1025])
def test_delta_chunk_edges(gpu, oracle, tluts, count):
    """The delta rule's chunk kernel at the edges of its sixteen-token stages
    and of its 1024-token launches, from a nonzero state: a dot of 128 products
    in another order differs by at most 128 * 2^-24 = 8e-6 of its magnitudes,
    and the decay keeps an error for a few tokens only, so 1e-4 of the largest
    value bounds outputs and state. The convolution state is the last three
    projected rows, shifted by as many blocks as the count leaves."""
    rng = syn.rng_for(65, count)
    layer = syn.linear_attention(rng, HIDDEN, tluts[1])
    d = hip.upload_linear_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    held = po.LinearAttentionStruct(layer)
    conv = rng.normal(0.0, 1.0, 8192 * 3).astype(np.float32)
    rec = rng.normal(0.0, 0.05, 32 * 128 * 128).astype(np.float32)
    dconv, drec = dev(conv), dev(rec)
    x = syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN))
    out = torch.empty((count, HIDDEN), dtype=torch.float32, device="cuda")
    hip.linear_attention_prefill(gpu, d, count, dev(x), out, dconv, drec)
    want = np.stack([po.linear_attention_forward(oracle, held, x[b], conv, rec, isa=16)
                     for b in range(count)])
    assert max_rel_error(out.cpu().numpy(), want) <= 1e-4
    assert np.max(np.abs(drec.cpu().numpy() - rec)) <= 1e-4 * np.max(np.abs(rec))
    assert np.max(np.abs(dconv.cpu().numpy() - conv)) <= 1e-4 * np.max(np.abs(conv))


@pytest.mark.parametrize("full", [False, True])
def test_prefill_layer(gpu, oracle, tluts, full):
    rng = syn.rng_for(63, int(full))
    etlut, ntlut = tluts
    layer = syn.decoder_layer(rng, full, HIDDEN, 64, 16, etlut, ntlut)
    d = hip.upload_decoder_layer(gpu, layer, gpu.expert_codebook(etlut), gpu.ne_codebook(ntlut))
    capacity = sum(c for _, c in CHUNKS)
    held = po.DecoderLayerStruct(layer, capacity=capacity)
    state, keep = hip.layer_state(full, capacity)
    for position, count in CHUNKS:
        h = syn.hidden_states(rng, count, HIDDEN)
        want = h.copy()
        for b in range(count):
            held.decode(oracle, position + b, want[b], isa=16)
        hidden = dev(h)
        hip.prefill_layer(gpu, d, position, count, hidden, state)
        assert max_rel_error(hidden.cpu().numpy(), want) <= 1e-3, (position, count)


def test_prefill_rejections(gpu, oracle, tluts):
    rng = syn.rng_for(64, 0)
    layer = syn.full_attention(rng, HIDDEN, tluts[1])
    d = hip.upload_full_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    x = torch.zeros((4, HIDDEN), dtype=torch.float32, device="cuda")
    out = torch.empty_like(x)
    cache = torch.zeros((5, 2, 256), dtype=torch.float32, device="cuda")
    with pytest.raises(hip.HipError, match="full attention state or input shape mismatch"):
        hip.full_attention_prefill(gpu, d, 2, 4, x, out, cache, cache.clone(), 5)  # 2 + 4 > 5
    with pytest.raises(hip.HipError, match="full attention state or input shape mismatch"):
        hip.full_attention_prefill(gpu, d, 0, 0, x, out, cache, cache.clone(), 5)
    torch.cuda.synchronize()


def test_chunk_rope_equals_single_tokens(gpu, tluts):
    """A chunk's keys are bit-identical with the keys of its tokens projected
    one at a time: the key projection runs each row in the same order at any
    batch below the MFMA path (8 rows), so the only difference could be the RoPE table,
    and the chunk's must be rope_table(position + b) itself (the reference
    builds its prefill table on the host, src/executor.cpp:1853-1866)."""
    rng = syn.rng_for(64, 0)
    layer = syn.full_attention(rng, HIDDEN, tluts[1])
    d = hip.upload_full_attention(gpu, layer, gpu.ne_codebook(tluts[1]))
    for position, count in ((0, 5), (1000, 7), (5000, 3)):
        capacity = position + count
        x = dev(syn.rms_normalized(syn.hidden_states(rng, count, HIDDEN)))
        chunk_keys = torch.zeros((capacity, 2, 256), dtype=torch.float32, device="cuda")
        chunk_values = torch.zeros_like(chunk_keys)
        out = torch.empty((count, HIDDEN), dtype=torch.float32, device="cuda")
        hip.full_attention_prefill(gpu, d, position, count, x, out, chunk_keys, chunk_values,
                                   capacity)
        one_keys = torch.zeros_like(chunk_keys)
        one_values = torch.zeros_like(chunk_keys)
        row = torch.empty(HIDDEN, dtype=torch.float32, device="cuda")
        for b in range(count):
            hip.full_attention_forward(gpu, d, position + b, x[b].contiguous(), row, one_keys,
                                       one_values, capacity)
        got = chunk_keys.cpu().numpy()[position:].view(np.uint32)
        want = one_keys.cpu().numpy()[position:].view(np.uint32)
        assert np.array_equal(got, want), (position, count)
