"""The product codec (ecf8_amd.huffman / utils / libecf8 host encoder and
validator) against the oracle and the golden vectors.  CPU only."""

from __future__ import annotations

import json
import os

import numpy as np
import pytest
import torch

from oracle import codec as oc

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")
CASES = sorted(json.load(open(os.path.join(GOLDEN, "index.json"))))


def _golden(name):
    return dict(np.load(os.path.join(GOLDEN, f"{name}.npz")))


def _random_counter(rng):
    k = int(rng.integers(1, 17))
    syms = sorted(rng.choice(16, k, replace=False).tolist())
    counts = (rng.pareto(0.3 + rng.random() * 3, k) * 500 + 1).astype(np.int64)
    if rng.random() < 0.3:  # many ties
        counts = rng.integers(1, 4, k)
    return {int(s): int(c) for s, c in zip(syms, counts)}


@pytest.mark.parametrize("seed", range(200))
def test_huffman_table_equals_restated_dahuffman(seed):
    from dfloat.huffman import HuffmanCodec

    counter = _random_counter(np.random.default_rng(seed))
    ours = HuffmanCodec.from_frequencies(counter).get_code_table()
    ref = oc.HuffmanTable.from_frequencies(counter).get_code_table()
    # same codes in the same listing order (the LUT row order depends on it)
    assert [(repr(k), v) for k, v in ours.items()] == [(repr(k), v) for k, v in ref.items()]


@pytest.mark.parametrize("seed", range(100))
def test_luts_equal_oracle(seed):
    from dfloat.utils import get_luts_from_huffman_table, get_nbit_codec

    counter = _random_counter(np.random.default_rng(1000 + seed))
    table = get_nbit_codec(counter, 16)[2]
    ref_table = oc.get_nbit_codec(counter, 16)[2]
    assert np.array_equal(get_luts_from_huffman_table(table).numpy(),
                          oc.get_luts_from_huffman_table(ref_table))


@pytest.mark.parametrize("name", CASES)
def test_product_compressor_reproduces_golden(name):
    from dfloat.compress import compress_flat

    g = _golden(name)
    tpb = int(g["threads_per_block"])
    flat = torch.from_numpy(g["flat"]).view(torch.float8_e4m3fn)
    res = compress_flat(flat, 8, tpb)
    for key in ("luts", "encoded", "packed_other_4bits", "output_positions", "gaps"):
        assert np.array_equal(res[key].numpy(), g[key]), key


@pytest.mark.parametrize("name", CASES)
def test_oracle_reproduces_golden(name):
    g = _golden(name)
    tpb = int(g["threads_per_block"])
    res = oc.compress_block(g["flat"], 8, tpb)
    assert np.array_equal(res["encoded"], g["encoded"])
    assert np.array_equal(res["output_positions"].view(np.uint8), g["output_positions"])
    out = oc.decode(g["luts"], g["encoded"], g["packed_other_4bits"], g["output_positions"],
                    g["gaps"], threads_per_block=tpb)
    assert np.array_equal(out, g["flat"])


@pytest.mark.parametrize("shape", [(4096, 4096), (1000, 2)])
def test_product_encoder_equals_c_oracle_at_size(shape, oracle_native):
    from dfloat.huffman import HuffmanCodec
    from ecf8_amd.synth import synthetic_fp8
    from dfloat.utils import encode_exponents_for_cuda, get_exponents_and_other_4bits_fp8_e4m3

    if shape == (1000, 2):
        w = torch.from_numpy(np.random.default_rng(0).integers(0, 256, 2000, dtype=np.uint8))
        w = w.view(torch.float8_e4m3fn)
    else:
        w = synthetic_fp8(*shape, 0.02, seed=0)[0].reshape(-1)
    exps, _ = get_exponents_and_other_4bits_fp8_e4m3(w.reshape(-1))
    vals, counts = torch.unique(exps, return_counts=True)
    counter = {int(v): int(c) for v, c in zip(vals.tolist(), counts.tolist())}
    codec = HuffmanCodec.from_frequencies(counter)
    enc, gaps, op = encode_exponents_for_cuda(exps, codec)
    ref_codec = oc.HuffmanTable.from_frequencies(counter)
    e2, g2, o2 = oracle_native.encode(exps.numpy(), ref_codec._table, ref_codec._eof)
    assert np.array_equal(enc.numpy(), e2)
    assert np.array_equal(gaps.numpy(), g2)
    assert np.array_equal(op.numpy(), o2)


# ------------------------------------------------------------- validator


def _valid_block():
    g = _golden("synth_128x256")
    return g


def _validate(g, **over):
    from ecf8_amd.decode import validate_format

    args = dict(luts=torch.from_numpy(g["luts"]), encoded_bytes=g["encoded"].size,
                packed_other_4bits_bytes=g["packed_other_4bits"].size,
                output_positions=torch.from_numpy(g["output_positions"]),
                gaps_bytes=g["gaps"].size)
    args.update(over)
    validate_format(**args)


def test_validator_accepts_golden_blocks():
    for name in CASES:
        g = _golden(name)
        _validate(g) if int(g["threads_per_block"]) == 512 else None


@pytest.mark.parametrize("fault", ["truncated_positions", "decreasing_positions", "last_not_n",
                                   "odd_packed", "bad_pointer", "too_many_luts", "gaps_size",
                                   "bad_entry", "first_not_zero"])
def test_validator_rejects_fault(fault):
    from ecf8_amd._lib import ECF8Error

    g = _valid_block()
    op = g["output_positions"].view(np.uint64).copy()
    luts = g["luts"].copy()
    over = {}
    if fault == "truncated_positions":
        over["output_positions"] = torch.from_numpy(op[:-1].view(np.uint8))
    elif fault == "decreasing_positions":
        op[1], op[2] = op[2], op[1]
        over["output_positions"] = torch.from_numpy(op.view(np.uint8))
    elif fault == "last_not_n":
        op[-1] -= 2
        over["output_positions"] = torch.from_numpy(op.view(np.uint8))
    elif fault == "first_not_zero":
        op[0] = 1
        over["output_positions"] = torch.from_numpy(op.view(np.uint8))
    elif fault == "odd_packed":
        over["packed_other_4bits_bytes"] = g["packed_other_4bits"].size - 1
    elif fault == "bad_pointer":
        luts[0, 5] = 256 - (luts.shape[0] - 1)  # points at the length row
        over["luts"] = torch.from_numpy(luts)
    elif fault == "too_many_luts":
        over["luts"] = torch.from_numpy(np.concatenate([luts] * 7))
    elif fault == "gaps_size":
        over["gaps_bytes"] = g["gaps"].size + 1
    elif fault == "bad_entry":
        luts[0, 7] = 100
        over["luts"] = torch.from_numpy(luts)
    with pytest.raises(ECF8Error):
        _validate(g, **over)


def test_encoder_rejects_symbol_without_code():
    from ecf8_amd._lib import ECF8Error
    from dfloat.huffman import HuffmanCodec
    from dfloat.utils import encode_exponents_for_cuda

    codec = HuffmanCodec.from_frequencies({3: 10, 4: 5})
    with pytest.raises(ECF8Error):
        encode_exponents_for_cuda(np.array([3, 4, 5], np.uint8), codec)


def test_product_length_limiter_equals_the_oracle_on_a_large_alphabet():
    """The product's limiter (dfloat/huffman.py, utils.py:249-265) never
    fires for 4-bit exponents: 16 symbols plus EOF are 17 leaves, so no code
    exceeds 16 bits.  It is generic over the alphabet, so it is checked on
    20 Fibonacci-weighted symbols (an unlimited tree 19 deep): same code
    table and same clamped counter as the oracle, longest code <= 16."""
    from dfloat.huffman import HuffmanCodec
    from dfloat.utils import get_nbit_codec

    counts = [1, 1]
    while len(counts) < 20:
        counts.append(counts[-1] + counts[-2])
    counter = {s: c for s, c in enumerate(counts)}
    unlimited = HuffmanCodec.from_frequencies(counter).get_code_table()
    assert max(b for b, _ in unlimited.values()) > 16
    codec, used, table = get_nbit_codec(counter, 16)
    _, ref_used, ref_table = oc.get_nbit_codec(counter, 16)
    assert max(b for b, _ in table.values()) <= 16
    assert {str(k): v for k, v in table.items()} == {str(k): v for k, v in ref_table.items()}
    assert dict(used) == dict(ref_used)
    assert codec.get_code_table() is table


def _huffman_codes(rng, kind):
    """(exponent distribution, code lengths, code values) of a prefix code."""
    from dfloat.huffman import get_nbit_codec

    p = {"flat": np.ones(16), "steep": 0.5 ** np.arange(16), "two": np.array([.9, .1] + [0] * 14),
         "fib": np.array([1, 1, 2, 3, 5, 8, 13, 21, 34, 55, 89, 144, 233, 377, 610, 987.])}[kind]
    p = p / p.sum()
    counter = {i: max(1, int(1e6 * v)) for i, v in enumerate(p) if v > 0}
    codec = get_nbit_codec(counter, max_n_bits=16)[0]
    bits, vals = np.zeros(16, np.uint8), np.zeros(16, np.uint32)
    for s, (b, v) in codec._table.items():
        if isinstance(s, (int, np.integer)):
            bits[s], vals[s] = b, v
    return p, bits, vals, *codec._table[codec._eof]


@pytest.mark.parametrize("kind", ["flat", "steep", "two", "fib"])
@pytest.mark.parametrize("bpt,tpb", [(8, 512), (8, 128), (2, 2), (3, 6), (64, 4096)])
def test_threaded_encoder_writes_the_same_bytes(kind, bpt, tpb):
    """Runs that start inside bytes, chunks and format-blocks, against the
    one-thread encoder, byte for byte with guard bytes past every output."""
    import ctypes

    from ecf8_amd._lib import lib

    L, rng = lib(), np.random.default_rng(bpt * 100 + tpb)
    p, bits, vals, eof_bits, eof_val = _huffman_codes(rng, kind)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    for n in (0, 1, 2, 65536 * 2 - 1, 65536 * 2, 65536 * 3 + 17, 65536 * 7 + 1):
        exps = rng.choice(16, n, p=p).astype(np.uint8)
        ref = [ctypes.c_int64() for _ in range(3)]
        assert L.ecf8_encoded_sizes(vp(exps), n, vp(bits), bpt, tpb, *map(ctypes.byref, ref)) == 0
        want = [np.zeros(ref[0].value, np.uint8), np.zeros(ref[1].value, np.uint8),
                np.zeros(ref[2].value, np.uint64)]
        assert L.ecf8_encode_exponents(vp(exps), n, vp(bits), vp(vals), eof_bits, eof_val, bpt, tpb,
                                       vp(want[0]), want[0].size, vp(want[1]), want[1].size,
                                       vp(want[2]), want[2].size) == 0
        for threads in (1, 2, 3, 7, 200):
            got = [ctypes.c_int64() for _ in range(3)]
            assert L.ecf8_encoded_sizes_threads(vp(exps), n, vp(bits), bpt, tpb, threads,
                                                *map(ctypes.byref, got)) == 0
            assert [g.value for g in got] == [r.value for r in ref]
            out = [np.full(w.size + 2, 0xA5, w.dtype) for w in want]
            assert L.ecf8_encode_exponents_threads(
                vp(exps), n, vp(bits), vp(vals), eof_bits, eof_val, bpt, tpb, threads, vp(out[0]),
                want[0].size, vp(out[1]), want[1].size, vp(out[2]), want[2].size) == 0
            for o, w in zip(out, want):
                assert np.array_equal(o[: w.size], w) and (o[w.size:] == 0xA5).all()
            if n > 65536 * 2 and threads > 1:  # refusals
                short = L.ecf8_encode_exponents_threads(
                    vp(exps), n, vp(bits), vp(vals), eof_bits, eof_val, bpt, tpb, threads,
                    vp(out[0]), want[0].size - 1, vp(out[1]), want[1].size, vp(out[2]),
                    want[2].size)
                assert short == 6
                bad = exps.copy()
                bad[n - 3] = 16
                assert L.ecf8_encode_exponents_threads(
                    vp(bad), n, vp(bits), vp(vals), eof_bits, eof_val, bpt, tpb, threads,
                    vp(out[0]), want[0].size, vp(out[1]), want[1].size, vp(out[2]),
                    want[2].size) == 4


@pytest.mark.parametrize("n", [2, 254, 131072, 131074, 400002])
def test_split_counts_and_nibbles(n):
    from dfloat.utils import get_exponents_and_other_4bits_fp8_e4m3, split_fp8_counted

    b = torch.from_numpy(np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8))
    w = b.view(torch.float8_e4m3fn)
    exps, packed, counts = split_fp8_counted(w)
    want_e, want_p = get_exponents_and_other_4bits_fp8_e4m3(w)
    assert torch.equal(exps, want_e) and torch.equal(packed, want_p)
    assert torch.equal(counts, torch.bincount(want_e, minlength=16))
    again = split_fp8_counted(b.repeat_interleave(2)[::2].view(torch.float8_e4m3fn))  # strided
    assert torch.equal(again[0], want_e) and torch.equal(again[1], want_p)


@pytest.mark.parametrize("n", [2, 400002])
def test_host_compression_under_another_default_device(n):
    """A host block compresses on the host, to the same tensors, where
    factory calls go to another device (meta has no memory to write to)."""
    from dfloat.compress import compress_flat

    b = np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8)
    w = torch.from_numpy(b).view(torch.float8_e4m3fn)
    want = compress_flat(w)
    with torch.device("meta"):
        got = compress_flat(w)
    for key in ("luts", "encoded", "packed_other_4bits", "output_positions", "gaps"):
        assert got[key].device.type == "cpu" and torch.equal(got[key], want[key]), key


@pytest.mark.parametrize("threads", [1, 2, 3, 16, 200])
def test_split_on_any_number_of_threads(threads):
    """Parts that divide the block evenly and not: the one-thread outputs."""
    from ecf8_amd._lib import lib

    for n in (2, 262142, 262146, 400002):
        w = torch.from_numpy(np.random.default_rng(n).integers(0, 256, n, dtype=np.uint8))
        got = []
        for t in (1, threads):
            out = (torch.full((n,), 99, dtype=torch.uint8), torch.zeros(n // 2, dtype=torch.uint8),
                   torch.full((16,), -1, dtype=torch.int64))
            assert lib().ecf8_split_fp8(w.data_ptr(), n, *(o.data_ptr() for o in out), t) == 0
            got.append(out)
        assert all(torch.equal(a, b) for a, b in zip(*got))


def test_small_blocks_compress_on_one_thread(monkeypatch):
    """Few weights on one thread, whatever torch has; many on torch's count,
    at most 16."""
    from dfloat import utils

    monkeypatch.setattr(torch, "get_num_threads", lambda: 64)
    got = [utils.host_threads(n) for n in (0, 2, 1 << 20, (5 << 19) - 1, 5 << 19, 1 << 24)]
    assert got == [1, 1, 1, 1, 10, 16]
    monkeypatch.setattr(torch, "get_num_threads", lambda: 3)
    assert utils.host_threads(1 << 24) == 3
