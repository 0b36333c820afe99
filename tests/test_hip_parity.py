"""HIP kernels vs the CPU oracle on the same seeded inputs (GPU).

Bars (from the north-star specification):
  * decoded levels and decoded fp16 weights: bit-exact with the reference
    decode (runtime.py:122-139, 291-301);
  * rotation: the fp32 transform matches the oracle's fp32 transform, so the
    fp16 result is compared bit-for-bit against fp16(oracle);
  * GEMV / forward: max-rel = max|y - y_ref| / max|y_ref| <= 2e-3 against
    the fp32/fp64-accumulated oracle (fp16 output).
"""

import zlib

import numpy as np
import pytest
import torch

from oracle import tcq_oracle as O
from turbopress_amd.synthetic import (
    QWEN3_0_6B_LAYER, make_activation, make_payload, payload_numpy, payload_to)

pytestmark = pytest.mark.gpu

GEMV_TOL = 2e-3


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ------------------------------------------------------------------ rotation
ROT_CASES = [(576, 64), (1536, 512), (1024, 1024), (3072, 1024), (128, 128),
             (2560, 512), (4096, 4096), (9728, 512), (2048, 2048), (96, 32), (8, 8)]


@pytest.mark.parametrize("d,block", ROT_CASES)
@pytest.mark.parametrize("batch", [1, 5])
def test_fwht_scale_matches_oracle(cuda, d, block, batch):
    from turbopress_amd.hip_kernel import fwht_scale
    gen = torch.Generator().manual_seed(7 + d + batch)
    rs = ((torch.randn(d, generator=gen).sign()) * (torch.rand(d, generator=gen) + 0.5)).to(torch.float16)
    x = (torch.randn(batch, d, generator=gen) * 3).to(torch.float16)
    got = fwht_scale(x.to(cuda), rs.to(cuda), block).cpu().numpy()
    ref32 = O.block_fwht(x.numpy().astype(np.float32) * rs.numpy().astype(np.float32), block)
    ref16 = ref32.astype(np.float16)
    assert got.shape == (batch, d)
    assert np.array_equal(got.view(np.uint16), ref16.view(np.uint16))


@pytest.mark.parametrize("rows,d,block,ldz", [
    (1, 4, 4, 8), (3, 4, 1, 4), (2, 1028, 4, 1280), (9, 1088, 64, 1280), (5, 6144, 2048, 6400), (7, 12288, 4096, 12288),
    (4099, 2560, 512, 2560), (4097, 96, 2, 256), (1500, 3072, 1024, 3328), (520, 4096, 4096, 4096),
    (2, 8192, 8192, 8448), (3, 1030, 2, 1280)])
@pytest.mark.parametrize("post", [False, True])
def test_rotated_rows_match_oracle(cuda, rows, d, block, ldz, post):
    """tp_block_fwht_rows (with and without scales before and after) and
    tp_fwht_scale_padded, one or several rows per wave, partial 1024- and
    4096-column segments, one block per four columns up to 4096 and beyond,
    rows of no multiple of 4: bit-exact with the oracle, zeros in the padding."""
    from turbopress_amd import _lib
    gen = torch.Generator().manual_seed(d + rows)
    rs = ((torch.randn(d, generator=gen).sign()) * (torch.rand(d, generator=gen) + 0.5)).to(torch.float16)
    x = (torch.randn(rows, d, generator=gen) * 3).to(torch.float16)
    xd, rd = x.to(cuda), rs.to(cuda)
    lib = _lib.lib()
    if post:
        out = torch.full((rows, d), float("nan"), dtype=torch.float16, device=cuda)
        st = lib.tp_block_fwht_rows(xd.data_ptr(), 0, rd.data_ptr(), out.data_ptr(), rows, d, block, _stream())
        ref = O.block_fwht(x.numpy().astype(np.float32), block) * rs.numpy().astype(np.float32)
    else:
        out = torch.full((rows, ldz), float("nan"), dtype=torch.float16, device=cuda)
        st = lib.tp_fwht_scale_padded(xd.data_ptr(), rd.data_ptr(), out.data_ptr(), rows, d, block, ldz, _stream())
        ref = np.zeros((rows, ldz), np.float32)
        ref[:, :d] = O.block_fwht(x.numpy().astype(np.float32) * rs.numpy().astype(np.float32), block)
    assert st == _lib.TP_OK
    assert np.array_equal(out.cpu().numpy().view(np.uint16), ref.astype(np.float16).view(np.uint16))


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 6])
@pytest.mark.parametrize("n,d,batch", [(1, 8, 1), (130, 1032, 4), (1500, 576, 16), (1500, 576, 17), (33, 3000, 7)])
def test_tiled_mode_matches_oracle(cuda, bits, n, d, batch):
    """mode "tiled" on both sides of its row bound (one GEMV launch / decoded
    row tiles), with bias, against the fp64 product of the exact weights
    codebook * scale and activations.  Each fp16 rounding is at most 2^-11 of
    its value: z and (row tiles) w once per term, the product and the sum with
    the bias once, so |y - ref| <= 2^-11 (4 sum |w z| + 2 |bias|), where the
    rotated z's own rounding is at most 2^-11 |z|."""
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(n, d, bits, 16, seed=n + d, bias=True)
    lin = PackedTCQLinear(p, mode="tiled", tile_rows=512)
    x = make_activation(batch, d, seed=batch)
    y = lin(x.to(cuda)).double().cpu().numpy()
    pn = payload_numpy(p)
    w = pn["codebook"].astype(np.float64)[O.levels_of(pn)] * pn["scales"].astype(np.float64)[:, None]
    rs = O.rot_scale(pn["signs_packed"], pn["inv_equil"], d).astype(np.float64)
    z = O.block_fwht(x.numpy().astype(np.float64) * rs, p["block"])
    ref = z @ w.T + pn["bias"].astype(np.float64)
    bound = 2.0 ** -11 * (4 * (np.abs(z) @ np.abs(w).T) + 2 * np.abs(pn["bias"].astype(np.float64)))
    assert np.all(np.abs(y - ref) <= bound)


@pytest.mark.parametrize("batch", [1, 16, 17])
def test_tiled_mode_refuses_row_tiles_of_zero_rows(cuda, batch):
    """tile_rows=0 raises on every forward, as the tile loop of
    runtime.py:326-331 does, whether or not the rows run through it."""
    from turbopress_amd.runtime import PackedTCQLinear
    lin = PackedTCQLinear(make_payload(48, 64, 3, 64, seed=1), mode="tiled", tile_rows=0)
    with pytest.raises(ValueError):
        lin(make_activation(batch, 64, seed=1).to(cuda))


def test_fwht_scale_rejects_bad_block(cuda):
    from turbopress_amd.hip_kernel import fwht_scale
    x = torch.zeros(1, 96, dtype=torch.float16, device=cuda)
    with pytest.raises(ValueError):
        fwht_scale(x, torch.ones(96, dtype=torch.float16, device=cuda), 64)


# -------------------------------------------------------------------- decode
DECODE_CASES = [(n, d, k, s) for s in (4, 8, 16, 64) for (n, d, k) in
                ((5, 77, 1), (9, 96, 2), (7, 102, 3), (3, 130, 4), (4, 64, 5), (2, 40, 7))]


@pytest.mark.parametrize("n,d,bits,n_states", DECODE_CASES)
def test_window_decode_levels_bit_exact(cuda, n, d, bits, n_states):
    from turbopress_amd.hip_kernel import window_decode_levels
    p = make_payload(n, d, bits, n_states, seed=n * d + bits)
    got = window_decode_levels(p["path_packed"].to(cuda),
                               None if p["member_packed"] is None else p["member_packed"].to(cuda),
                               d, bits, n_states).cpu().numpy()
    assert np.array_equal(got, O.levels_of(payload_numpy(p)))


@pytest.mark.parametrize("n,d,bits,n_states", [(33, 576, 2, 64), (17, 1024, 3, 64),
                                               (11, 2560, 4, 64), (9, 200, 3, 16)])
def test_decode_rows_bit_exact(cuda, n, d, bits, n_states):
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(n, d, bits, n_states, seed=3)
    lin = PackedTCQLinear(p, mode="hip")
    pn = payload_numpy(p)
    for r0, r1 in ((0, n), (3, 8), (n - 1, n)):
        got = lin.decode_rows(r0, r1).cpu().numpy()
        ref = O.decode_rows(pn, r0, r1)
        assert np.array_equal(got.view(np.uint16), ref.view(np.uint16)), (r0, r1)


@pytest.mark.parametrize("bits", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("n,d,n_states", [(1, 1, 64), (3, 7, 4), (2, 9, 64), (37, 63, 16), (5, 512, 64), (6, 520, 8),
                                          (4, 1031, 64), (70, 64, 64)])
def test_decode_natural_streams_at_every_rate(cuda, n, d, bits, n_states):
    """tp_decode_rows and tp_window_decode_levels, 8 columns per thread: rows
    ending inside a byte of either stream, one to several 512-column spans,
    wide and element stores (out strides of no multiple of 8), a row slice."""
    from turbopress_amd import _lib
    p = make_payload(n, d, bits, n_states, seed=n + d + bits)
    pn = payload_numpy(p)
    path = p["path_packed"].to(cuda)
    mem = None if p["member_packed"] is None else p["member_packed"].to(cuda)
    scales, cb = p["scales"].to(cuda), p["codebook"].to(cuda)
    mp, ms = (0, 0) if mem is None else (mem.data_ptr(), mem.stride(0))
    lib = _lib.lib()
    for stride in (d, (d + 7) // 8 * 8 + 8, d + 3):
        w = torch.full((n, stride), 7.0, dtype=torch.float16, device=cuda)
        lev = torch.full((n, stride), 255, dtype=torch.uint8, device=cuda)
        r0 = n // 2
        assert lib.tp_decode_rows(path[r0:].data_ptr(), path.stride(0), mp + r0 * ms, ms, scales[r0:].data_ptr(),
                                  cb.data_ptr(), n - r0, d, bits, n_states, w[r0:].data_ptr(), stride,
                                  _stream()) == _lib.TP_OK
        assert lib.tp_window_decode_levels(path.data_ptr(), path.stride(0), mp, ms, n, d, bits, n_states,
                                           lev.data_ptr(), stride, _stream()) == _lib.TP_OK
        assert np.array_equal(lev[:, :d].cpu().numpy(), O.levels_of(pn)) and bool((lev[:, d:] == 255).all())
        assert np.array_equal(w[r0:, :d].cpu().numpy().view(np.uint16), O.decode_rows(pn, r0, n).view(np.uint16))
        assert bool((w[:r0] == 7.0).all()) and bool((w[:, d:] == 7.0).all())


# ---------------------------------------------------------------------- GEMV
GEMV_CASES = [
    # (n, d, bits, n_states, batch)
    (1536, 576, 2, 64, 1),      # config 0: SmolLM2-135M up-proj
    (192, 256, 3, 64, 2),       # tests/test_runtime.py:164-174 shape
    (200, 96, 2, 8, 4),
    (130, 200, 4, 16, 3),
    (64, 128, 1, 4, 1),
    (96, 320, 5, 64, 9),
]
# the natural-stream GEMV's edges: 1, 4 and 8 rows at once and remainders, one
# wave per row and four, rows of no multiple of 8 columns, more columns than
# one span of four waves
GEMV_CASES += [(n, d, k, 64, b) for k in (1, 5, 6, 7) for n, d, b in
               ((1, 1, 1), (5, 515, 3), (66, 1032, 5), (7, 1100, 8), (3, 4104, 17), (4100, 1536, 2))]


@pytest.mark.parametrize("n,d,bits,n_states,batch", GEMV_CASES)
def test_packed_gemv_matches_fp64_oracle(cuda, n, d, bits, n_states, batch):
    from turbopress_amd.hip_kernel import packed_gemv
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(n, d, bits, n_states, seed=n + d)
    lin = PackedTCQLinear(p, mode="hip")
    z = (torch.randn(batch, d, generator=torch.Generator().manual_seed(1))).to(torch.float16)
    y = packed_gemv(z.to(cuda), lin).float().cpu().numpy()
    ref = O.gemv_fp64(payload_numpy(p), z.numpy().astype(np.float64))
    assert O.max_rel(y, ref) <= GEMV_TOL


@pytest.mark.parametrize("n,d,bits,batch", [(16, 64, 5, 33), (192, 256, 1, 199), (70, 1100, 7, 9), (5, 515, 6, 37),
                                            (33, 1032, 5, 2048), (300, 2056, 5, 44)])
def test_natural_streams_take_any_rows_in_one_launch(cuda, n, d, bits, batch):
    """packed_gemv of more than 8 rows at rates without a device layout: last
    groups of 1, 3, 4, 5 and 8 rows, every row against the fp64 product
    relative to the row's own largest value, one graph node, replays equal to
    the eager result."""
    import ctypes
    from turbopress_amd import _lib
    from turbopress_amd.hip_kernel import packed_gemv
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(n, d, bits, 64, seed=n + d)
    lin = PackedTCQLinear(p, mode="hip")
    z = torch.randn(batch, d, generator=torch.Generator().manual_seed(1)).to(torch.float16)
    zd = z.to(cuda)
    y = packed_gemv(zd, lin)
    ref = O.gemv_fp64(payload_numpy(p), z.numpy().astype(np.float64))
    err = np.abs(y.double().cpu().numpy() - ref).max(axis=1)
    assert np.all(err <= GEMV_TOL * np.abs(ref).max(axis=1))
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        out = packed_gemv(zd, lin)
    count = ctypes.c_size_t(0)
    assert _lib.lib().hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    assert count.value == 1
    graph.instantiate()
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, y)


@pytest.mark.parametrize("mode,bits", [("tiled", 2), ("tiled", 4), ("hip", 5), ("hip", 7)])
@pytest.mark.parametrize("d,batch", [(13, 1), (2051, 4), (1031, 8)])
def test_unused_infinite_levels_do_not_reach_the_output(cuda, mode, bits, d, batch):
    """The natural-stream GEMV over rows of no multiple of 8 columns: the
    stream bits past a row's end decode to levels 0..3, whose entries are
    infinite or NaN here and which no weight uses (every member code is at
    least 1); the products must match the fp64 ones of the weights alone."""
    from turbopress_amd.runtime import PackedTCQLinear
    n, mb = 5, bits - 1
    p = make_payload(n, d, bits, 64, seed=d)
    field = torch.zeros(n, (d * mb + 7) // 8 * 8, dtype=torch.uint8)
    field[:, :d * mb:mb] = 1  # member code 1 everywhere, zero bits after the row
    p["member_packed"] = (field.reshape(n, -1, 8) << torch.arange(8, dtype=torch.uint8)).sum(-1).to(torch.uint8)
    p["codebook"][:4] = torch.tensor([float("inf"), float("-inf"), float("nan"), float("inf")], dtype=torch.float16)
    lin = PackedTCQLinear(p, mode=mode)
    x = make_activation(batch, d, seed=batch)
    y = lin(x.to(cuda)).float().cpu().numpy()
    pn = payload_numpy(p)
    rs = O.rot_scale(pn["signs_packed"], pn["inv_equil"], d).astype(np.float32)
    z = O.block_fwht(x.numpy().astype(np.float32) * rs, p["block"]).astype(np.float16)
    assert O.max_rel(y, O.gemv_fp64(pn, z.astype(np.float64))) <= GEMV_TOL


@pytest.mark.parametrize("mode", ["hip", "triton", "tiled", "cached"])
@pytest.mark.parametrize("n,d,bits", [(1536, 576, 2), (256, 1024, 3), (72, 640, 4)])
def test_forward_modes_match_tiled_oracle(cuda, mode, n, d, bits):
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(n, d, bits, 64, seed=11, bias=True)
    lin = PackedTCQLinear(p, mode=mode, tile_rows=100)
    x = make_activation(2, d, seed=5)
    y = lin(x.to(cuda)).float().cpu().numpy()
    ref = O.tiled_forward(payload_numpy(p), x.numpy())
    assert y.shape == (2, n)
    assert O.max_rel(y, ref) <= GEMV_TOL, mode


@pytest.mark.parametrize("name", sorted(QWEN3_0_6B_LAYER))
def test_qwen3_0_6b_layer_linears(cuda, name):
    """Config 1: every Qwen3-0.6B projection at k=3, batch 1."""
    from turbopress_amd.runtime import PackedTCQLinear
    d, n = QWEN3_0_6B_LAYER[name]
    p = make_payload(n, d, 3, 64, seed=zlib.crc32(name.encode()) % 1000)
    lin = PackedTCQLinear(p, mode="hip")
    x = make_activation(1, d, seed=1)
    y = lin(x.to(cuda)).float().cpu().numpy()
    assert O.max_rel(y, O.tiled_forward(payload_numpy(p), x.numpy())) <= GEMV_TOL


def test_forward_errors_match_reference(cuda):
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(64, 128, 2, 8)
    lin = PackedTCQLinear(p, mode="hip")
    with pytest.raises(ValueError):
        lin(torch.randn(2, 64, device=cuda, dtype=torch.float16))
    with pytest.raises(RuntimeError):
        lin(torch.randn(2, 128, dtype=torch.float16))  # CPU input: no CPU path
    with pytest.raises(ValueError):
        PackedTCQLinear(p, mode="warp")
    with pytest.raises(ValueError):
        PackedTCQLinear({"format": 1})


@pytest.mark.parametrize("n,d,bits", [(9728, 2560, 3), (2560, 9728, 2), (100, 300, 4)])
def test_packed_bytes_exact(cuda, n, d, bits):
    """packed_bytes follows the reference's accounting (runtime.py:337-356)
    with the device layout in place of the (k+1)-bit level stream: exactly
    k bits per weight of the padded 16-row x 256-column tiles, plus the fp16
    side tensors; cached mode counts the fp16 weights."""
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(n, d, bits, 64, seed=5, bias=True)
    n_pad, d_pad = -(-n // 16) * 16, -(-d // 256) * 256
    side = 2 * (n + (1 << (bits + 1))) + 2 * n  # scales, codebook, bias
    signs = (d + 7) // 8
    hip = PackedTCQLinear(p, mode="hip")
    assert hip.tiled_packed.numel() == n_pad * d_pad * bits // 8
    assert hip.packed_bytes() == n_pad * d_pad * bits // 8 + signs + 2 * (2 * d) + side
    tiled = PackedTCQLinear(p, mode="tiled")
    natural = n * ((d + 7) // 8) + n * ((d * (bits - 1) + 7) // 8)
    assert tiled.packed_bytes() == natural + signs + 2 * (2 * d) + side
    if n * d <= 1 << 20:
        cached = PackedTCQLinear(p, mode="cached")
        assert cached.packed_bytes() == 2 * n * d + side


def test_packed_bytes_and_attributes(cuda):
    from turbopress_amd.runtime import PackedTCQLinear
    p = make_payload(256, 256, 2, 8)
    hip = PackedTCQLinear(p, mode="hip")
    cached = PackedTCQLinear(p, mode="cached")
    assert hip.levels_packed is not None and hip._w_cache is None
    assert cached.path_packed is None and cached._w_cache is not None
    assert hip.packed_bytes() < 2 * 256 * 256 / 6
    assert cached.packed_bytes() >= 2 * 256 * 256


@pytest.mark.gpu
def test_read_probe_runs_and_checks_arguments(cuda):
    """The streaming-read probe reads a buffer without writing it (its sink
    stays zero for an all-zero buffer) and rejects sizes that are not whole
    16-byte words."""
    from turbopress_amd import _lib
    lib = _lib.lib()
    buf = torch.zeros(1 << 20, dtype=torch.int32, device=cuda)
    sink = torch.zeros(1, dtype=torch.int32, device=cuda)
    stream = torch.cuda.current_stream(cuda).cuda_stream
    assert lib.tp_read_probe(buf.data_ptr(), buf.numel() * 4, sink.data_ptr(), stream) == 0
    torch.cuda.synchronize()
    assert int(sink.item()) == 0
    assert lib.tp_read_probe(buf.data_ptr(), 20, sink.data_ptr(), stream) != 0
