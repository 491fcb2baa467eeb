"""GPU parity of the decoder layer around the W8A16 GEMM (qtts/models/talker.py:246-271), through the C ABI.

* ``qtts_rms_norm`` against the fp64 oracle (qtts/layers/norm.py:50-76): every element
  within one unit in the last place, at most one in a hundred not the oracle's value
  rounded; and against torch-CPU's eager RMSNorm fixtures within one unit (the bound
  the reference's own tests/test_norm.py:56-72 sets between its fused and eager paths).
* ``qtts_w8a16_fused_gemm_strips`` with the RMSNorm prologue against the oracle's GEMM of
  the oracle's normalized rows (W8A16 tolerance: |y - ref| <= 1e-2 RMS + half an ulp),
  and, where the norm runs as its own pass, bit for bit against qtts_rms_norm followed
  by qtts_w8a16_gemm_strips.
* The residual epilogue against torch's ``residual + linear(x)`` on this library's own
  GEMM output, bit for bit, fused (up to 8 rows) or not, in place or not; with the
  SiLU prologue as well (the down projection).
"""

from __future__ import annotations

import os

import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_gemm import PREDICTOR, TALKER, assert_close

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
NORMED = [TALKER[0], TALKER[2], PREDICTOR[0], PREDICTOR[2], (100, 512)]  # qkv and gate_up
RESIDUAL = [TALKER[1], TALKER[3], PREDICTOR[1], PREDICTOR[3], (48, 512)]  # o_proj and down
_TD = {torch.bfloat16: O.DT_BF16, torch.float16: O.DT_F16, torch.float32: O.DT_F32}


@pytest.fixture(scope="module")
def ops():
    from qtts_amd import ops as _ops
    assert _ops.device_supported(), "GPU is not a gfx950"
    _ops.reserve_workspace(torch.device("cuda"), 64 << 20)
    return _ops


def _bits(t: torch.Tensor) -> np.ndarray:
    t = t.contiguous().cpu()
    if t.dtype == torch.float32:
        return t.numpy()
    return t.view(torch.int16).numpy().view(np.uint16)


def _ulp(v: np.ndarray, dtype: torch.dtype) -> np.ndarray:
    mant = {torch.bfloat16: 7, torch.float16: 10, torch.float32: 23}[dtype]
    lo = {torch.bfloat16: -126, torch.float16: -14, torch.float32: -126}[dtype]
    e = np.maximum(np.floor(np.log2(np.maximum(np.abs(v), 1e-38))), lo)
    return 2.0 ** (e - mant)


def _round(v: np.ndarray, dtype: torch.dtype) -> torch.Tensor:
    return torch.from_numpy(np.ascontiguousarray(v, np.float64)).to(dtype)


def _weights(ops, n, k, dtype, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.02).to(dtype)
    q, s = ops.pack_int8(w, dtype)
    return q, s, ops.to_strips(q)


def _oracle_gemm(h: torch.Tensor, q, s, b):
    return O.w8a16_ref(h.float().cpu().numpy(), q.cpu().numpy(), s.float().cpu().numpy(),
                       None if b is None else b.float().cpu().numpy())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rms_norm_vs_oracle(ops, dtype):
    for m, k in ((1, 2048), (5, 1024), (3, 512), (4, 100), (2, 6144), (9, 8)):
        g = torch.Generator(device="cuda").manual_seed(m * 31 + k)
        x = (torch.randn(m, k, device="cuda", generator=g) * 2).to(dtype)
        x[0, : k // 4] *= 30.0
        w = (1 + 0.2 * torch.randn(k, device="cuda", generator=g)).to(dtype)
        y = ops.rms_norm(x, w, 1e-6)
        ref = O.rms_norm(_bits(x), _bits(w), 1e-6, _TD[dtype])
        got = y.double().cpu().numpy()
        units = 4 if dtype == torch.float32 else 1  # fp32: the roundings of inv and two products
        assert np.all(np.abs(got - ref) <= units * _ulp(ref, dtype)), f"{dtype} m={m} k={k}"
        if dtype != torch.float32:
            off = int((y.cpu() != _round(ref, dtype)).sum())
            assert off <= max(1, y.numel() // 100), f"{dtype} m={m} k={k}: {off} elements not rounded"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k", [8, 504, 512, 520, 1024, 1032, 2048, 2056, 4096, 4104, 8192, 8200])
def test_rms_norm_row_lengths(ops, dtype, k):
    """Every vector-count branch of the row kernel and the lengths around it, strided rows included, held to
    the bound of test_rms_norm_vs_oracle."""
    g = torch.Generator(device="cuda").manual_seed(k)
    x = (torch.randn(5, k + 8, device="cuda", generator=g) * 2).to(dtype)[:, :k]
    w = (1 + 0.2 * torch.randn(k, device="cuda", generator=g)).to(dtype)
    y = ops.rms_norm(x, w, 1e-6)
    ref = O.rms_norm(_bits(x), _bits(w), 1e-6, _TD[dtype])
    want = _round(ref, dtype).double().numpy()
    err = np.abs(y.double().cpu().numpy() - want)
    assert (err <= _ulp(want, dtype)).all()
    assert int((err > 0).sum()) <= max(1, y.numel() // 100)


@pytest.mark.parametrize("m,k", [(3, 8200), (5, 16384), (2, 65536), ((1 << 22) + 3, 8)])
def test_rms_norm_past_the_register_kernel(ops, m, k):
    """Longer rows and more of them than the register kernel takes: within one unit of the value in 64 bits."""
    g = torch.Generator(device="cuda").manual_seed(k)
    x = (torch.randn(m, k, device="cuda", generator=g) * 2).to(torch.bfloat16)
    w = (1 + 0.2 * torch.randn(k, device="cuda", generator=g)).to(torch.bfloat16)
    y = ops.rms_norm(x, w, 1e-6)
    for rows in (slice(0, 4096), slice(max(0, m - 4096), m)):
        xd = x[rows].double()
        want = (xd * torch.rsqrt(xd.square().mean(1, keepdim=True) + 1e-6) * w.double()).cpu().numpy()
        assert (np.abs(y[rows].double().cpu().numpy() - want) <= _ulp(want, torch.bfloat16)).all()


def test_rms_norm_golden(ops):
    z = np.load(os.path.join(GOLDEN, "rms_norm.npz"))
    eps = float(z["eps"])
    for dt, tdt in (("bf16", torch.bfloat16), ("f16", torch.float16)):
        for width in (2048, 1024, 512):
            x = torch.from_numpy(z[f"{dt}.{width}.x"].view(np.int16)).view(tdt).cuda()
            w = torch.from_numpy(z[f"{dt}.{width}.w"].view(np.int16)).view(tdt).cuda()
            want = torch.from_numpy(z[f"{dt}.{width}.y"].view(np.int16)).view(tdt)
            y = ops.rms_norm(x, w, eps).cpu()
            diff = (y.double() - want.double()).abs().numpy()
            assert np.all(diff <= _ulp(want.double().numpy(), tdt)), f"{dt} width={width}"


@pytest.mark.parametrize("n,k", NORMED)
def test_norm_prologue(ops, n, k):
    from qtts_amd.ops import PRO_RMS_NORM
    for dtype in (torch.bfloat16, torch.float16):
        q, s, qs = _weights(ops, n, k, dtype, seed=n + k)
        for m in (1, 2, 3, 5, 8, 9, 12, 16):  # 9-16: fused in two row parts of 8
            g = torch.Generator(device="cuda").manual_seed(m + 5 * k)
            x = (torch.randn(m, k, device="cuda", generator=g) * 3).to(dtype)
            nw = (1 + 0.1 * torch.randn(k, device="cuda", generator=g)).to(dtype)
            b = (torch.randn(n, device="cuda", generator=g) * 0.1).to(dtype) if m != 2 else None
            h_ref = _round(O.rms_norm(_bits(x), _bits(nw), 1e-6, _TD[dtype]), dtype)
            ref = _oracle_gemm(h_ref, q, s, b)
            h = ops.rms_norm(x, nw, 1e-6)
            for algo in (0, ops.algo_code(1, 0, 4, 8), ops.algo_code(1, 0, 2, 8), ops.algo_code(1, 2, 8, 8),
                         ops.algo_code(1, 0, 16, 6)):
                what = f"{dtype} n={n} k={k} m={m} algo={algo:#x}"
                y = ops.w8a16_fused_gemm_strips(x, qs, n, s, b, prologue=PRO_RMS_NORM, norm_weight=nw, algo=algo)
                assert_close(y, ref, what)
                plain = ops.w8a16_gemm_strips(h, qs, n, s, b, algo)
                if ((algo >> 8) & 0xFF) > 1:  # split K: the norm runs as its own pass
                    assert torch.equal(y, plain), what
                else:  # up to 16 rows: fused, its sums in another order
                    assert_close(y, _oracle_gemm(h, q, s, b), what + " vs separate norm")


@pytest.mark.parametrize("n,k", RESIDUAL)
def test_residual_epilogue(ops, n, k):
    for dtype in (torch.bfloat16, torch.float16):
        q, s, qs = _weights(ops, n, k, dtype, seed=3 * n + k)
        for m in (1, 2, 3, 5, 8, 12, 16, 24, 40):  # past 16: half strips in row parts, else the separate add
            g = torch.Generator(device="cuda").manual_seed(m + n)
            x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
            r = (torch.randn(m, n, device="cuda", generator=g) * 4).to(dtype)
            b = (torch.randn(n, device="cuda", generator=g) * 0.1).to(dtype) if m % 2 else None
            half = ops.algo_code(ops.ALGO_SKINNY_HALF)
            for algo in (0, ops.algo_code(1, 0, 4, 8), ops.algo_code(1, 3, 2, 8), ops.algo_code(1, 0, 8, 12), half):
                if m > 16 and algo not in (0, half):
                    continue  # past 16 rows: the automatic choice and half strips in row parts
                if algo == ops.algo_code(1, 0, 8, 12) and m > 8 and n > 2048:
                    continue  # 8 waves of 12 chunks: staged rows only (9-16 rows: on at most 128 strips)
                what = f"{dtype} n={n} k={k} m={m} algo={algo:#x}"
                lin = ops.w8a16_gemm_strips(x, qs, n, s, b, algo)
                want = r + lin
                y = ops.w8a16_fused_gemm_strips(x, qs, n, s, b, residual=r, algo=algo)
                assert torch.equal(y, want), what
                hidden = r.clone()
                out = ops.w8a16_fused_gemm_strips(x, qs, n, s, b, residual=hidden, out=hidden, algo=algo)
                assert out is hidden and torch.equal(hidden, want), what + " in place"
            assert_close(lin, _oracle_gemm(x, q, s, b), f"{dtype} n={n} k={k} m={m} vs oracle")


@pytest.mark.parametrize("n,k", [TALKER[3], PREDICTOR[3], (48, 512)])
def test_silu_and_residual(ops, n, k):
    from qtts_amd.ops import PRO_SILU_MUL
    for dtype in (torch.bfloat16, torch.float16):
        _, s, qs = _weights(ops, n, k, dtype, seed=n * k)
        f32 = s.float()
        for m in (1, 2, 3):
            g = torch.Generator(device="cuda").manual_seed(11 * m + k)
            gu = (torch.randn(m, 2 * k, device="cuda", generator=g) * 3).to(dtype)
            r = torch.randn(m, n, device="cuda", generator=g).to(dtype)
            for scale in (s, f32):
                for algo in (0, ops.algo_code(1, 0, 16, 6), ops.algo_code(1, 2, 4, 8),
                             ops.algo_code(ops.ALGO_SKINNY_HALF)):
                    what = f"{dtype} n={n} k={k} m={m} algo={algo:#x} scale {scale.dtype}"
                    want = r + ops.w8a16_silu_mul_gemm_strips(gu, qs, n, scale, None, algo)
                    y = ops.w8a16_fused_gemm_strips(gu, qs, n, scale, prologue=PRO_SILU_MUL, residual=r, algo=algo)
                    assert torch.equal(y, want), what


def test_fused_graph_replays(ops):
    """The norm prologue (a workgroup barrier over per-wave sums) and the residual epilogue
    under graph capture: every replay equals the eager result, with other calls between."""
    from qtts_amd.ops import PRO_RMS_NORM
    n, k = 12288, 2048
    _, s, qs = _weights(ops, n, k, torch.bfloat16, seed=1)
    x = torch.randn(1, k, device="cuda").to(torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(k, device="cuda")).to(torch.bfloat16)
    r = torch.randn(1, n, device="cuda").to(torch.bfloat16)

    def call(xx):
        return ops.w8a16_fused_gemm_strips(xx, qs, n, s, prologue=PRO_RMS_NORM, norm_weight=nw, residual=None), \
            ops.w8a16_fused_gemm_strips(xx, qs, n, s, residual=r[:, :n])

    eager = call(x)
    static = x.clone()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        call(static)
    torch.cuda.current_stream().wait_stream(st)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call(static)
    for i in range(4):
        other = call(torch.randn(1, k, device="cuda").to(torch.bfloat16))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out[0], eager[0]) and torch.equal(out[1], eager[1]), f"replay {i}"
        assert other[0].shape == (1, n)


def test_fused_errors(ops):
    from qtts_amd import _lib
    n, k = 64, 128
    _, s, qs = _weights(ops, n, k, torch.bfloat16, seed=2)
    x = torch.randn(2, k, device="cuda").to(torch.bfloat16)
    with pytest.raises(ValueError, match="norm weight"):
        ops.w8a16_fused_gemm_strips(x, qs, n, s, prologue=ops.PRO_RMS_NORM)
    with pytest.raises(ValueError, match="residual"):
        ops.w8a16_fused_gemm_strips(x, qs, n, s, residual=torch.zeros(2, n + 1, device="cuda", dtype=torch.bfloat16))
    buf = torch.zeros(2 * n + 8, device="cuda", dtype=torch.bfloat16)
    st = _lib.load().qtts_w8a16_fused_gemm_strips(
        x.data_ptr(), _lib.BF16, 2, k, k, 0, None, 0.0, qs.data_ptr(), n, s.data_ptr(), _lib.BF16, None,
        buf[8:].data_ptr(), n, buf.data_ptr(), n, 0, None, 0, None)
    assert st != 0 and "overlaps" in _lib.last_error()
    st = _lib.load().qtts_w8a16_fused_gemm_strips(
        x.data_ptr(), _lib.BF16, 2, k, k, 7, None, 0.0, qs.data_ptr(), n, s.data_ptr(), _lib.BF16, None,
        None, 0, buf.data_ptr(), n, 0, None, 0, None)
    assert st != 0 and "prologue" in _lib.last_error()


@pytest.mark.parametrize("m,n,k", [(8, 2048, 2048), (16, 1024, 3072), (17, 2048, 2048), (40, 2048, 2048), (41, 2048, 2048),
                                   (64, 1024, 2048), (65, 1024, 2048)])
def test_residual_without_a_workspace(ops, m, n, k):
    """A residual call that the decode kernels' half strips cover (up to 64 rows, their weight reads within 20 MiB) runs
    without a workspace and gives the bits it gives with one, whichever kernel the automatic choice takes; past
    them the call is refused."""
    from qtts_amd import _lib
    q, s, qs = _weights(ops, n, k, torch.bfloat16, 9)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, device="cuda", generator=g).to(torch.bfloat16)
    res = torch.randn(m, n, device="cuda", generator=g).to(torch.bfloat16)
    y = torch.empty_like(res)
    st = _lib.load().qtts_w8a16_fused_gemm_strips(
        x.data_ptr(), _lib.BF16, m, k, k, ops.PRO_NONE, None, 0.0, qs.data_ptr(), n, s.data_ptr(), _lib.BF16, None,
        res.data_ptr(), n, y.data_ptr(), n, 0, None, 0, torch.cuda.current_stream().cuda_stream)
    if m <= 16 or (m <= 64 and (m + 7) // 8 * n * k <= 20 << 20):
        assert st == 0, _lib.last_error()
        assert torch.equal(y, ops.w8a16_fused_gemm_strips(x, qs, n, s, residual=res))
    else:
        assert st != 0 and "workspace" in _lib.last_error()


@pytest.mark.parametrize("m,n,k", [(12, 512, 4096), (12, 512, 6144), (17, 512, 2048)])
def test_gate_up_without_a_workspace(ops, m, n, k):
    """gate_up with its activation needs no workspace where the decode kernel's pairs are built (16 rows, K <= 4096);
    elsewhere a call that comes without is refused, whichever kernel would run it."""
    from qtts_amd import _lib
    q, s, qs = _weights(ops, n, k, torch.bfloat16, 9)
    x = torch.randn(m, k, device="cuda").to(torch.bfloat16)
    act = torch.empty(m, n // 2, device="cuda", dtype=torch.bfloat16)
    st = _lib.load().qtts_w8a16_gate_up_silu_strips(
        x.data_ptr(), _lib.BF16, m, k, k, ops.PRO_NONE, None, 0.0, qs.data_ptr(), n, s.data_ptr(), _lib.BF16, None,
        act.data_ptr(), n // 2, 0, None, 0, torch.cuda.current_stream().cuda_stream)
    if m <= 16 and k <= 4096:
        assert st == 0, _lib.last_error()
        assert torch.equal(act, ops.w8a16_gate_up_silu_strips(x, qs, n, s))
    else:
        assert st != 0 and "workspace" in _lib.last_error()


# (m, n, k): tiles of 32 x 64 with one and two chunks a stage, whole and split K, ragged rows and
# columns; then each 8-wave tile of the automatic choice.
TILE_EPILOGUES = [(65, 100, 192), (17, 4128, 64), (70, 2048, 6144), (129, 1056, 1024), (1003, 2048, 128),
                  (1003, 4096, 64), (1000, 6400, 64), (1003, 12288, 64)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", TILE_EPILOGUES)
def test_tile_residual_epilogue(ops, m, n, k, dtype):
    """Past the decode rows the residual rides in the tile kernel's epilogue: bit for bit torch's
    ``residual + linear(x)`` on the plain GEMM, in place and with a row stride of its own."""
    q, s, qs = _weights(ops, n, k, dtype, 3)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    b = torch.randn(n, device="cuda", generator=g).to(dtype)
    for pad in (0, 3):  # 3: rows that are not 8-byte aligned
        res = torch.randn(m, n + pad, device="cuda", generator=g).to(dtype)[:, :n]
        for bias in (None, b):
            want = res + ops.w8a16_gemm_strips(x, qs, n, s, bias)
            assert torch.equal(ops.w8a16_fused_gemm_strips(x, qs, n, s, bias, residual=res), want)
    same = res.clone()
    ops.w8a16_fused_gemm_strips(x, qs, n, s, b, residual=same, out=same)
    assert torch.equal(same, want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", [(m, n // 32 * 32, k) for m, n, k in TILE_EPILOGUES])
def test_tile_silu_pair_epilogue(ops, m, n, k, dtype):
    """GatedMLP's activation in the tile kernel's epilogue: bit for bit silu_mul of the plain tile
    GEMM, after a plain input or a separate RMSNorm."""
    from qtts_amd import _lib
    q, s, qs = _weights(ops, n, k, dtype, 4)
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    nw = (1 + 0.1 * torch.randn(k, device="cuda", generator=g)).to(dtype)
    for bias in (None, torch.randn(n, device="cuda", generator=g).to(dtype)):
        for norm in (False, True):
            h = ops.rms_norm(x, nw) if norm else x
            # the automatic tile at every row count (the plain automatic choice keeps small weights on the skinny kernel)
            want = ops.silu_mul(ops.w8a16_gemm_strips(h, qs, n, s, bias, _lib.algo_code(_lib.ALGO_TILE)))
            kw = {"prologue": ops.PRO_RMS_NORM, "norm_weight": nw} if norm else {}
            assert torch.equal(ops.w8a16_gate_up_silu_strips(x, qs, n, s, bias, **kw), want)


# (m, n, k): row edges of the 16-row blocks (with 5 to 8 rows for the norm inside), ragged columns, each built K
WIDE = [(5, 4096, 1024), (6, 4096, 1024), (7, 6144, 1024), (8, 1024, 1024), (9, 4096, 1024), (16, 100, 1024), (17, 6144, 1024), (33, 4096, 1024), (48, 1040, 1024),
        (65, 6144, 1024), (96, 6144, 1024), (128, 6144, 1024), (9, 12288, 2048), (31, 12288, 2048), (47, 4096, 2048),
        (128, 4096, 2048), (27, 2048, 2048), (127, 2048, 2048), (12, 1000, 3072), (97, 1024, 3072), (13, 2048, 6144),
        (32, 2048, 6144), (64, 2048, 6144)]
# K between the tiles' full runs: waves whose runs differ by one chunk, each group of tiles at the ends of its range of K
WIDE_K = [(5, 4096, 640), (9, 1040, 576), (16, 4096, 960), (48, 1000, 704), (17, 6144, 1088), (33, 2048, 1088), (64, 1040, 1984),
          (128, 4096, 1984), (9, 4096, 2112), (27, 1000, 2624), (97, 1024, 3008), (12, 4096, 3136), (32, 2048, 5120), (64, 2048, 6080),
          (27, 12288, 1536),
          # grids whose row blocks are not a multiple of 8 columns apart; few strips of odd chunks, on the decode kernel
          (39, 5408, 1536), (90, 1312, 6144), (100, 1056, 3072), (16, 544, 3136), (9, 224, 1984)]


def _ref64(h, q, s, b):
    """The dequantize-then-matmul of the packed codes in float64 (torch on the GPU: the oracle's formula, faster)."""
    y = h.double() @ (q.double() * s.double()[:, None]).t()
    return (y if b is None else y + b.double()).cpu().numpy()


def _bar_product(y, gate, up, what, dtype):
    """The GEMM bar carried through silu(g) * u to first order: |d silu| <= 1.1 |dg|, half an output ulp each for the
    roundings of g, u and silu(g) in between (dtype's ulp: 7 fraction bits, or 10 down to 2^-24)."""
    def half(v):
        e = np.floor(np.log2(np.maximum(np.abs(v), 1e-30)))
        return 2.0 ** (e - 7 if dtype == torch.bfloat16 else np.maximum(e, -14) - 10) / 2
    rms_g, rms_u = (np.sqrt(np.mean(v * v)) for v in (gate, up))
    silu = gate / (1 + np.exp(-gate))
    dg, du = 1e-2 * rms_g + half(gate), 1e-2 * rms_u + half(up)
    bound = (1.1 * dg + half(silu)) * np.abs(up) + np.abs(silu) * du + 1.1 * dg * du + half(silu * up)
    err = np.abs(y - silu * up)
    assert (err <= bound).all(), f"{what}: {err.max()} {int((err > bound).sum())}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", WIDE + WIDE_K)
def test_wide_calls(ops, m, n, k, dtype):
    """The automatic choice at 9-128 rows (the one-round tiles): every form against float64, the
    residual bit for bit the plain call's, strided rows, and rows that do not meet (a row of infinities and
    one of NaN leave the others' bits alone)."""
    q, s, qs = _weights(ops, n, k, dtype, 5)
    g = torch.Generator(device="cuda").manual_seed(m * 7 + k)
    x = torch.randn(m, k + 8, device="cuda", generator=g).to(dtype)[:, :k]
    b = torch.randn(n, device="cuda", generator=g).to(dtype)
    nw = (1 + 0.1 * torch.randn(k, device="cuda", generator=g)).to(dtype)
    what = f"wide m={m} n={n} k={k} {dtype}"
    y = ops.w8a16_gemm_strips(x, qs, n, s, b)
    assert_close(y, _ref64(x, q, s, b), what)
    res = torch.randn(m, n + 3, device="cuda", generator=g).to(dtype)[:, :n]
    assert torch.equal(ops.w8a16_fused_gemm_strips(x, qs, n, s, b, residual=res), res + y), what
    hn = _round(O.rms_norm(_bits(x.contiguous()), _bits(nw), 1e-6, _TD[dtype]), dtype).cuda()
    yn = ops.w8a16_fused_gemm_strips(x, qs, n, s, None, prologue=ops.PRO_RMS_NORM, norm_weight=nw)
    assert_close(yn, _ref64(hn, q, s, None), what + " norm")
    odd = x.clone()
    odd[0], odd[m // 2] = float("inf"), float("nan")
    rest = [i for i in range(m) if i not in (0, m // 2)]
    assert torch.equal(ops.w8a16_gemm_strips(odd, qs, n, s, b)[rest], y[rest]), what
    if n % 32 == 0:
        for h, kw in ((x, {}), (hn, {"prologue": ops.PRO_RMS_NORM, "norm_weight": nw})):
            full = _ref64(h, q, s, b)
            act = ops.w8a16_gate_up_silu_strips(x, qs, n, s, b, **kw)
            _bar_product(act.double().cpu().numpy(), full[:, : n // 2], full[:, n // 2:], what + str(list(kw)), dtype)


# (m, n, k): the plain (or norm) call and the one with the activation take the same waves over the same K
@pytest.mark.parametrize("norm,m,n,k", [(False, 33, 4096, 1024), (False, 48, 1024, 704), (False, 31, 12288, 2048), (False, 27, 12288, 1536),
                                        (False, 17, 6144, 1088), (False, 33, 2048, 2048), (False, 17, 2048, 3072), (False, 32, 2048, 6144),
                                        (True, 5, 4096, 1024), (True, 8, 4096, 960), (True, 33, 4096, 1024), (True, 64, 6144, 1024),
                                        (True, 12, 4096, 2048), (True, 31, 4096, 1984)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("sdt", [None, torch.float32])
def test_wide_silu_pair_bits(ops, norm, m, n, k, dtype, sdt):
    """The wide kernel's activation: bit for bit silu_mul of its call without it (gate, up and silu(gate) each rounded once)."""
    q, s, qs = _weights(ops, n, k, dtype, 7)
    s = s if sdt is None else (s.float() * (1 + 2.0 ** -13)).to(sdt)
    g = torch.Generator(device="cuda").manual_seed(m * 3 + k)
    x = torch.randn(m, k, device="cuda", generator=g).to(dtype)
    kw = {"prologue": ops.PRO_RMS_NORM, "norm_weight": (1 + 0.1 * torch.randn(k, device="cuda", generator=g)).to(dtype)} if norm else {}
    for bias in (None, torch.randn(n, device="cuda", generator=g).to(dtype)):
        full = ops.w8a16_fused_gemm_strips(x, qs, n, s, bias, **kw) if norm else ops.w8a16_gemm_strips(x, qs, n, s, bias)
        assert torch.equal(ops.w8a16_gate_up_silu_strips(x, qs, n, s, bias, **kw), ops.silu_mul(full)), (m, n, k, dtype)


@pytest.mark.parametrize("m,n,k", [(9, 4096, 1024), (33, 6144, 1024), (47, 4096, 2048), (97, 1024, 3072), (64, 2048, 6144)] + WIDE_K)
def test_wide_fp8_codes(ops, m, n, k):
    """The same kernel on e4m3 codes: against float64."""
    g = torch.Generator(device="cuda").manual_seed(m + n)
    w = (torch.randn(n, k, device="cuda", generator=g) * 0.02).to(torch.bfloat16)
    q, s = ops.pack_fp8(w)
    x = torch.randn(m, k, device="cuda", generator=g).to(torch.bfloat16)
    assert_close(ops.fp8w_gemm_strips(x, ops.fp8w_strips(q), n, s), _ref64(x, q.float(), s, None), f"wide fp8 {m} {n} {k}")


# (m, n, k) of the half strips: idle waves (K / 128 below the waves), runs that differ by one, whole ones; ragged rows and columns;
# more rows of fewer strips, to the last row part that one round holds
HALF = [(5, 200, 640), (8, 2048, 768), (7, 1000, 1152), (16, 1024, 1920), (8, 2040, 2048), (12, 1000, 2176), (16, 1024, 3072),
        (13, 1000, 5120), (8, 2048, 6016), (5, 2048, 6144), (17, 512, 640), (31, 500, 2048), (72, 200, 1024), (65, 195, 3072),
        (256, 64, 1920), (1024, 16, 2048), (1001, 9, 6144)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,n,k", HALF)
def test_wide_half_strips(ops, m, n, k, dtype):
    """The half strips' automatic calls: against float64 on int8 and e4m3 codes, the residual bit for bit the plain call's, and
    rows that do not meet."""
    q, s, qs = _weights(ops, n, k, dtype, 6)
    g = torch.Generator(device="cuda").manual_seed(m * 5 + k)
    x = torch.randn(m, k + 8, device="cuda", generator=g).to(dtype)[:, :k]
    b = torch.randn(n, device="cuda", generator=g).to(dtype)
    what = f"half m={m} n={n} k={k} {dtype}"
    y = ops.w8a16_gemm_strips(x, qs, n, s, b)
    assert_close(y, _ref64(x, q, s, b), what)
    res = torch.randn(m, n + 3, device="cuda", generator=g).to(dtype)[:, :n]
    assert torch.equal(ops.w8a16_fused_gemm_strips(x, qs, n, s, b, residual=res), res + y), what
    odd = x.clone()
    odd[0], odd[m // 2] = float("inf"), float("nan")
    rest = [i for i in range(m) if i not in (0, m // 2)]
    assert torch.equal(ops.w8a16_gemm_strips(odd, qs, n, s, b)[rest], y[rest]), what
    qf, sf = ops.pack_fp8((torch.randn(n, k, device="cuda", generator=g) * 0.02).to(dtype))
    assert_close(ops.fp8w_gemm_strips(x, ops.fp8w_strips(qf), n, sf, b), _ref64(x, qf.float(), sf, b), what + " e4m3")
