"""GPU parity of the prefill GEMM (64- and 80-row tiles, direct LDS loads).

Against the oracle within the quantized-matmul tolerance (1e-2 relative / 2e-2
absolute in bf16), at the edges of its tiles: row counts around 16, 64 and 80,
column counts around 128 and 256 and not a multiple of 8, an odd number of
k-steps (whose scale rows start on odd values at G = 128), every group width.
The W4A16 forms also perform the LDS-staged kernel's MFMA chains in its order,
so their outputs must be its bits.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import moe as OM
from oracle import mxfp4 as X
from oracle import w4a16 as OW
from oracle.bf16 import bf16_bits_to_f32

from ._helpers import assert_close_bf16, from_bits, random_bf16_bits, to_bits

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _require_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from local_kimi_amd import _lib

    _lib.load()


def _dev(a):
    if a.dtype == np.uint16:
        return from_bits(a, DEV)
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def _w4(rng, n, k, g):
    return OW.quantise(random_bf16_bits(rng, (n, k), 0.02), g)


def _mx(rng, n, k):
    return X.quantize(bf16_bits_to_f32(random_bf16_bits(rng, (n, k), 0.02)))


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("m,n,k", [(16, 8, 128), (17, 130, 384), (63, 250, 256), (64, 256, 640),
                                   (65, 128, 384), (129, 1001, 128), (200, 264, 1152)])
def test_dense_tiles_match_oracle_and_staged_kernel(rng, group, m, n, k):
    from local_kimi_amd._lib import forced_path
    from local_kimi_amd.kernels import w4a16_dense_gemm

    x = random_bf16_bits(rng, (m, k))
    p, s = _w4(rng, n, k, group)
    args = (_dev(x), _dev(p), _dev(s))
    y = w4a16_dense_gemm(*args)
    with forced_path("dense_gemm", "lds"):
        staged = w4a16_dense_gemm(*args)
    assert torch.equal(y, staged), "prefill and LDS-staged kernels differ"
    assert_close_bf16(to_bits(y), OW.dense(x, p, s, group), what=f"dense {m}x{n}x{k} G={group}")


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("m,n,k", [(16, 8, 128), (33, 250, 384), (65, 300, 1152)])
def test_mxfp4_dense_tiles_match_oracle(rng, f16, m, n, k):
    from local_kimi_amd.kernels import mxfp4_gemm

    p, s = _mx(rng, n, k)
    if f16:
        x = rng.normal(0, 1, (m, k)).astype(np.float16)
        y = mxfp4_gemm(torch.from_numpy(x).to(DEV), _dev(p), _dev(s)).float().cpu().numpy()
        want = x.astype(np.float64) @ X.dequantize(p, s).astype(np.float64).T
        # one rounding to fp16 (2^-11) of an fp32 sum
        assert np.abs(y - want).max() <= 2.0 ** -10 * np.abs(want).max()
    else:
        x = random_bf16_bits(rng, (m, k))
        assert_close_bf16(to_bits(mxfp4_gemm(_dev(x), _dev(p), _dev(s))), X.linear(x, p, s),
                          what=f"mxfp4 {m}x{n}x{k}")


@pytest.mark.parametrize("weights", ["g32", "g64", "g128", "mxfp4"])
@pytest.mark.parametrize("h,inter,tokens", [(384, 256, 97), (256, 384, 300)])
def test_moe_block_tiles_match_oracle_and_staged_kernel(rng, weights, h, inter, tokens):
    """Few experts, so tiles of every height up to 80 rows; the staged kernel
    (path knob moe_gemm=lds) on the same routes gives the same bits (W4A16)."""
    from local_kimi_amd._lib import forced_path
    from local_kimi_amd.kernels import mxfp4_moe_block, w4a16_moe_forward

    e_routed, k = 7, 2
    group = 32 if weights == "mxfp4" else int(weights[1:])
    one = _mx if weights == "mxfp4" else lambda r, n, kk: _w4(r, n, kk, group)

    def bank(n, kk):
        enc = [one(rng, n, kk) for _ in range(e_routed + 1)]
        return np.stack([p for p, _ in enc]), np.stack([s for _, s in enc])

    banks = (*bank(inter, h), *bank(inter, h), *bank(h, inter))
    x = random_bf16_bits(rng, (tokens, h))
    # uneven experts: from a few rows to most of the batch
    logits = (rng.normal(0, 1, (tokens, e_routed)) +
              np.linspace(-2.5, 2.5, e_routed)).astype(np.float32)
    block = mxfp4_moe_block if weights == "mxfp4" else w4a16_moe_forward
    args = (_dev(x), _dev(logits), None, *(_dev(b) for b in banks), k, 2.446)
    with forced_path("moe_gemm", "stream64"):
        y, idx, _ = block(*args)
    with forced_path("moe_gemm", "lds"):
        y0, idx0, _ = block(*args)
    assert torch.equal(idx, idx0)
    if weights == "mxfp4":
        ey, eidx, _ = X.moe_block(x, logits, None, *banks, top_k=k, routed_scaling_factor=2.446)
    else:
        assert torch.equal(y, y0), "prefill and LDS-staged kernels differ"
        ey, eidx, _ = OM.moe_block(x, logits, None, *banks, top_k=k, routed_scaling_factor=2.446,
                                   group_size=group)
    assert np.array_equal(idx.cpu().numpy(), eidx)
    assert_close_bf16(to_bits(y), ey, what=f"{weights} moe block h={h} i={inter} T={tokens}")


def test_dense_group_32_without_workspace_still_runs(rng):
    """The C entry took G = 32 without a workspace; it still does, same bits."""
    from local_kimi_amd import _lib
    from local_kimi_amd.kernels import w4a16_dense_gemm

    m, n, k = 40, 96, 256
    x, (p, s) = random_bf16_bits(rng, (m, k)), _w4(rng, n, k, 32)
    dx, dp, ds = _dev(x), _dev(p), _dev(s)
    y = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    _lib.call("lk_w4a16_dense_gemm_ws", dx.data_ptr(), dp.data_ptr(), ds.data_ptr(), y.data_ptr(),
              m, n, k, 32, None, 0, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(y, w4a16_dense_gemm(dx, dp, ds))


@pytest.mark.parametrize("group", [32, 128])
@pytest.mark.parametrize("m,n,k", [(16, 250, 4096), (70, 576, 5248), (130, 129, 9216)])
def test_dense_split_over_k_matches_oracle(rng, group, m, n, k):
    """Too few blocks to fill the chip: runs of k with fp32 sums. The split only
    reorders fp32 additions, so it stays within the same tolerance, and within
    1e-5 of the unsplit sums' magnitude before the rounding to bf16 (2^-8)."""
    from local_kimi_amd import _lib
    from local_kimi_amd.kernels import w4a16_dense_gemm

    x, (p, s) = random_bf16_bits(rng, (m, k)), _w4(rng, n, k, group)
    assert _lib.query("lk_dense_gemm_workspace", m, n, k, group, 1, 0) > \
        2 * m * k + (4 if group == 32 else 1) * 4 * m * (k // 128) + 1024  # it does split
    dx, dp, ds = _dev(x), _dev(p), _dev(s)
    y = w4a16_dense_gemm(dx, dp, ds)
    assert_close_bf16(to_bits(y), OW.dense(x, p, s, group), what=f"split {m}x{n}x{k} G={group}")
    if group == 128:  # the smaller workspace of the older query: unsplit
        whole = torch.empty_like(y)
        ws = torch.empty(_lib.query("lk_w4a16_dense_gemm_workspace", m, k, group),
                         dtype=torch.uint8, device=DEV)
        _lib.call("lk_w4a16_dense_gemm_ws", dx.data_ptr(), dp.data_ptr(), ds.data_ptr(),
                  whole.data_ptr(), m, n, k, group, ws.data_ptr(), ws.numel(),
                  torch.cuda.current_stream().cuda_stream)
        diff = (y.float() - whole.float()).abs()
        assert bool((diff <= 2.0**-7 * whole.float().abs() + 1e-5 * whole.float().abs().max()).all())


def test_fused_qkv_and_mxfp4_split_over_k_match_oracle(rng):
    from local_kimi_amd.kernels import fused_qkv_w4a16, mxfp4_gemm

    m, n, k = 20, 136, 4096
    x = random_bf16_bits(rng, (m, k))
    mats = [_w4(rng, n, k, 32) for _ in range(3)]
    out = fused_qkv_w4a16(_dev(x), *(_dev(a) for pair in mats for a in pair))
    for y, (p, s) in zip(out, mats):
        assert_close_bf16(to_bits(y), OW.dense(x, p, s, 32), what="split fused qkv")
    p, s = _mx(rng, n, 9216)
    x = random_bf16_bits(rng, (m, 9216))
    assert_close_bf16(to_bits(mxfp4_gemm(_dev(x), _dev(p), _dev(s))), X.linear(x, p, s),
                      what="split mxfp4")
    xh = rng.normal(0, 1, (m, 9216)).astype(np.float16)
    y = mxfp4_gemm(torch.from_numpy(xh).to(DEV), _dev(p), _dev(s)).float().cpu().numpy()
    want = xh.astype(np.float64) @ X.dequantize(p, s).astype(np.float64).T
    assert np.abs(y - want).max() <= 2.0 ** -10 * np.abs(want).max()


@pytest.mark.parametrize("group", [32, 128])
def test_rows_are_paired_only_for_the_kernel_that_reads_them(rng, group):
    """Scales off the direct loads' dwords: the staged kernel runs, with its bits,
    and the workspace for paired rows is left as it was."""
    from local_kimi_amd import _lib
    from local_kimi_amd.kernels import w4a16_dense_gemm

    m, n, k = 40, 96, 256
    x, (p, s) = random_bf16_bits(rng, (m, k)), _w4(rng, n, k, group)
    dx, dp, ds = _dev(x), _dev(p), _dev(s)
    moved = torch.empty(ds.numel() + 1, dtype=torch.bfloat16, device=DEV)
    moved[1:].copy_(ds.view(-1))
    ws = torch.full((_lib.query("lk_dense_gemm_workspace", m, n, k, group, 1, 0),), 0xA5,
                    dtype=torch.uint8, device=DEV)
    y = torch.empty((m, n), dtype=torch.bfloat16, device=DEV)
    _lib.call("lk_w4a16_dense_gemm_ws", dx.data_ptr(), dp.data_ptr(), moved.data_ptr() + 2,
              y.data_ptr(), m, n, k, group, ws.data_ptr(), ws.numel(),
              torch.cuda.current_stream().cuda_stream)
    assert torch.equal(y, w4a16_dense_gemm(dx, dp, ds))
    assert bool((ws == 0xA5).all())


def _shifted(t, by):
    """A copy of t, `by` bytes off the allocator's alignment."""
    buf = torch.empty(t.numel() * t.element_size() + 16, dtype=torch.uint8, device=DEV)
    return buf[by:by + t.numel() * t.element_size()].view(t.dtype).view(t.shape).copy_(t)


@pytest.mark.parametrize("by", [4, 8, 12])
@pytest.mark.parametrize("weights", ["g32", "g64", "g128", "mxfp4"])
def test_operands_on_any_dword_keep_the_prefill_gemm(rng, weights, by):
    """Codes, scales, rows and outputs on a dword that no 16-byte line starts at:
    the same bits, from the same kernel (a dense W4A16 call writes its workspace)."""
    from local_kimi_amd import _lib
    from local_kimi_amd._lib import forced_path
    from local_kimi_amd.kernels import mxfp4_gemm, mxfp4_moe_block, w4a16_moe_forward

    m, n, k = 100, 264, 640
    stream = torch.cuda.current_stream().cuda_stream
    if weights == "mxfp4":
        x, (p, s) = random_bf16_bits(rng, (m, k)), _mx(rng, n, k)
        dx, dp, ds = _dev(x), _dev(p), _dev(s)
        assert torch.equal(mxfp4_gemm(*(_shifted(t, by) for t in (dx, dp, ds))), mxfp4_gemm(dx, dp, ds))
        group, one, block = 32, _mx, mxfp4_moe_block
    else:
        group = int(weights[1:])
        x, (p, s) = random_bf16_bits(rng, (m, k)), _w4(rng, n, k, group)
        dx, dp, ds = _dev(x), _dev(p), _dev(s)
        out = []
        for args in ((dx, dp, ds), tuple(_shifted(t, by) for t in (dx, dp, ds))):
            ws = torch.full((_lib.query("lk_dense_gemm_workspace", m, n, k, group, 1, 0),), 0xA5,
                            dtype=torch.uint8, device=DEV)
            y = torch.empty((m * n,), dtype=torch.bfloat16, device=DEV)
            y = _shifted(y, 0 if args[0] is dx else by)
            _lib.call("lk_w4a16_dense_gemm_ws", *(t.data_ptr() for t in args), y.data_ptr(), m, n, k,
                      group, ws.data_ptr(), ws.numel(), stream)
            assert not bool((ws == 0xA5).all()), "not the prefill GEMM"
            out.append(y)
        assert torch.equal(*out)
        one, block = (lambda r, nn, kk: _w4(r, nn, kk, group)), w4a16_moe_forward

    e_routed, top_k, h, inter, tokens = 7, 2, 384, 256, 150

    def bank(nn, kk):
        enc = [one(rng, nn, kk) for _ in range(e_routed + 1)]
        return _dev(np.stack([c for c, _ in enc])), _dev(np.stack([c for _, c in enc]))

    banks = (*bank(inter, h), *bank(inter, h), *bank(h, inter))
    hx = _dev(random_bf16_bits(rng, (tokens, h)))
    logits = _dev(rng.normal(0, 1, (tokens, e_routed)).astype(np.float32))
    with forced_path("moe_gemm", "stream64"):
        y0 = block(hx, logits, None, *banks, top_k, 2.446)[0]
        y1 = block(_shifted(hx, by), logits, None, *(_shifted(b, by) for b in banks), top_k, 2.446)[0]
    assert torch.equal(y0, y1)


def test_rows_beyond_the_pairing_run_staged(rng):
    """2^27 row k-steps (34 GB of rows) at G = 32: more than one pairing launch
    takes, and than the direct loads' offsets reach."""
    from local_kimi_amd._lib import forced_path
    from local_kimi_amd.kernels import w4a16_dense_gemm

    m, n, k = 1 << 20, 32, 16384
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GB of device memory")
    p, s = _w4(rng, n, k, 32)
    x = torch.zeros((m, k), dtype=torch.bfloat16, device=DEV)
    x[-80:] = torch.randn(80, k, device=DEV).to(torch.bfloat16)
    x[:16] = x[-16:]
    y = w4a16_dense_gemm(x, _dev(p), _dev(s))
    with forced_path("dense_gemm", "lds"):
        want = w4a16_dense_gemm(x[-80:].clone(), _dev(p), _dev(s))
    assert torch.equal(y[-80:], want)
    assert torch.equal(y[:16], want[-16:])
    assert not bool(y[16:-80].any())


@pytest.mark.parametrize("m,n,k", [(700, 2304, 9216), (1600, 1001, 8192)])
def test_dense_split_of_256_column_blocks_matches_oracle(rng, m, n, k):
    """256-column blocks in four runs of k (G = 128): a ragged last row tile, odd
    widths; the oracle on rows of every kind of tile."""
    from local_kimi_amd.kernels import w4a16_dense_gemm

    x, (p, s) = random_bf16_bits(rng, (m, k)), _w4(rng, n, k, 128)
    y = to_bits(w4a16_dense_gemm(_dev(x), _dev(p), _dev(s)))
    rows = np.unique(np.concatenate(([0, 15, 16, 63, 64, m - 65, m - 1], rng.integers(0, m, 8))))
    assert_close_bf16(y[rows], OW.dense(x[rows], p, s, 128), what=f"wide split {m}x{n}x{k}")


@pytest.mark.parametrize("k", [128, 384])
@pytest.mark.parametrize("n", [5000, 5001])
@pytest.mark.parametrize("weights", ["g32", "g64", "g128", "bf16", "f16"])
def test_dense_256_column_blocks(rng, weights, n, k):
    """Enough blocks (21 x 20) for 256 columns each: a ragged last row tile and
    last column block, values one by one (n = 5001), an odd number of k-steps,
    the even split over the XCDs. W4A16 against the LDS-staged kernel's bits,
    and everything against the oracle on sampled rows."""
    from local_kimi_amd._lib import forced_path
    from local_kimi_amd.kernels import mxfp4_gemm, w4a16_dense_gemm

    m = 1301
    rows = np.array([0, 15, 16, 63, 64, 700, 1279, 1280, 1300])
    if weights[0] == "g":
        group = int(weights[1:])
        x, (p, s) = random_bf16_bits(rng, (m, k)), _w4(rng, n, k, group)
        args = (_dev(x), _dev(p), _dev(s))
        y = w4a16_dense_gemm(*args)
        with forced_path("dense_gemm", "lds"):
            assert torch.equal(y, w4a16_dense_gemm(*args))
        assert_close_bf16(to_bits(y)[rows], OW.dense(x[rows], p, s, group), what=f"{weights} {n} {k}")
        return
    p, s = _mx(rng, n, k)
    if weights == "bf16":
        x = random_bf16_bits(rng, (m, k))
        y = mxfp4_gemm(_dev(x), _dev(p), _dev(s))
        assert_close_bf16(to_bits(y)[rows], X.linear(x[rows], p, s), what=f"mxfp4 {n} {k}")
    else:
        x = rng.normal(0, 1, (m, k)).astype(np.float16)
        y = mxfp4_gemm(torch.from_numpy(x).to(DEV), _dev(p), _dev(s)).float().cpu().numpy()[rows]
        want = x[rows].astype(np.float64) @ X.dequantize(p, s).astype(np.float64).T
        # one rounding to fp16 (2^-11) of an fp32 sum
        assert np.abs(y - want).max() <= 2.0 ** -10 * np.abs(want).max()
