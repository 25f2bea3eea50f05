"""The W4A16 quantiser's wide kernel (groups of 32, 64, 128) against the oracle,
bit for bit: exact ties, zero groups, subnormal, tiny and huge groups (whose
quotients leave the corrected-reciprocal range), group counts that do not fill
a block, weights at an address that takes the one-thread-per-group kernel, and
the non-finite check."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import w4a16 as OW
from oracle.bf16 import f32_to_bf16_bits

from ._helpers import from_bits, to_bits

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module", autouse=True)
def _require_gpu():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")


def _weights(rng, n, k):
    w = rng.normal(0, 0.02, (n, k)).astype(np.float32)
    w[0, :] = 0.0
    w[1 % n, :] = 1e-39                                    # subnormal
    w[2 % n, :] = rng.normal(0, 1, k) * np.float32(2.0**-120)
    w[3 % n, :] = rng.normal(0, 1, k) * np.float32(2.0**100)
    w[4 % n, :] = (np.arange(k) % 29 - 14) * 0.5           # absmax 7: every half is a tie
    w[5 % n, :] = ((np.arange(k) % 29 - 14) * 0.5) * 2.0**-95
    return f32_to_bf16_bits(w)


@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("n,k", [(7, 256), (33, 768)])
@pytest.mark.parametrize("shift", [0, 2])
def test_quantise_matches_oracle(rng, group, n, k, shift):
    from local_kimi_amd.quant import quantise

    bits = _weights(rng, n, k)
    flat = torch.empty(n * k + 8, dtype=torch.bfloat16, device=DEV)
    w = flat[shift:shift + n * k].view(n, k)  # shift 2: a 4-byte aligned address
    w.copy_(from_bits(bits, DEV))
    got = quantise(w, group_size=group)
    packed, scales = OW.quantise(bits, group)
    assert np.array_equal(to_bits(got.scales), scales)
    assert np.array_equal(got.packed.cpu().numpy(), packed)


@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_quantise_rejects_non_finite(rng, group, bad):
    from local_kimi_amd.quant import quantise

    w = torch.randn(5, 512, device=DEV).to(torch.bfloat16)
    w[4, 511] = bad
    with pytest.raises(ValueError, match="finite"):
        quantise(w, group_size=group)
    w[4, 511] = 0.0
    quantise(w, group_size=group)


@pytest.mark.parametrize("group", [32, 64, 128, 256])
@pytest.mark.parametrize("shift", [0, 2])
def test_c_quantiser_on_non_finite_weights(rng, group, shift):
    """The C entry without a flag: a NaN (quiet or signalling) is left out of its
    group's absmax and coded -7, an infinity makes the scale infinite; the other
    groups are the oracle's. The same at every width and address."""
    from local_kimi_amd import _lib

    n, k = 6, 512
    bits = f32_to_bf16_bits(rng.normal(0, 0.02, (n, k)).astype(np.float32))
    bits[0, 3], bits[1, 300], bits[2, 511] = 0x7FC0, 0xFFC1, 0x7F81
    bits[4, 17], bits[5, 200] = 0x7F80, 0xFF80
    nan = (bits & 0x7FFF) > 0x7F80
    inf = (bits & 0x7FFF) == 0x7F80
    packed, scales = OW.quantise(np.where(nan | inf, 0, bits).astype(np.uint16), group)
    codes = np.stack((packed & 15, packed >> 4), -1).reshape(n, k)
    codes[nan | inf] = 9
    wide = inf.reshape(n, -1, group).any(-1)
    codes[np.repeat(wide, group, 1) & ~inf] = 0
    scales[wide] = 0x7F80

    flat = torch.empty(n * k + 8, dtype=torch.bfloat16, device=DEV)
    w = flat[shift:shift + n * k]
    w.copy_(from_bits(bits, DEV).view(-1))
    got_p = torch.empty((n, k // 2), dtype=torch.uint8, device=DEV)
    got_s = torch.empty((n, k // group), dtype=torch.bfloat16, device=DEV)
    _lib.call("lk_w4a16_quantise", w.data_ptr(), got_p.data_ptr(), got_s.data_ptr(), n, k, group,
              torch.cuda.current_stream().cuda_stream)
    assert np.array_equal(to_bits(got_s), scales)
    assert np.array_equal(got_p.cpu().numpy(), (codes[:, 0::2] | codes[:, 1::2] << 4).astype(np.uint8))


def test_quantise_takes_more_weights_than_a_launch_has_threads(rng):
    """2^35 weights: a thread per 8 of them is more than a launch holds, a thread
    per group is not."""
    from local_kimi_amd.quant import quantise

    n, k = 1 << 21, 1 << 14
    if torch.cuda.mem_get_info()[0] < 110 << 30:
        pytest.skip("needs 110 GB of device memory")
    some = f32_to_bf16_bits(rng.normal(0, 0.02, (3, k)).astype(np.float32))
    w = torch.zeros((n, k), dtype=torch.bfloat16, device=DEV)
    rows = [0, n // 2 + 1, n - 1]
    for r, bits in zip(rows, some):
        w[r] = from_bits(bits, DEV)
    got = quantise(w)
    packed, scales = OW.quantise(some, 32)
    for i, r in enumerate(rows):
        assert np.array_equal(got.packed[r].cpu().numpy(), packed[i])
        assert np.array_equal(to_bits(got.scales[r]), scales[i])
    assert not bool(got.packed[1:n // 2].any()) and bool((got.scales[1:n // 2] == 1).all())
    del w, got
    torch.cuda.empty_cache()
