"""Vision attention from LDS: views, magnitudes and masked-like keys against 64 bits.

P is rounded to bf16 (2^-9 relative each) and so is the output: with 256 keys the P roundings
average out below one output rounding, so 2^-7 of a row's largest value covers both."""
import pytest
import torch

from flash_vla_amd.arena import ScratchPool
from flash_vla_amd.backends.hip import _abi
from flash_vla_amd.backends.hip import vision_wrappers as VW
from flash_vla_amd.backends.hip import wrappers as W

pytestmark = pytest.mark.gpu


def _ref(qkv):
    n = qkv.shape[0]
    q, k, v = qkv.double().reshape(n, 256, 3, 16, 72).permute(2, 0, 3, 1, 4)
    p = torch.softmax(q @ k.transpose(-1, -2) / 72 ** 0.5, -1)
    return (p @ v).transpose(1, 2).reshape(n, 256, 1152)


@pytest.mark.parametrize("views", [1, 4, 13])
@pytest.mark.parametrize("scale", [0.0, 1.0, 6.0])       # flat, ordinary, nearly one-hot
def test_against_64_bits(views, scale):
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    g = torch.Generator(device="cuda").manual_seed(views)
    qkv = torch.randn(views, 256, 3456, generator=g, device="cuda")
    qkv[..., :2304] *= scale
    qkv[:, 100:140, 1152:2304] -= 4 * scale              # a run of keys that most queries skip
    qkv = qkv.bfloat16()
    with W.use_pool(ScratchPool()):
        out = VW.vision_attention(qkv)
    ref = _ref(qkv)
    assert torch.all((out.double() - ref).abs() <= 2.0 ** -7 * ref.abs().amax(-1, keepdim=True))


def test_non_finite():
    """A key with an infinity (weight 0 or NaN by the query's sign), a NaN query, an infinite V:
    what the formula gives, in their own head and view alone."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    g = torch.Generator(device="cuda").manual_seed(7)
    qkv = torch.randn(2, 256, 3456, generator=g, device="cuda")
    qkv[0, :, 72 + 3] = qkv[0, :, 72 + 3].abs() + 0.1     # head 1's queries, dim 3
    qkv[0, 200, 72 + 3] = -1.0
    qkv[0, 150, 1152 + 72 + 3] = -float("inf")
    qkv[0, 30, 5 * 72] = float("nan")
    qkv[1, 250, 2304 + 15 * 72 + 71] = float("inf")
    qkv = qkv.bfloat16()
    with W.use_pool(ScratchPool()):
        out = VW.vision_attention(qkv).double()
    ref = _ref(qkv)
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    ok = ref.isfinite()
    assert torch.all((out[ok] - ref[ok]).abs() <= 2.0 ** -7 * ref[ok].abs().max())


def test_wide_row_pitch():
    """Rows 5,000,000 elements apart, past 32-bit offsets over a view: bitwise the packed result."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    g = torch.Generator(device="cuda").manual_seed(8)
    qkv = torch.randn(256, 3456, generator=g, device="cuda").bfloat16()
    pitch = 5_000_000
    wide = torch.empty(256 * pitch, dtype=torch.bfloat16, device="cuda").view(256, pitch)[:, :3456]
    wide.copy_(qkv)
    outs = [torch.zeros(256, 1152, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for t, out in zip((qkv, wide), outs):
        _abi.call("pi0hip_vision_attention", t.data_ptr(), t.stride(0), out.data_ptr(), 1152, 1, 256,
                  16, 72, 72 ** -0.5, None, 0, W._stream())
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)
    torch.cuda.empty_cache()
