"""The 8-wave block GEMMs and the batched decoder's kernels at ragged row counts.

Every tile accumulates each output over k in the same order, so a call's rows must be, bit for
bit, those of the same entry called on at most 200 of them at a time (which the strip tiles
serve; the oracle tests cover those). Sizes are one row into a tile's range or one short of
its end; nothing may be stored past row M."""
import pytest
import torch

from flash_vla_amd.backends.hip import _abi
from flash_vla_amd.backends.hip import wrappers as W

pytestmark = pytest.mark.gpu
DEV = "cuda"
CHUNK = 200


def rnd(shape, seed, scale=1.0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


def _rows_equal(M, N, call, init=None):
    """call(row0, rows, out): the entry on rows row0 .. row0 + rows - 1, into `out`'s rows."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    whole = torch.full((M + 3, N), 7.0, dtype=torch.bfloat16, device=DEV)
    if init is not None:
        whole[:M].copy_(init)
    parts = whole.clone()
    call(0, M, whole)
    for r in range(0, M, CHUNK):
        call(r, min(CHUNK, M - r), parts[r:])
    torch.cuda.synchronize()
    assert torch.isfinite(whole).all()
    assert torch.equal(whole, parts)
    assert torch.all(whole[M:] == 7.0), "stored past row M"


@pytest.mark.parametrize("M", [257, 384, 385, 513, 768, 769, 1153])
def test_gated_ffn_blocks(M):
    K, N = 2048, 16384
    x, g, u = rnd((M, K), 1), rnd((K, N), 2, 0.02), rnd((K, N), 3, 0.02)
    gp, up = W.packed_weight_ptr(g, 32), W.packed_weight_ptr(u, 32)
    _rows_equal(M, N, lambda r, n, out: _abi.call(
        "pi0hip_tile_gated_ffn", x[r:].data_ptr(), K, gp, up, out.data_ptr(), N, n, N, K,
        W._stream()))


def _wide(x, pitch):
    """x's rows `pitch` elements apart (gigabytes, of which only the rows are touched)."""
    w = torch.empty(x.shape[0] * pitch, dtype=x.dtype, device=DEV).view(-1, pitch)[:, :x.shape[1]]
    w.copy_(x)
    return w


def test_wide_row_pitches():
    """A pitch past the tall tiles' 32-bit offsets (384 rows x 6,000,000 elements), and past
    those of the resource over all rows of a batch: bitwise the contiguous call's result."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    x, g, u = rnd((300, 128), 31), rnd((128, 128), 32, 0.1), rnd((128, 128), 33, 0.1)
    outs = [torch.zeros(300, 128, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    for xs, out in zip((x, _wide(x, 6_000_000)), outs):
        _abi.call("pi0hip_tile_gated_ffn", xs.data_ptr(), xs.stride(0), W.packed_weight_ptr(g, 32),
                  W.packed_weight_ptr(u, 32), out.data_ptr(), 128, 300, 128, 128, W._stream())
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)
    x, g, u = rnd((256, 1024), 34), rnd((1024, 64), 35, 0.02), rnd((1024, 64), 36, 0.02)
    outs = [torch.zeros(256, 64, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    for xs, out in zip((x, _wide(x, 9_000_000)), outs):
        W.decoder_norm_gated_ffn(xs, g, u, out, None)
    assert torch.isfinite(outs[0]).all() and torch.equal(*outs)
    torch.cuda.empty_cache()


@pytest.mark.parametrize("M", [1025, 2049, 4097, 6201])
def test_residual_blocks(M):
    K, N = 3072, 2048      # not a K of the whole-K kernel, which sums in another order
    x, w, r0 = rnd((M, K), 4), rnd((K, N), 5, 0.02), rnd((M, N), 6)
    wp = W.packed_weight_ptr(w, 32)
    _rows_equal(M, N, lambda r, n, out: _abi.call(
        "pi0hip_tile_linear_residual", x[r:].data_ptr(), K, wp, out.data_ptr(), N, n, N, K, 1,
        None, 0, W._stream()), r0)


@pytest.mark.parametrize("K", [2048, 4096])
@pytest.mark.parametrize("M", [65, 96, 204, 225, 255, 256, 257, 511])
def test_whole_k_residual(M, K):
    """32 x 32 outputs over the whole K (up to 256 rows at N = 1024; past it the unsplit 32 x 128
    strip), against a 64-bit product: bf16 rounding of the output
    alone is 2^-9 of a value, the fp32 sums' order adds 1e-6 of the row's scale."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    N = 1024
    x, w, r0 = rnd((M, K), 19), rnd((K, N), 20, 0.02), rnd((M, N), 21)
    out = torch.full((M + 3, N), 7.0, dtype=torch.bfloat16, device=DEV)
    out[:M].copy_(r0)
    _abi.call("pi0hip_tile_linear_residual", x.data_ptr(), K, W.packed_weight_ptr(w, 32),
              out.data_ptr(), N, M, N, K, 1, None, 0, W._stream())
    torch.cuda.synchronize()
    ref = x.double() @ w.double() + r0.double()
    tol = 2.0 ** -8 * ref.abs() + 1e-5 * ref.abs().max()
    assert torch.all((out[:M].double() - ref).abs() <= tol)
    assert torch.all(out[M:] == 7.0), "stored past row M"


@pytest.mark.parametrize("M,split", [(300, 8), (511, 8), (640, 8), (1001, 8), (1101, 4), (2047, 4),
                                     (2305, 4)])
def test_split_k_blocks(M, split):
    K, N = 8192, 2048
    x, w, r0 = rnd((M, K), 7), rnd((K, N), 8, 0.02), rnd((M, N), 9)
    wp = W.packed_weight_ptr(w, 32)
    ws = torch.empty(_abi.lib().pi0hip_tile_workspace_bytes(M, N, split), dtype=torch.uint8, device=DEV)
    _rows_equal(M, N, lambda r, n, out: _abi.call(
        "pi0hip_tile_linear_residual", x[r:].data_ptr(), K, wp, out.data_ptr(), N, n, N, K, split,
        ws.data_ptr(), ws.numel(), W._stream()), r0)


@pytest.mark.parametrize("M", [300, 993, 1153, 2047])
def test_bias_blocks(M):
    K, N = 1152, 3456
    x, w, b = rnd((M, K), 10), rnd((K, N), 11, 0.03), rnd(N, 12, 0.5)
    wp = W.packed_weight_ptr(w, 32)
    _rows_equal(M, N, lambda r, n, out: _abi.call(
        "pi0hip_tile_linear", x[r:].data_ptr(), K, wp, b.data_ptr(), out.data_ptr(), N, n, N, K,
        W._stream()))


@pytest.mark.parametrize("M", [1601, 1921, 2881, 4097])
def test_bias_gelu_blocks(M):
    K, N, N_pad = 1152, 4304, 4352
    x, w, b = rnd((M, K), 13), rnd((K, N), 14, 0.03), rnd(N, 15, 0.5)
    wp = W.packed_weight_ptr(w, 32, (K, N_pad))
    _rows_equal(M, N, lambda r, n, out: _abi.call(
        "pi0hip_tile_linear_bias_gelu", x[r:].data_ptr(), K, wp, b.data_ptr(), out.data_ptr(), N,
        n, N, K, N_pad, K, W._stream()))


@pytest.mark.parametrize("M", [769, 1601, 3201, 4801])
def test_qkv_rope_blocks(M):
    K, heads, hd = 2048, 8, 256
    x, w, rope = rnd((M, K), 16), rnd((K, (heads + 2) * hd), 17, 0.02), rnd((M, hd), 18)
    wp = W.packed_weight_ptr(w, 32)

    def call(r, n, out):       # Q, K and V side by side in three of out's column ranges
        q, k, v = (torch.full((n, c), 7.0, dtype=torch.bfloat16, device=DEV)
                   for c in (heads * hd, hd, hd))
        _abi.call("pi0hip_tile_qkv_rope", x[r:].data_ptr(), K, wp, rope[r:].data_ptr(),
                  q.data_ptr(), k.data_ptr(), v.data_ptr(), hd, n, K, heads, hd, W._stream())
        out[:n].copy_(torch.cat([q, k, v], 1))

    _rows_equal(M, (heads + 2) * hd, call)


@pytest.mark.parametrize("B,T", [(5, 13), (2, 33), (3, 41), (8, 64)])
def test_batched_qkv_rows(B, T):
    """The batch's 32-row workgroups against one request at a time (M = T <= 64), bit for bit."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    K, heads, hd = 1024, 8, 256
    x, w, rope = rnd((B * T, K), 22), rnd((K, (heads + 2) * hd), 23, 0.02), rnd((T, hd), 24)

    def run(xs, batch):
        rows = xs.shape[0]
        q = torch.zeros(rows * heads, hd, dtype=torch.bfloat16, device=DEV)
        k = torch.zeros((batch, T + 1, hd), dtype=torch.bfloat16, device=DEV)
        v, nf = k.clone(), torch.zeros(rows, dtype=torch.bfloat16, device=DEV)
        args = (k[:, :T], v[:, :T]) if batch > 1 else (k[0, :T], v[0, :T])
        W.decoder_norm_qkv_rope(xs, w, rope, q, *args, nf)
        return q.view(batch, T, -1), k, v, nf

    def row(b, t):           # states first
        return b if t == 0 else B + b * (T - 1) + t - 1

    q, k, v, nf = run(x, B)
    for b in range(B):
        idx = torch.tensor([row(b, t) for t in range(T)], device=DEV)
        q1, k1, v1, nf1 = run(x[idx].contiguous(), 1)
        assert torch.equal(q[b], q1[0]) and torch.equal(k[b], k1[0]) and torch.equal(v[b], v1[0])
        assert torch.equal(nf[idx], nf1)


@pytest.mark.parametrize("M", [65, 128, 129, 192, 193, 256])
def test_batched_gate_rows(M):
    """All rows of a batch streamed past a column tile, against 64 rows at a time, bit for bit."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    K, N = 1024, 4096
    x, g, u = rnd((M, K), 25), rnd((K, N), 26, 0.02), rnd((K, N), 27, 0.02)
    out = torch.full((M + 3, N), 7.0, dtype=torch.bfloat16, device=DEV)
    W.decoder_norm_gated_ffn(x, g, u, out[:M], None)
    for r in range(0, M, 64):
        n = min(64, M - r)
        part = torch.zeros(n, N, dtype=torch.bfloat16, device=DEV)
        W.decoder_norm_gated_ffn(x[r:r + n], g, u, part, None)
        assert torch.equal(out[r:r + n], part)
    assert torch.all(out[M:] == 7.0), "stored past row M"


@pytest.mark.parametrize("B,L", [(3, 769), (8, 256), (5, 415), (2, 1024), (2, 815)])
@pytest.mark.parametrize("scale", [1.0, 6.0])           # ordinary, nearly one-hot
def test_encoder_attention_many_rows(B, L, scale):
    """The 128-row workgroups (from 128 of them on; the last case stays below) against 64 bits:
    P's and the output's bf16 roundings, 2^-9 each, and the smaller form's bf16 logits."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from flash_vla_amd.arena import ScratchPool
    from flash_vla_amd.backends.hip import encoder_wrappers as EW
    q, k, v = rnd((B * L * 8, 256), 28, scale), rnd((B, L, 256), 29), rnd((B, L, 256), 30)
    with W.use_pool(ScratchPool()):
        out = EW.encoder_attention(q, k, v, 1 / 16).reshape(B, L * 8, 256).double()
    wide = B * ((L * 8 + 127) // 128) >= 128
    p = torch.softmax(q.double().reshape(B, L * 8, 256) @ k.double().transpose(1, 2) / 16, -1)
    ref = p @ v.double()
    err = ((out - ref).norm() / ref.norm()).item()
    # bf16 logits: 2^-9 of a logit of about 4 scale, so 4 scale 2^-9 on P
    assert err <= (4e-3 if wide else 4e-3 + scale * 2.0 ** -7), err
    assert torch.isfinite(out).all()


def _same_specials(out, ref, tol):
    """NaN where the reference has NaN, its infinities, and elsewhere its values within tol."""
    out, ref = out.double(), ref.double()
    assert torch.equal(out.isnan(), ref.isnan())
    inf = ref.isinf()
    assert torch.equal(out[inf], ref[inf])
    ok = ~inf & ~ref.isnan()
    assert ok.any() and torch.all((out[ok] - ref[ok]).abs() <= tol * ref[ok].abs().max())


def _gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(0.7978845608028654 * (v + 0.044715 * v ** 3)))


@pytest.mark.parametrize("entry,M,K,N", [
    ("gated", 300, 128, 128),              # 192-row blocks
    ("residual", 2100, 384, 2048),         # 128 x 256 blocks
    ("residual", 96, 2048, 128),           # 32 x 32 outputs over the whole K
    ("decoder gate", 130, 1024, 64)])      # rows streamed past a column tile
def test_non_finite_rows(entry, M, K, N):
    """A row with a NaN or an infinity gives what the formula gives, and no other row notices."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    x, w, u, r0 = rnd((M, K), 37), rnd((K, N), 38, 0.05), rnd((K, N), 39, 0.05), rnd((M, N), 40)
    for row, v in ((1, float("nan")), (33, float("inf")), (65, -float("inf")), (M - 1, float("inf"))):
        x[row, (7 * row) % K] = v
    out = r0.clone()
    xd = x.double()
    if entry == "residual":
        _abi.call("pi0hip_tile_linear_residual", x.data_ptr(), K, W.packed_weight_ptr(w, 32),
                  out.data_ptr(), N, M, N, K, 1, None, 0, W._stream())
        ref = xd @ w.double() + r0.double()
    elif entry == "gated":
        _abi.call("pi0hip_tile_gated_ffn", x.data_ptr(), K, W.packed_weight_ptr(w, 32),
                  W.packed_weight_ptr(u, 32), out.data_ptr(), N, M, N, K, W._stream())
        ref = _gelu(xd @ w.double()) * (xd @ u.double())
    else:
        W.decoder_norm_gated_ffn(x, w, u, out, None)
        f = torch.rsqrt(xd.square().mean(1, keepdim=True) + 1e-6).bfloat16().double()
        ref = _gelu(f * (xd @ w.double())) * (f * (xd @ u.double()))
    _same_specials(out, ref, 2.0 ** -7)     # the bf16 result, and the row factor's rounding twice


@pytest.mark.parametrize("B,L", [(2, 1024), (1, 100)])        # 128-row workgroups, 32-row ones
def test_encoder_attention_non_finite(B, L):
    """Keys with an infinity (weight 0 or NaN by the query's sign), a NaN query, an infinite V."""
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    from flash_vla_amd.arena import ScratchPool
    from flash_vla_amd.backends.hip import encoder_wrappers as EW
    q, k, v = rnd((B * L * 8, 256), 41), rnd((B, L, 256), 42), rnd((B, L, 256), 43)
    q[:, 5] = q[:, 5].abs() + 0.1
    q[3, 5] = -1.0                          # the one query that the key below attracts
    q[9, 0] = float("nan")
    k[:, 40, 5] = -float("inf")
    v[:, 70, 200] = float("inf")
    with W.use_pool(ScratchPool()):
        out = EW.encoder_attention(q, k, v, 1 / 16).reshape(B, L * 8, 256)
    p = torch.softmax(q.double().reshape(B, L * 8, 256) @ k.double().transpose(1, 2) / 16, -1)
    # P's 2^-9 roundings average out, the narrow form's bf16 logits add 4 x 2^-9
    _same_specials(out, p @ v.double(), 2.0 ** -5)
