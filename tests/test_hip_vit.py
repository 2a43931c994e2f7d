"""float32 ViT kernels and the end-to-end dynamic-quantized ViT against the CPU
restatement (oracle/vit.py).  float32 steps: 1e-4 relative (summation orders
differ); the quantized Linears inside are bit-exact given equal inputs, but
float32 noise ahead of a dynamic quantizer can move an activation across a
rounding tie, so end-to-end agreement is stated as a tolerance."""

import ctypes as C

import numpy as np
import pytest

import lucid_amd as L
import lucid_amd.nn.functional as F
import oracle as O
import oracle.vit as V
import workloads
from lucid_amd import _C

pytestmark = pytest.mark.gpu


def hip(a):
    return L.tensor(a, device="hip")


def rel(a, b):
    return float(np.max(np.abs(a.astype(np.float64) - b.astype(np.float64))) /
                 max(1e-30, np.max(np.abs(b.astype(np.float64)))))


@pytest.mark.parametrize("rows,cols", [(12608, 768), (7, 768), (5, 33), (1, 1), (64, 1000), (3, 4)])
def test_layer_norm(rows, cols):
    rng = np.random.default_rng(rows + cols)
    x = (rng.standard_normal((rows, cols)) * 2 + 0.5).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    b = (0.1 * rng.standard_normal(cols)).astype(np.float32)
    got = F.layer_norm(hip(x), cols, hip(g), hip(b), 1e-6).numpy()
    exp = V.layer_norm(x, g, b, 1e-6)
    assert np.max(np.abs(got - exp)) <= 1e-4 * max(1.0, np.max(np.abs(exp)))


@pytest.mark.parametrize("n", [1, 3, 1024, 12608 * 3072 // 8 + 5])
def test_gelu_and_add(n):
    rng = np.random.default_rng(n)
    x = (rng.standard_normal(n) * 2).astype(np.float32)
    y = rng.standard_normal(n).astype(np.float32)
    got = F.gelu(hip(x)).numpy()
    exp = V.gelu(x)
    assert np.max(np.abs(got - exp)) <= 2e-6
    assert np.array_equal(F.add(hip(x), hip(y)).numpy(), x + y)


def test_gelu_against_float64():
    """erf by a formula good to 1.5e-7, in float32: 4e-7 absolute at most (measured 3.8e-7), 1.5e-7 relative overall."""
    from scipy.special import erf
    x = np.concatenate([np.linspace(-12, 12, 1 << 20), np.random.default_rng(0).standard_normal(1 << 20)]).astype(np.float32)
    d = x.astype(np.float64)
    exp, got = 0.5 * d * (1 + erf(d / np.sqrt(2))), F.gelu(hip(x)).numpy()
    assert np.max(np.abs(got - exp)) <= 4e-7 and rel(got, exp) <= 1.5e-7
    edge = F.gelu(hip(np.array([np.inf, -np.inf, np.nan, 0, 3e38, -3e38], np.float32))).numpy()
    assert edge[0] == np.inf and np.isnan(edge[1:3]).all() and (edge[3:] == np.array([0, 3e38, 0], np.float32)).all()


@pytest.mark.parametrize("B,T,H", [(2, 197, 12), (1, 1, 1), (3, 16, 2), (2, 17, 3), (1, 208, 2), (4, 50, 12),
                                   (2, 70, 3), (1, 130, 2), (1, 193, 1), (2, 144, 2)])   # 5, 9, 13 tiles: the last one shared
def test_attention_on_packed_qkv(B, T, H):
    rng = np.random.default_rng(B * 1000 + T * 10 + H)
    qkv = rng.standard_normal((B, T, 3 * H * 64)).astype(np.float32)
    got = F.scaled_dot_product_attention_qkv(hip(qkv), H).numpy()
    exp = V.attention_qkv(qkv, H)
    assert rel(got, exp) < 1e-4


@pytest.mark.parametrize("B,T,H,std", [(1, 197, 64, 1.0), (5, 65, 13, 1.0),
                                       (4, 129, 67, 1.0), (43, 17, 12, 3.0),     # blocks that take a second item, heads not in eights
                                       (22, 197, 12, 2.0), (1, 208, 65, 0.1),
                                       (3, 64, 171, 1.0),                          # four tiles: one per wavefront for any count
                                       (8, 65, 16, 1.0), (3, 65, 43, 1.0), (2, 128, 128, 1.0), (1, 65, 257, 1.0),   # the last
                                       # count with one tile per wavefront, the first and last with a block per head, the first with two
                                       (4, 144, 42, 1.0), (1, 129, 169, 1.0), (8, 130, 32, 2.0), (2, 192, 121, 1.0),
                                       (16, 197, 8, 1.0), (1, 193, 129, 1.0), (8, 208, 28, 0.1), (1, 193, 225, 1.0)])
def test_attention_against_float64(B, T, H, std):
    """Scores and results are sums of 64 and T products, each exact to 2^-24 and accumulated in float32, behind
    exponentials good to an ulp: relative errors of a few 2^-24 per output (measured 1.4e-7 to 6e-7, growing with the scores)."""
    rng = np.random.default_rng(T + H)
    qkv = (rng.standard_normal((B, T, 3 * H * 64)) * std).astype(np.float32)
    out = F.scaled_dot_product_attention_qkv(hip(qkv), H, track_range=True)
    got = out.numpy()
    q, k, v = (qkv.astype(np.float64).reshape(B, T, 3, H, 64)[:, :, i].transpose(0, 2, 1, 3) for i in range(3))
    s = q @ k.transpose(0, 1, 3, 2) * 0.125
    p = np.exp(s - s.max(-1, keepdims=True))
    exp = ((p / p.sum(-1, keepdims=True)) @ v).transpose(0, 2, 1, 3).reshape(B, T, H * 64)
    assert np.linalg.norm(got - exp) <= 2e-6 * np.linalg.norm(exp)
    kmn, kmx, _, _ = _range_of(out)
    assert kmn == got.min() and kmx == got.max()
    qkv[0, T // 2, 2 * H * 64 + 5] = np.nan  # one value of head 0 of the first batch: its column of every query
    bad = F.scaled_dot_product_attention_qkv(hip(qkv), H, track_range=True)
    assert np.isnan(bad.numpy()[0, :, 5]).all() and np.isnan(bad.numpy()).sum() == T
    assert np.isnan(_range_of(bad)[0])


@pytest.mark.parametrize("B,T,H", [(1, 208, 2), (1, 17, 3), (6, 197, 12), (16, 193, 12), (21, 197, 12)])
@pytest.mark.parametrize("mag", [1e38, -1e38, 1e-30])
def test_attention_of_values_near_the_ends_of_the_range(B, T, H, mag):
    """A result is a mean of V's rows and no larger than the largest of them: sums on the way there stay finite for every
    finite V that the mean keeps finite, and small ones lose nothing.  The bound of the test above."""
    rng = np.random.default_rng(B + T)
    qkv = rng.uniform(0.5, 2.0, (B, T, 3, H, 64)).astype(np.float32)
    qkv[:, :, :2] = 0.03125 * rng.standard_normal((B, T, 2, H, 64))  # scores close to each other
    v = qkv[:, :, 2].astype(np.float64) * np.where(np.arange(64) % 2, mag, abs(mag))  # one sign per column
    qkv[:, :, 2] = v
    out = F.scaled_dot_product_attention_qkv(hip(qkv.reshape(B, T, -1)), H, track_range=True)
    got = out.numpy()
    q, k, v = (qkv[:, :, i].astype(np.float64).transpose(0, 2, 1, 3) for i in range(3))
    s = q @ k.transpose(0, 1, 3, 2) * 0.125
    p = np.exp(s - s.max(-1, keepdims=True))
    exp = ((p / p.sum(-1, keepdims=True)) @ v).transpose(0, 2, 1, 3).reshape(B, T, H * 64)
    assert np.isfinite(got).all()
    assert np.linalg.norm((got - exp) / mag) <= 2e-6 * np.linalg.norm(exp / mag)
    kmn, kmx, _, _ = _range_of(out)
    assert kmn == got.min() and kmx == got.max()


def test_attention_of_a_row_beyond_32_bits():
    """The first count of heads whose 32 token rows of the packed activation span more than 2^32 bytes: offsets of 64 bits,
    blocks that take many items with one tile of queries per wavefront.  The bound of the tests above, on every head."""
    T, H = 2, (1 << 32) // (3 * 64 * 4 * 32) + 1
    rng = np.random.default_rng(H)
    qkv = rng.standard_normal((T, 3, H, 64), dtype=np.float32)
    x = hip(qkv.reshape(1, T, -1))
    got = F.scaled_dot_product_attention_qkv(x, H).numpy().reshape(T, H, 64)
    q, k, v = (qkv[:, i].transpose(1, 0, 2).astype(np.float64) for i in range(3))
    s = q @ k.transpose(0, 2, 1) * 0.125
    p = np.exp(s - s.max(-1, keepdims=True))
    exp = ((p / p.sum(-1, keepdims=True)) @ v).transpose(1, 0, 2)
    err = np.linalg.norm((got - exp).transpose(1, 0, 2).reshape(H, -1), axis=1)
    assert (err <= 4e-6 * np.linalg.norm(exp.transpose(1, 0, 2).reshape(H, -1), axis=1)).all()  # per head: twice the bound overall
    assert np.linalg.norm(got - exp) <= 2e-6 * np.linalg.norm(exp)
    with pytest.raises(L.ShapeMismatch):  # a kept range stays limited to 16384 heads
        F.scaled_dot_product_attention_qkv(x, H, track_range=True)


def test_attention_rejects_what_the_kernel_does_not_cover():
    with pytest.raises(NotImplementedError):
        F.scaled_dot_product_attention_qkv(hip(np.zeros((1, 4, 3 * 2 * 32), np.float32)), 2)  # head dim 32
    with pytest.raises(NotImplementedError):
        F.scaled_dot_product_attention_qkv(hip(np.zeros((1, 209, 3 * 64), np.float32)), 1)  # 209 tokens


@pytest.mark.parametrize("M,N,K", [(12544, 768, 768), (1, 1, 1), (130, 70, 19), (64, 200, 768), (257, 129, 33)])
def test_float_linear(M, N, K):
    rng = np.random.default_rng(M + N + K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    got = F.linear_f32(hip(x), hip(w), hip(b)).numpy()
    exp = x.astype(np.float64) @ w.astype(np.float64).T + b
    assert rel(got, exp) < 1e-5
    got = F.linear_f32(hip(x), hip(w)).numpy()
    assert rel(got, x.astype(np.float64) @ w.astype(np.float64).T) < 1e-5


def test_patchify_and_token_assembly_are_exact():
    rng = np.random.default_rng(3)
    img = rng.standard_normal((3, 3, 32, 48)).astype(np.float32)
    rows = L.Tensor.empty((3 * 6, 3 * 256), L.float32, "hip")
    d_img = hip(img)
    _C.call("lq_patchify_f32", d_img.data_ptr, rows.data_ptr, 3, 3, 32, 48, 16, None)
    assert np.array_equal(rows.numpy(), V.patch_rows(img, 16))
    emb = rng.standard_normal((3, 6, 40)).astype(np.float32)
    cls = rng.standard_normal(40).astype(np.float32)
    pos = rng.standard_normal((7, 40)).astype(np.float32)
    out = L.Tensor.empty((3, 7, 40), L.float32, "hip")
    d_emb, d_cls, d_pos = hip(emb), hip(cls), hip(pos)  # held: a temporary's memory is reused at once
    _C.call("lq_assemble_tokens_f32", d_emb.data_ptr, d_cls.data_ptr, d_pos.data_ptr, out.data_ptr, 3, 7, 40, None)
    exp = np.concatenate([np.broadcast_to(cls, (3, 1, 40)), emb], axis=1) + pos[None]
    assert np.array_equal(out.numpy(), exp.astype(np.float32))


@pytest.mark.parametrize("B,C,H,W,p,D,bias", [
    (3, 3, 32, 48, 16, 40, True),      # less than one tile either way
    (5, 3, 96, 96, 16, 200, True),     # 180 patch rows: a ragged second row tile, images straddling tiles
    (2, 1, 30, 18, 6, 130, False),     # patch not a multiple of 4: the element-by-element gather
    (1, 2, 8, 8, 4, 8, True),
    (2, 3, 12, 20, 4, 24, True),       # K = 48: a partial k tile
    (64, 3, 224, 224, 16, 768, True),  # ViT-B/16 at the bench batch
])
def test_patch_embedding_in_one_launch_equals_the_three_steps(B, C, H, W, p, D, bias):
    """lq_patch_embed_f32 against lq_patchify_f32 -> lq_sgemm_nt_f32 -> lq_assemble_tokens_f32
    bit for bit (same products, same summation order), and the chain's gather and
    assembly against numpy above."""
    rng = np.random.default_rng(B * 1000 + D)
    n, K = (H // p) * (W // p), C * p * p
    img = hip(rng.standard_normal((B, C, H, W)).astype(np.float32))
    w = hip((rng.standard_normal((D, K)) / np.sqrt(K)).astype(np.float32))
    bv = hip(rng.standard_normal(D).astype(np.float32)) if bias else None
    cls = hip(rng.standard_normal(D).astype(np.float32))
    pos = hip(rng.standard_normal((n + 1, D)).astype(np.float32))
    rows = L.Tensor.empty((B * n, K), L.float32, "hip")
    _C.call("lq_patchify_f32", img.data_ptr, rows.data_ptr, B, C, H, W, p, None)
    emb = F.linear_f32(rows, w, bv)
    exp = L.Tensor.empty((B, n + 1, D), L.float32, "hip")
    _C.call("lq_assemble_tokens_f32", emb.data_ptr, cls.data_ptr, pos.data_ptr, exp.data_ptr, B, n + 1, D, None)
    got = L.tensor(np.full((B, n + 1, D), np.nan, np.float32), device="hip")
    _C.call("lq_patch_embed_f32", img.data_ptr, w.data_ptr, bv.data_ptr if bias else None, cls.data_ptr,
            pos.data_ptr, got.data_ptr, B, C, H, W, p, D, None)
    assert np.array_equal(got.numpy(), exp.numpy())


def test_patch_embedding_of_an_image_that_is_not_16_byte_aligned():
    """The aligned-load form needs a 16-byte aligned image; one that starts 4 bytes further takes
    the element-by-element gather and gives the same bits."""
    rng = np.random.default_rng(12)
    B, C, H, W, p, D = 2, 3, 32, 32, 16, 40
    n, K = 4, C * p * p
    flat = hip(rng.standard_normal(B * C * H * W + 1).astype(np.float32))
    shifted = L.Tensor((B, C, H, W), L.float32, "hip", buf=flat._buf, offset=flat._offset + 4)
    aligned = hip(flat.numpy()[1:].reshape(B, C, H, W).copy())
    w = hip((rng.standard_normal((D, K)) / np.sqrt(K)).astype(np.float32))
    bv, cls = hip(rng.standard_normal(D).astype(np.float32)), hip(rng.standard_normal(D).astype(np.float32))
    pos = hip(rng.standard_normal((n + 1, D)).astype(np.float32))
    outs = []
    for img in (shifted, aligned):
        assert (img.data_ptr % 16 == 0) == (img is aligned)
        out = L.tensor(np.full((B, n + 1, D), np.nan, np.float32), device="hip")
        _C.call("lq_patch_embed_f32", img.data_ptr, w.data_ptr, bv.data_ptr, cls.data_ptr, pos.data_ptr, out.data_ptr,
                B, C, H, W, p, D, None)
        outs.append(out.numpy())
    assert np.array_equal(outs[0], outs[1]) and np.isfinite(outs[0]).all()


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (1, 33, 4), (31, 32, 31), (32, 31, 32), (33, 65, 33), (65, 64, 128), (64, 96, 132),
                                   (200, 40, 97), (1600, 1664, 36), (1632, 1664, 36), (2689, 1152, 40), (4096, 3073, 68),
                                   (2660, 3457, 68), (3000, 3200, 33)])
@pytest.mark.parametrize("shift", [0, 1])
def test_float_gemm_of_any_size(M, N, K, shift):
    """Both tile sizes (2600 tiles of 32 x 32 are the line; 588 large tiles run three per CU), K of whole and partial turns, rows
    that are no 16 bytes, operands that begin at none: within the roundings of the additions, each at most
    2^-24 of the sum of the terms' magnitudes (six per 16 k, the halves and wavefronts, the product's own and the bias)."""
    rng = np.random.default_rng(M + N + K)
    flat = [rng.standard_normal(n + shift).astype(np.float32) for n in (M * K, N * K)]
    bias = rng.standard_normal(N).astype(np.float32)
    a, w = (L.Tensor(s, L.float32, "hip", buf=hip(f)._buf, offset=4 * shift) for f, s in zip(flat, ((M, K), (N, K))))
    out, bv = L.tensor(np.full((M, N), np.nan, np.float32), device="hip"), hip(bias)
    _C.call("lq_sgemm_nt_f32", a.data_ptr, w.data_ptr, bv.data_ptr, out.data_ptr, M, N, K, None)
    a64, w64 = (f[shift:].reshape(s).astype(np.float64) for f, s in zip(flat, ((M, K), (N, K))))
    bound = (6 * ((K + 15) // 16) + 12) * 2.0 ** -24 * (np.abs(a64) @ np.abs(w64).T + np.abs(bias))
    assert (np.abs(out.numpy() - (a64 @ w64.T + bias)) <= bound).all()


@pytest.mark.parametrize("M,N,K,shift", [(2300, 1147, 1155, 0), (1990, 1027, 259, 0), (1600, 1152, 256, 1), (2300, 1147, 36, 1)])
def test_float_gemm_of_unaligned_rows_leaves_the_small_tiles_sooner(M, N, K, shift):
    """More than 2000 tiles of 32 x 32 (1500 at addresses between 16 bytes): the sums are those of the large tiles, which a
    problem of more rows takes anyway.  M and N are below the line of aligned rows."""
    rng = np.random.default_rng(K)
    a, w = (hip(rng.standard_normal(n + shift).astype(np.float32)) for n in (4000 * K, N * K))
    outs = [L.Tensor.empty((m, N), L.float32, "hip") for m in (M, 4000)]
    for o in outs:
        _C.call("lq_sgemm_nt_f32", a.data_ptr + 4 * shift, w.data_ptr + 4 * shift, None, o.data_ptr, o.shape[0], N, K, None)
    assert -(-M // 32) * -(-N // 32) <= 2600 and np.array_equal(outs[0].numpy(), outs[1].numpy()[:M])


@pytest.mark.parametrize("B,C,H,W,p,D", [(33, 1, 40, 40, 4, 2561), (27, 3, 33, 33, 3, 2560), (34, 1, 60, 60, 6, 2500)])
def test_patch_embedding_on_tiles_that_run_three_per_cu(B, C, H, W, p, D):
    """513 to 768 tiles of 128 x 128 (pixels by aligned quads, one by one, and beside an aligned weight): within the roundings
    of the additions, as for the float GEMM, with one more for the position."""
    rng = np.random.default_rng(D)
    n, K = (H // p) * (W // p), C * p * p
    assert 512 < -(-B * n // 128) * -(-D // 128) <= 768
    img = rng.standard_normal((B, C, H, W)).astype(np.float32)
    w, bias, cls, pos = (rng.standard_normal(s).astype(np.float32) for s in ((D, K), (D,), (D,), (n + 1, D)))
    out = L.tensor(np.full((B, n + 1, D), np.nan, np.float32), device="hip")
    held = [hip(v) for v in (img, w, bias, cls, pos)]
    _C.call("lq_patch_embed_f32", *[t.data_ptr for t in held], out.data_ptr, B, C, H, W, p, D, None)
    rows, got = V.patch_rows(img, p).astype(np.float64), out.numpy()
    exact = (rows @ w.T.astype(np.float64)).reshape(B, n, D) + bias + pos[1:].astype(np.float64)
    size = (np.abs(rows) @ np.abs(w).T.astype(np.float64)).reshape(B, n, D) + np.abs(bias) + np.abs(pos[1:])
    assert (np.abs(got[:, 1:] - exact) <= (6 * ((K + 15) // 16) + 13) * 2.0 ** -24 * size).all()
    assert np.array_equal(got[:, 0], np.broadcast_to(cls + pos[0], (B, D)))


def test_patch_embedding_refuses_a_ragged_image():
    z = L.Tensor.empty((1, 3, 20, 32), L.float32, "hip")
    o = L.Tensor.empty((1, 3, 8), L.float32, "hip")
    with pytest.raises(Exception, match="whole number"):
        _C.call("lq_patch_embed_f32", z.data_ptr, z.data_ptr, None, z.data_ptr, z.data_ptr, o.data_ptr,
                1, 3, 20, 32, 16, 8, None)


SMALL = dict(image=64, patch=16, dim=128, depth=2, heads=2, mlp=256, classes=10)


def test_vit_b16_block_stage_by_stage():
    """Every step of a ViT-B/16 block fed with the CPU path's own input for that
    step: the quantized Linears are bit-exact, the float32 steps agree to
    rounding order."""
    cfg = workloads.VIT_B16
    p = workloads.vit_float_params(cfg, seed=4)
    rng = np.random.default_rng(11)
    images = rng.uniform(0, 1, (2, 3, 224, 224)).astype(np.float32)
    model = workloads.QViT(cfg, params=p)
    st = {}
    V.vit_forward(p, images, cfg, stages=st)
    blk = model.blocks[0]
    tok, b = st["tokens"], "blocks.0."
    h = V.layer_norm(tok, p[b + "norm1.weight"], p[b + "norm1.bias"], 1e-6)
    assert rel(blk.norm1(hip(tok)).numpy(), h) < 1e-5
    wq, ws = V.quantize_weight(p[b + "qkv.weight"])
    assert np.array_equal(blk.qkv.weight_int8.numpy(), wq) and np.array_equal(blk.qkv.weight_scale.numpy(), ws)
    qkv = V.dynamic_linear(h, wq, ws, p[b + "qkv.bias"])
    assert np.array_equal(blk.qkv(hip(h)).numpy(), qkv)
    a = V.attention_qkv(qkv, cfg["heads"])
    assert rel(F.scaled_dot_product_attention_qkv(hip(qkv), cfg["heads"]).numpy(), a) < 1e-5
    wq, ws = V.quantize_weight(p[b + "proj.weight"])
    pr = V.dynamic_linear(a, wq, ws, p[b + "proj.bias"])
    assert np.array_equal(blk.proj(hip(a)).numpy(), pr)
    x1 = (tok + pr).astype(np.float32)
    h2 = V.layer_norm(x1, p[b + "norm2.weight"], p[b + "norm2.bias"], 1e-6)
    wq, ws = V.quantize_weight(p[b + "fc1.weight"])
    f1 = V.dynamic_linear(h2, wq, ws, p[b + "fc1.bias"])
    assert np.array_equal(blk.fc1(hip(h2)).numpy(), f1)
    ge = V.gelu(f1)
    assert np.max(np.abs(F.gelu(hip(f1)).numpy() - ge)) <= 2e-6
    wq, ws = V.quantize_weight(p[b + "fc2.weight"])
    assert np.array_equal(blk.fc2(hip(ge)).numpy(), V.dynamic_linear(ge, wq, ws, p[b + "fc2.bias"]))


# bound = twice the error measured on MI355X for that configuration (1.35e-7 and 1.82e-2)
@pytest.mark.parametrize("cfg,batch,bound", [(SMALL, 3, 3e-7), (workloads.VIT_B16, 2, 3.7e-2)])
def test_vit_end_to_end_against_the_cpu_path(cfg, batch, bound):
    """Free-running comparison.  A dynamic quantizer turns an input difference d
    (here float32 rounding order, 1e-7) into an RMS difference of sqrt(d * step)
    on the elements that cross a rounding tie, so after a few layers two correct
    implementations differ at the level of the quantization step itself
    (~0.4 % of the activation range per layer); the bound of the 12-layer model is that
    level, not a rounding-error bound, while the 2-layer model stays at rounding level.
    Stage-by-stage parity is the test above."""
    p = workloads.vit_float_params(cfg, seed=4)
    rng = np.random.default_rng(11)
    images = rng.uniform(0, 1, (batch, 3, cfg["image"], cfg["image"])).astype(np.float32)
    model = workloads.QViT(cfg, params=p)
    got = model(hip(images)).numpy()
    exp = V.vit_forward(p, images, cfg)
    assert got.shape == exp.shape == (batch, cfg["classes"])
    err = rel(got, exp)
    print(f"ViT dim {cfg['dim']} depth {cfg['depth']} batch {batch}: end-to-end max error / max |logit| = {err:.2e}")
    assert err < bound


def _range_of(t):
    """(min, max) a dynamic quantizer would derive from the tensor's kept range."""
    s = L.Tensor.empty((), L.float32, "hip")
    z = L.Tensor.empty((), L.float32, "hip")
    mn = L.Tensor.empty((), L.float32, "hip")
    mx = L.Tensor.empty((), L.float32, "hip")
    _C.call("lq_calc_qparams_from_range", t._range.data_ptr, 0, 0, 255, 0, 1e-8, s.data_ptr, z.data_ptr,
            mn.data_ptr, mx.data_ptr, None)
    return mn.numpy(), mx.numpy(), s.numpy(), z.numpy()


@pytest.mark.parametrize("rows,cols", [(12608, 768), (5, 33), (17, 1000)])
def test_kept_ranges_equal_a_separate_minmax_pass(rows, cols):
    import lucid_amd.quantization as Q

    rng = np.random.default_rng(rows * 3 + cols)
    x = (rng.standard_normal((rows, cols)) * 3 - 0.5).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    b = (0.1 * rng.standard_normal(cols)).astype(np.float32)
    for out in (F.layer_norm(hip(x), cols, hip(g), hip(b), 1e-6, track_range=True),
                F.gelu(hip(x), track_range=True)):
        mn, mx = Q.minmax(out)
        s, z = Q.calculate_qparams(mn, mx, Q.per_tensor_affine, Q.quint8)
        kmn, kmx, ks, kz = _range_of(out)
        y = out.numpy()
        assert kmn == y.min() == mn.numpy() and kmx == y.max() == mx.numpy()
        assert ks.tobytes() == s.numpy().tobytes() and kz.tobytes() == z.numpy().tobytes()


def test_kept_range_of_attention_and_nan_propagation():
    rng = np.random.default_rng(2)
    qkv = rng.standard_normal((3, 197, 3 * 12 * 64)).astype(np.float32)
    out = F.scaled_dot_product_attention_qkv(hip(qkv), 12, track_range=True)
    kmn, kmx, _, _ = _range_of(out)
    y = out.numpy()
    assert kmn == y.min() and kmx == y.max()
    x = rng.standard_normal((64, 256)).astype(np.float32)
    x[17, 5] = np.nan
    kmn, kmx, ks, _ = _range_of(F.gelu(hip(x), track_range=True))
    assert np.isnan(kmn) and np.isnan(kmx) and np.isnan(ks)  # Reduce.cpp:87-125 propagates NaN


@pytest.mark.parametrize("M,K,N", [(12608 // 8, 768, 3072), (300, 96, 200), (129, 64, 72)])
def test_gelu_and_kept_range_in_the_gemm_epilogue(M, K, N):
    """fc1 -> GELU fused: the bits of linear followed by the stand-alone GELU kernel, and the
    kept range gives the qparams that min / max of the result give."""
    import lucid_amd.nn as nn
    import lucid_amd.nn.functional as F
    import lucid_amd.quantization as Q
    from lucid_amd import _C
    rng = np.random.default_rng(M + N)
    lin = nn.Linear(K, N)
    q = Q.quantize_dynamic(nn.Sequential(lin))[0]
    x = L.tensor(rng.standard_normal((M, K)).astype(np.float32), device="hip")
    want = F.gelu(q(x)).numpy()
    fused = q(x, activation="gelu", track_range=True)
    got = fused.numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    s = L.Tensor.empty((), L.float32, "hip")
    z = L.Tensor.empty((), L.float32, "hip")
    _C.call("lq_calc_qparams_from_range", fused._range.data_ptr, 0, 0, 255, 0, 1e-8, s.data_ptr, z.data_ptr,
            None, None, None)
    ws, wz = O.calc_qparams(np.float32([want.min()]), np.float32([want.max()]), False, 0, 255, False)
    assert s.numpy() == ws[0] and z.numpy() == wz[0]


def test_vit_block_fused_and_unfused_gelu_agree(monkeypatch):
    import workloads as W
    cfg = dict(W.VIT_B16, depth=1, dim=192, heads=3, mlp=768)
    model = W.QViT(cfg, seed=3)
    x = L.tensor(np.random.default_rng(0).standard_normal((2, 3, 224, 224)).astype(np.float32), device="hip")
    a = model(x).numpy()
    monkeypatch.setattr(W.ViTBlock, "fuse_gelu", False)
    b = model(x).numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(394, 768), (12608, 768), (5, 192), (7, 2048), (64, 4), (1, 4),
                                       (2048, 64), (2049, 64), (2050, 1028)])
def test_layernorm_dynamic_quantize_equals_layernorm_then_quantize(rows, cols):
    """LayerNorm that writes the next dynamic Linear's codes directly: codes, scale and zero
    point are the bits of layer_norm(track_range) + calc_qparams_from_range + quantize."""
    from lucid_amd import _C
    import lucid_amd.quantization as Q
    rng = np.random.default_rng(rows + cols)
    x = (rng.standard_normal((rows, cols)) * 2 + 0.3).astype(np.float32)
    g = (1 + 0.1 * rng.standard_normal(cols)).astype(np.float32)
    b = (0.1 * rng.standard_normal(cols)).astype(np.float32)
    xt, gt, bt = hip(x), hip(g), hip(b)
    fused = F.layer_norm_dynamic_quantize(xt, cols, gt, bt, 1e-6, Q.quint8)
    assert fused is not None
    q, s, z = fused
    y = F.layer_norm(xt, cols, gt, bt, 1e-6, track_range=True)
    s2, z2 = L.Tensor.empty((), L.float32, "hip"), L.Tensor.empty((), L.float32, "hip")
    _C.call("lq_calc_qparams_from_range", y._range.data_ptr, 0, 0, 255, 0, 1e-8, s2.data_ptr, z2.data_ptr, None, None,
            None)
    q2 = L.Tensor.empty((rows, cols), L.int8, "hip")
    _C.call("lq_quantize", y.data_ptr, q2.data_ptr, _C.I8, -128, 1, 1, rows * cols, s2.data_ptr, z2.data_ptr, 0, 0, 255,
            None)
    assert np.array_equal(s.numpy().view(np.uint32), s2.numpy().view(np.uint32))
    assert np.array_equal(z.numpy().view(np.uint32), z2.numpy().view(np.uint32))
    assert np.array_equal(q.numpy(), q2.numpy())


def test_layernorm_dynamic_quantize_declines_other_rows():
    import lucid_amd.quantization as Q
    x = hip(np.zeros((4, 2052), np.float32))
    w = hip(np.ones(2052, np.float32))
    assert F.layer_norm_dynamic_quantize(x, 2052, w, w, 1e-6, Q.quint8) is None


@pytest.mark.parametrize("n", [1, 3, 4, 5, 8191, 8192, 8195, 1 << 22, (1 << 22) + 2])  # tails, one block and one more, one launch and two
@pytest.mark.parametrize("nan", [False, True])
def test_codes_straight_from_a_kept_range(n, nan):
    """``lq_quantize_from_range_i8`` writes the scale, zero point and codes of the two calls it stands for."""
    from lucid_amd.nn.functional import _new_range
    rng = np.random.default_rng(n)
    a = (rng.standard_normal(n) * 3 + 1).astype(np.float32)
    if nan:
        a[n // 2] = np.nan
    x = L.tensor(a, device="hip")
    y, kept = L.Tensor.empty((n,), L.float32, "hip"), _new_range()
    _C.call("lq_gelu_f32", x.data_ptr, y.data_ptr, n, kept.data_ptr, None)
    one, two = [[L.Tensor.empty((), L.float32, "hip"), L.Tensor.empty((), L.float32, "hip"), L.Tensor.empty((n,), L.int8, "hip")]
                for _ in range(2)]
    _C.call("lq_calc_qparams_from_range", kept.data_ptr, 0, 0, 255, 0, 1e-8, one[0].data_ptr, one[1].data_ptr, None, None, None)
    _C.call("lq_quantize", y.data_ptr, one[2].data_ptr, _C.I8, -128, 1, 1, n, one[0].data_ptr, one[1].data_ptr, 0, 0, 255, None)
    _C.call("lq_quantize_from_range_i8", y.data_ptr, n, kept.data_ptr, 0, 0, 255, 0, 1e-8, -128, two[0].data_ptr,
            two[1].data_ptr, two[2].data_ptr, None)
    for a1, a2 in zip(one, two):
        assert a1.numpy().tobytes() == a2.numpy().tobytes()
    if n > 8:  # an address that vectors cannot take
        _C.call("lq_quantize", y.data_ptr + 4, one[2].data_ptr, _C.I8, -128, 1, 1, n - 1, one[0].data_ptr, one[1].data_ptr, 0, 0,
                255, None)
        _C.call("lq_quantize_from_range_i8", y.data_ptr + 4, n - 1, kept.data_ptr, 0, 0, 255, 0, 1e-8, -128, two[0].data_ptr,
                two[1].data_ptr, two[2].data_ptr, None)
        assert np.array_equal(one[2].numpy()[:n - 1], two[2].numpy()[:n - 1])


@pytest.mark.parametrize("n", [1, 63, 511, 512, 513, 1024, 1025, 4096, 4097, 16384])
@pytest.mark.parametrize("nan", [False, True])
def test_range_of_any_number_of_slots(n, nan):
    """The first slots of a range are read before their number is known: what lies past it (here NaNs, beyond any other value)
    does not count, the last slot does, whether it is among the first ones or not - for all three readers of a range."""
    import lucid_amd.quantization as Q
    rng = np.random.default_rng(n)
    words = _C.range_buffer_words()
    slots = (words - 4) // 2
    buf = np.full(words, np.nan, np.float32)
    buf[:1].view(np.uint32)[0] = n
    lo, hi = -rng.random(n).astype(np.float32), rng.random(n).astype(np.float32)
    lo[-1], hi[n // 2] = -2, 3
    if nan:
        lo[-1] = hi[-1] = np.nan
    buf[4:4 + n], buf[4 + slots:4 + slots + n] = lo, hi
    r, f32 = L.tensor(buf, device="hip"), lambda: L.Tensor.empty((), L.float32, "hip")
    x, w = (L.tensor(rng.standard_normal(m).astype(np.float32), device="hip") for m in (4096, 64))
    q = L.Tensor.empty((4096,), L.int8, "hip")
    mn, mx, sz = f32(), f32(), [(f32(), f32()) for _ in range(3)]
    args = (0, 0, 255, 0, 1e-8)
    _C.call("lq_calc_qparams_from_range", r.data_ptr, *args, *(v.data_ptr for v in sz[0]), mn.data_ptr, mx.data_ptr, None)
    _C.call("lq_quantize_from_range_i8", x.data_ptr, 4096, r.data_ptr, *args, -128, *(v.data_ptr for v in sz[1]), q.data_ptr, None)
    stats = L.tensor(np.tile(np.float32([0, 1]), 64), device="hip")
    _C.call("lq_layernorm_quantize_from_range_i8", x.data_ptr, w.data_ptr, w.data_ptr, stats.data_ptr, 64, 64, r.data_ptr, *args,
            -128, *(v.data_ptr for v in sz[2]), q.data_ptr, None)
    if nan:
        assert np.isnan(mn.numpy()) and np.isnan(mx.numpy()) and all(np.isnan(s.numpy()) for s, _ in sz)
    else:
        assert mn.numpy() == -2 and mx.numpy() == hi.max()
        want = Q.calculate_qparams(mn, mx, Q.per_tensor_affine, Q.quint8)
        for s, z in sz:
            assert s.numpy().tobytes() == want[0].numpy().tobytes() and z.numpy().tobytes() == want[1].numpy().tobytes()


def test_layernorm_codes_of_no_rows_still_give_the_qparams():
    """``lq_layernorm_quantize_from_range_i8`` stands for two calls, of which the first does not look at the rows."""
    from lucid_amd.nn.functional import _new_range
    rng = np.random.default_rng(3)
    x, w = (L.tensor(rng.standard_normal(n).astype(np.float32), device="hip") for n in (64, 64))
    kept, stats, q = _new_range(), L.Tensor.empty((2,), L.float32, "hip"), L.Tensor.empty((64,), L.int8, "hip")
    _C.call("lq_gelu_f32", x.data_ptr, x.data_ptr, 64, kept.data_ptr, None)
    want, got = ([L.tensor(np.float32(-7), device="hip") for _ in range(2)] for _ in range(2))
    _C.call("lq_calc_qparams_from_range", kept.data_ptr, 0, 0, 255, 0, 1e-8, *(t.data_ptr for t in want), None, None, None)
    _C.call("lq_layernorm_quantize_from_range_i8", x.data_ptr, w.data_ptr, w.data_ptr, stats.data_ptr, 0, 64, kept.data_ptr, 0, 0,
            255, 0, 1e-8, -128, *(t.data_ptr for t in got), q.data_ptr, None)
    assert [t.numpy().tobytes() for t in got] == [t.numpy().tobytes() for t in want]


def test_vit_block_with_and_without_fused_layernorm_quantize_agree(monkeypatch):
    import workloads as W
    cfg = dict(W.VIT_B16, depth=2, dim=192, heads=3, mlp=768)
    model = W.QViT(cfg, seed=4)
    x = L.tensor(np.random.default_rng(1).standard_normal((2, 3, 224, 224)).astype(np.float32), device="hip")
    a = model(x).numpy()
    monkeypatch.setattr(W.ViTBlock, "fuse_ln_quant", False)
    b = model(x).numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
