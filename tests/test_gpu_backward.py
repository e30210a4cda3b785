"""Backward of the varlen and dense ops vs autograd through the CPU oracle's forward (the reference's contract:
``areno/accel/attention.py:104-118,170-183`` call native backward kernels, ``csrc/attention.cu:244-524``, which return
fp32 gradients cast to the inputs' dtypes).

Bar: the gradients are sums of 16-bit inputs accumulated in fp32 and cast back to the input dtype, so they are compared
relative to the largest gradient of the tensor: 3e-2 for bf16, 1e-2 for fp16 (one or two units of the output
format's rounding at that magnitude, plus the rounding of the saved output that both this build and the reference
use for dO . O), 1e-4 for fp32."""

import ctypes
import math

import pytest
import torch

from areno_amd.accel import attention as ops
from areno_amd.accel import cabi
from oracle import attention_ref as ar
from tests.gpu_util import DEV

pytestmark = pytest.mark.gpu

REL = {torch.bfloat16: 3e-2, torch.float16: 1e-2, torch.float32: 1e-4}


def _close(got, want, rel, what):
    got, want = got.detach().cpu().float(), want.detach().float()
    assert torch.isfinite(got).all(), f"{what}: non-finite gradient"
    err = (got - want).abs().max().item()
    bound = rel * max(want.abs().max().item(), 1e-3)
    assert err <= bound, f"{what}: max-abs {err:.4g} > {bound:.4g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("window_left", [None, 0, 9])
@pytest.mark.parametrize("hq,hkv,d", [(8, 2, 64), (6, 3, 128), (4, 4, 192), (4, 1, 256), (4, 4, 80), (4, 1, 96), (2, 1, 8), (6, 2, 200)])
def test_varlen_backward(dtype, window_left, hq, hkv, d):
    g = torch.Generator().manual_seed(hq * 17 + d)
    lens = [5, 1, 70, 0, 33]
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    q = torch.randn(t, hq, d, generator=g).to(dtype)
    k = torch.randn(t, hkv, d, generator=g).to(dtype)
    v = torch.randn(t, hkv, d, generator=g).to(dtype)
    go = torch.randn(t, hq, d, generator=g).to(dtype)
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    out = ops.areno_varlen_causal_attention(qd, kd, vd, cu.to(DEV), window_left=window_left)
    assert out.requires_grad
    out.backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    want = ar.ref_varlen(qf, kf, vf, cu, ar.window_left_arg(window_left), d**-0.5)
    want.backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        assert got.dtype == dtype and got.shape == ref.shape
        _close(got, ref, REL[dtype], f"{name} {dtype} d={d} window={window_left}")


@pytest.mark.parametrize("last", [129, 161])
@pytest.mark.parametrize("parts,dq_rows", [("1", "16"), ("2", "32"), ("4", "16"), ("4", "32")])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,window_left", [(8, 2, 128, None), (4, 4, 64, None), (6, 1, 64, 40), (4, 2, 128, 200), (2, 1, 128, 0)])
def test_varlen_backward_long_sequences_on_the_matrix_core_kernels(dtype, hq, hkv, d, window_left, parts, dq_rows, last, monkeypatch):
    """16-bit inputs at head dims 64 / 128 take the matrix-core backward: sequences longer than its blocks (of 64 or 128
    query rows, of 128, 64 or 32 keys) and tiles of 32, blocks that hold several sequences (and empty ones), query groups,
    windows shorter and longer than a tile.  The dkv kernel in three of its shapes: key blocks of 128 rows, of 64 with the
    stream of query tiles in two parts, of 32 with four parts and in pairs (the library reads the variable at every launch;
    left alone it picks by the size of the launch).  The last sequence's length makes the number of 32-row blocks
    even (1 327 tokens: every block has a partner in the four-part shape's pairs) or odd (1 359: the middle one has
    none)."""
    monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)  # the dq kernel with 16 and with 32 query rows per wave
    g = torch.Generator().manual_seed(hq * 31 + d)
    lens = [300, 1, 0, 700, 5, 63, 64, 65, last]
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    q = torch.randn(t, hq, d, generator=g).to(dtype)
    k = torch.randn(t, hkv, d, generator=g).to(dtype)
    v = torch.randn(t, hkv, d, generator=g).to(dtype)
    go = torch.randn(t, hq, d, generator=g).to(dtype)
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    ops.areno_varlen_causal_attention(qd, kd, vd, cu.to(DEV), window_left=window_left).backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    ar.ref_varlen(qf, kf, vf, cu, ar.window_left_arg(window_left), d**-0.5).backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        _close(got, ref, REL[dtype], f"{name} {dtype} {hq}/{hkv} d={d} window={window_left}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,window_left", [(4, 2, 256, None), (6, 2, 256, 70), (3, 3, 192, None), (4, 1, 192, 97), (2, 1, 256, 0)])
@pytest.mark.parametrize("lens", [[300, 1, 0, 130, 5, 95, 97, 161], [127], [129, 31], [1]])
def test_varlen_backward_of_wide_heads_on_the_matrix_core_kernels(dtype, hq, hkv, d, window_left, lens, monkeypatch):
    """Head dims 192 and 256: sequences longer than the dkv kernel's blocks (64 or 32 packed keys), blocks that hold
    several sequences, lengths one off a tile, windows shorter and longer than a block.  The bar is the
    file's."""
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", "16")  # (and not the kernels that a launch's estimate may prefer)
    g = torch.Generator().manual_seed(hq * 31 + d + len(lens))
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype) for h in (hq, hkv, hkv, hq))
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    ops.areno_varlen_causal_attention(qd, kd, vd, cu.to(DEV), window_left=window_left).backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    ar.ref_varlen(qf, kf, vf, cu, ar.window_left_arg(window_left), d**-0.5).backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        _close(got, ref, REL[dtype], f"{name} {dtype} {hq}/{hkv} d={d} window={window_left}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,dq_rows", [(4, 2, 64, "16"), (4, 2, 64, "32"), (4, 2, 128, "16"), (4, 2, 128, "32"), (3, 3, 192, "16"), (2, 1, 256, "16")])
@pytest.mark.parametrize("falling", [False, True])
def test_varlen_backward_where_the_softmax_reference_moves(dtype, hq, hkv, d, dq_rows, falling, monkeypatch):
    """Keys whose scores grow along the sequence (spread 0.2 to 8: by more than 2^8 within a row, several times, and by
    less in other tiles) or fall along it, over an odd number of tiles and a single one: the dq kernel's lazily raised
    reference.  The bar is the file's: the gradients' largest values come from single keys, whose probabilities and
    products round as everywhere."""
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)
    g = torch.Generator().manual_seed(d + falling)
    lens = [321, 30, 0, 65]
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    first, last = (8.0, 0.2) if falling else (0.2, 8.0)
    ramp = torch.cat([torch.linspace(first, last, n) for n in lens])[:, None, None]
    q, k, v, go = (torch.randn(t, h, d, generator=g) for h in (hq, hkv, hkv, hq))
    k = k * ramp
    q, k, v, go = (x.to(dtype) for x in (q, k, v, go))
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    ops.areno_varlen_causal_attention(qd, kd, vd, cu.to(DEV)).backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    ar.ref_varlen(qf, kf, vf, cu, -1, d**-0.5).backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        _close(got, ref, REL[dtype], f"{name} {dtype} d={d} falling={falling}")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("scale", [0.0, -0.05])
@pytest.mark.parametrize("d", [64, 128, 192, 256])
def test_varlen_backward_with_a_scale_that_is_not_positive(dtype, scale, d):
    """The op takes any softmax scale: 0 (every visible key weighs the same) and negative ones (a row's maximum is
    that of its negated products).  Masked keys count for nothing either way.  The bar is the file's."""
    g = torch.Generator().manual_seed(d)
    lens = [130, 0, 33]
    t = sum(lens)
    cu = torch.tensor([0, 130, 130, 163], dtype=torch.int32)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype) for h in (4, 2, 2, 4))
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    ops.areno_varlen_causal_attention(qd, kd, vd, cu.to(DEV), softmax_scale=scale).backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    ar.ref_varlen(qf, kf, vf, cu, -1, scale).backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        _close(got, ref, REL[dtype], f"{name} {dtype} d={d} scale={scale}")


def _c_backward(go, q, k, v, out, cu, grad_dtype, scale, window_left=-1, cu_k=None, ctx=None):
    """The C entry on gradient buffers full of NaN: what it leaves unwritten shows."""
    t, hq, d = q.shape
    grads = [torch.full(x.shape, float("nan"), dtype=grad_dtype, device=DEV) for x in (q, k, v)]
    workspace = torch.empty(t * hq * 8, dtype=torch.uint8, device=DEV)
    ptr = lambda x: None if x is None else ctypes.c_void_p(x.data_ptr())  # noqa: E731
    status = cabi.lib().areno_hip_attention_backward_typed(
        *map(ptr, (go, q, k, v, out, *grads)), cabi.dtype_code(grads[0]), cabi.dtype_code(q), ctypes.c_int64(t),
        ctypes.c_int64(k.shape[0]), hq, k.shape[1], d, ptr(cu), ptr(cu_k), ptr(ctx), cu.numel() - 1, window_left, ctypes.c_float(scale),
        ptr(workspace), ctypes.c_size_t(workspace.numel()), ctypes.c_void_p(cabi.current_stream_ptr()))  # fmt: skip
    cabi.check(status, "areno_hip_attention_backward_typed")
    return grads


@pytest.mark.parametrize("d,dq_rows", [(64, "16"), (64, "32"), (128, "16"), (128, "32"), (192, "16"), (256, "16"), (96, "16")])
@pytest.mark.parametrize("dtype,grad_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("behind", [1, 70, 300])
def test_gradients_of_rows_behind_the_last_sequence_are_zeros(d, dq_rows, dtype, grad_dtype, behind, monkeypatch):
    """A padded pack: its rows behind the last sequence get zeros, the others the gradients that they have without the
    padding, bit for bit (every row has one owner, which does the same for it)."""
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)
    g = torch.Generator().manual_seed(d + behind)
    t, hq, hkv = 163, 4, 2
    padded = [torch.randn(t + behind, h, d, generator=g).to(dtype).to(DEV) for h in (hq, hq, hkv, hkv, hq)]
    plain = [x[:t].contiguous() for x in padded]
    cu = torch.tensor([0, 130, 130, 163], dtype=torch.int32, device=DEV)
    for got, want in zip(_c_backward(*padded, cu, grad_dtype, d**-0.5), _c_backward(*plain, cu, grad_dtype, d**-0.5)):
        assert torch.isfinite(want).all()
        assert torch.equal(got[:t], want)
        assert (got[t:] == 0).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d", [(32, 1, 256), (8, 1, 192), (4, 4, 256), (16, 4, 192)])
@pytest.mark.parametrize("lens", [[1], [1] * 64, [2, 0, 1] * 100, [4] * 200, [8] * 30, [16] * 8, [32] * 4, [1] * 30 + [200]])
def test_many_short_sequences_of_wide_heads(dtype, hq, hkv, d, lens):
    """Launches on either side of the estimate that sends short sequences of wide heads to the vector-ALU kernels.  The
    bar is the file's."""
    g = torch.Generator().manual_seed(d + hq)
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype) for h in (hq, hkv, hkv, hq))
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    ops.areno_varlen_causal_attention(qd, kd, vd, cu.to(DEV)).backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    ar.ref_varlen(qf, kf, vf, cu, -1, d**-0.5).backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        _close(got, ref, REL[dtype], f"{name} {dtype} {hq}/{hkv} d={d} lens={lens[:3]}")


def _gradients_in_64_bits(go, q, k, v, out, lens, window_left, scale):
    """dQ, dK, dV of the packed op from the output that the forward saved (whose rounding is not the backward's)."""
    go, q, k, v, out = (x.double().cpu() for x in (go, q, k, v, out))
    grads = [torch.zeros_like(x) for x in (q, k, v)]
    group, at = q.shape[1] // k.shape[1], 0
    for n in lens:
        rows, i = slice(at, at + n), torch.arange(n)
        at += n
        seen = (i[None] <= i[:, None]) & (i[None] >= i[:, None] - (n if window_left is None else window_left))
        for h in range(q.shape[1]):
            qh, kh, vh, gh = q[rows, h], k[rows, h // group], v[rows, h // group], go[rows, h]
            prob = torch.softmax((scale * qh @ kh.T).masked_fill(~seen, float("-inf")), -1)
            ds = prob * (gh @ vh.T - (gh * out[rows, h]).sum(-1, keepdim=True))
            grads[0][rows, h] = scale * ds @ kh
            grads[1][rows, h // group] += scale * ds.T @ qh
            grads[2][rows, h // group] += prob.T @ gh
    return grads


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hq,hkv,d,window_left", [(4, 2, 256, None), (3, 3, 192, 70), (4, 1, 192, None), (2, 1, 256, 40), (2, 1, 200, None)])
@pytest.mark.parametrize("size", [1.0, 2.0**-12, 2.0**12])
@pytest.mark.parametrize("fixed", [True, False])
def test_wide_heads_keep_their_weights_in_32_bits(dtype, hq, hkv, d, window_left, size, fixed, monkeypatch):
    """Head dims above 128 with gradients in fp32: probabilities and dS are not rounded to 16 bits on the way (2e-4 and
    more would show), nor limited to fp16's range (a loss scaled up or down).  The bar, in the 2-norm: a score of up
    to 2^4 in the exponent and its sum over 256 products put 2^4 * 2^-24 * a few on every weight, 4e-6."""
    if fixed:  # on the matrix cores
        monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", "16")
    g = torch.Generator().manual_seed(d + hq)
    lens = [300, 1, 0, 131]
    t = sum(lens)
    cu = torch.tensor([0, 300, 301, 301, 432], dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype).to(DEV) for h in (hq, hkv, hkv, hq))
    go = go * size
    out = ops.areno_varlen_causal_attention(q, k, v, cu, window_left=window_left)
    got = _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5, -1 if window_left is None else window_left)
    for x, want, name in zip(got, _gradients_in_64_bits(go, q, k, v, out, lens, window_left, d**-0.5), ("dq", "dk", "dv")):
        err = ((x.cpu().double() - want).norm() / want.norm()).item()
        assert err <= 4e-6, f"{name} {dtype} d={d} window={window_left} size={size}: {err:.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("parts", ["1", "2", "4", None])
@pytest.mark.parametrize("hq,hkv,d,window_left", [(4, 1, 128, None), (2, 2, 128, 33), (8, 2, 64, None), (3, 3, 64, 31)])
@pytest.mark.parametrize("lens,scale", [([31, 33, 32, 97, 128, 129], 0.1), ([1], 0.1), ([161, 0, 1, 2, 95], 2.0), ([64, 65, 63], 1e-3), ([33], 1e-37)])
def test_key_gradients_where_blocks_and_tiles_end(dtype, parts, hq, hkv, d, window_left, lens, scale, monkeypatch):
    """The dkv kernel of head dims 64 and 128 in each of its shapes and as the launch's size picks them: sequences one off
    its blocks (32, 64, 128 keys) and tiles, windows one off a tile, small and large scales.  The bar, in the 2-norm: P and dS are rounded to the inputs' type, by half a unit
    in the last place at most; one unit."""
    if parts is not None:
        monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    g = torch.Generator().manual_seed(d + len(lens))
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype).to(DEV) for h in (hq, hkv, hkv, hq))
    out = ops.areno_varlen_causal_attention(q, k, v, cu, window_left=window_left, softmax_scale=scale)
    got = _c_backward(go, q, k, v, out, cu, torch.float32, scale, -1 if window_left is None else window_left)
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for x, want, name in zip(got, _gradients_in_64_bits(go, q, k, v, out, lens, window_left, scale), ("dq", "dk", "dv")):
        err = (x.cpu().double() - want).norm().item()
        assert err <= unit * max(want.norm().item(), scale), f"{name} {dtype} {hq}/{hkv} d={d} lens={lens}: {err / want.norm().item():.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("parts", ["1w", "4s", None])
@pytest.mark.parametrize("hq,hkv,d,window_left", [(4, 1, 128, None), (16, 16, 128, 33), (8, 2, 64, None), (16, 16, 64, 31)])
@pytest.mark.parametrize("lens", [[31, 33, 32, 97, 128, 129], [1], [161, 0, 1, 2, 95], [40] * 42 + [0, 7, 1]])
def test_key_gradients_of_lone_waves_and_of_single_blocks(dtype, parts, hq, hkv, d, window_left, lens, monkeypatch):
    """The dkv kernel's workgroups of one wave (which a launch of 42 short sequences and 16 kv heads takes by itself) and of four
    parts with a block each, sequences one off blocks and tiles.  The bar is that of the other shapes."""
    if parts is not None:
        monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    g = torch.Generator().manual_seed(d + len(lens))
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype).to(DEV) for h in (hq, hkv, hkv, hq))
    out = ops.areno_varlen_causal_attention(q, k, v, cu, window_left=window_left)
    got = _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5, -1 if window_left is None else window_left)
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for x, want, name in zip(got, _gradients_in_64_bits(go, q, k, v, out, lens, window_left, d**-0.5), ("dq", "dk", "dv")):
        err = (x.cpu().double() - want).norm().item()
        assert err <= unit * max(want.norm().item(), d**-0.5), f"{name} {dtype} {hq}/{hkv} d={d} lens={lens[:6]}: {err / want.norm().item():.3g}"


@pytest.mark.parametrize("parts", ["1w", "1", "2", "4"])
@pytest.mark.parametrize("dq_rows", ["16", "32"])
@pytest.mark.parametrize("d", [64, 128])
def test_probabilities_of_large_scores(d, dq_rows, parts, monkeypatch):
    """Single tokens with integer queries and keys (every sum of their products is exact): P is 1, dO is 1 and dV is what
    the dkv kernel made of P.  Its exponent is a difference of a score and a log-sum-exp of the same size, x, which holds
    the score rounded once (half a unit in the last place, 2^-24 x at most; a quarter more for the exponential and the
    logarithm); then P is rounded to fp16 (2^-11 at most)."""
    monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)
    g = torch.Generator().manual_seed(d)
    t, h, scale = 200, 4, 0.0917
    q, k = (torch.randint(-300, 301, (t, h, d), generator=g).to(torch.float16).to(DEV) for _ in range(2))
    v = torch.randn(t, h, d, generator=g).to(torch.float16).to(DEV)
    cu = torch.arange(t + 1, dtype=torch.int32, device=DEV)
    dv = _c_backward(torch.ones_like(v), q, k, v, v, cu, torch.float32, scale)[2].double()
    x = scale / math.log(2) * (q.double() * k.double()).sum(-1, keepdim=True).abs()
    assert x.max() > 3e4
    assert ((dv - 1).abs() <= 1.25 * math.log(2) * 2.0**-24 * x + 2.0**-11).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("parts", ["1", "2"])
@pytest.mark.parametrize("hq,hkv,d,window_left", [(4, 2, 256, None), (3, 3, 192, 33), (4, 1, 192, None), (2, 1, 256, 31)])
@pytest.mark.parametrize("lens", [[63, 64, 65, 1, 129], [33, 0, 31, 2, 97], [32]])
def test_wide_heads_where_blocks_and_tiles_end(dtype, parts, hq, hkv, d, window_left, lens, monkeypatch):
    """Head dims 192 and 256, the dkv kernel with its stream of tiles in one part and in two: sequences one off blocks of 64
    and 32 rows and off tiles, windows one off a tile.  The bar is that of the 32-bit weights above."""
    monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", "16")  # (and not the kernels that a launch's estimate may prefer)
    g = torch.Generator().manual_seed(d + len(lens))
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype).to(DEV) for h in (hq, hkv, hkv, hq))
    out = ops.areno_varlen_causal_attention(q, k, v, cu, window_left=window_left)
    got = _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5, -1 if window_left is None else window_left)
    for x, want, name in zip(got, _gradients_in_64_bits(go, q, k, v, out, lens, window_left, d**-0.5), ("dq", "dk", "dv")):
        err = ((x.cpu().double() - want).norm() / want.norm()).item()
        assert err <= 4e-6, f"{name} {dtype} {hq}/{hkv} d={d} lens={lens}: {err:.3g}"


@pytest.mark.parametrize("name,value,asked", [("PARTS", "1", True), ("PARTS", "2", True), ("DQ_ROWS", "32", True), ("DQ_ROWS", "48", False), ("PARTS", "4", False)])
@pytest.mark.parametrize("d", [192, 256])
def test_switches_ask_for_the_wide_heads_matrix_core_kernels(d, name, value, asked, monkeypatch):
    """Single tokens of wide heads are the vector-ALU kernels'; a switch with a value that names one of the matrix-core
    kernels' shapes takes them there (other bits come out of it), any other value changes nothing."""
    g = torch.Generator().manual_seed(d)
    t = 64
    cu = torch.tensor(list(range(0, 2 * t, 2)) + [2 * t], dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(2 * t, h, d, generator=g).to(torch.bfloat16).to(DEV) for h in (32, 1, 1, 32))
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    grads = lambda: _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5)  # noqa: E731
    plain = grads()
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", "16")
    matrix = grads()
    assert not torch.equal(plain[1], matrix[1])
    monkeypatch.delenv("ARENO_BACKWARD_DQ_ROWS")
    monkeypatch.setenv(f"ARENO_BACKWARD_{name}", value)
    got = grads()
    assert torch.equal(got[1], plain[1]) != asked
    assert torch.equal(got[0], (matrix if asked else plain)[0])


@pytest.mark.parametrize("seqs", [1, 63, 64, 65, 130])
@pytest.mark.parametrize("dq_rows", ["16", "32"])
@pytest.mark.parametrize("hq,hkv,d,dtype", [(2, 1, 64, torch.float16), (2, 2, 128, torch.bfloat16), (2, 1, 256, torch.bfloat16)])
def test_blocks_find_their_sequence_among_many(seqs, dq_rows, hq, hkv, d, dtype, monkeypatch):
    """A block looks its sequence up 64 at a time: around 64 and 128 of them, empty ones between them and at both ends, and
    more than one block long.  The bar of the 16-bit kernels above, one unit of the inputs' type, in the 2-norm."""
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)
    g = torch.Generator().manual_seed(seqs)
    lens = [(0, 3, 37, 0, 141, 1, 65)[i % 7] for i in range(seqs)] if seqs > 1 else [150]
    t = sum(lens)
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(t, h, d, generator=g).to(dtype).to(DEV) for h in (hq, hkv, hkv, hq))
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    got = _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5)
    unit = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for x, want, name in zip(got, _gradients_in_64_bits(go, q, k, v, out, lens, None, d**-0.5), ("dq", "dk", "dv")):
        err = ((x.cpu().double() - want).norm() / want.norm()).item()
        assert err <= unit, f"{name} {dtype} d={d} seqs={seqs}: {err:.3g}"


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 192), (torch.float16, 256), (torch.bfloat16, 96), (torch.float32, 64)])
@pytest.mark.parametrize("window_left", [2**31 - 1, 2**31 - 100, 2**30, 2**30 - 1])
def test_a_window_as_wide_as_its_type_holds_is_none(dtype, d, window_left):
    """Gradients with the widest windows: those without one, bit for bit (positions and the window are added in 32 bits)."""
    g = torch.Generator().manual_seed(d)
    cu = torch.tensor([0, 70, 73, 273], dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(273, h, d, generator=g).to(dtype).to(DEV) for h in (4, 2, 2, 4))
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    want = _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5)
    assert all(x.abs().max() > 0 for x in want)
    for got, x, name in zip(_c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5, window_left), want, ("dq", "dk", "dv")):
        assert torch.equal(got, x), f"{name} {dtype} d={d} window={window_left}"


def _with_contexts(q, k, v, go, q_lens, k_lens, ctxs, window_left, scale):
    """The forward's output (in the inputs' type) and dQ, dK, dV in 64 bits where sequence s has its queries at positions ctxs[s]
    and on, and keys of its own."""
    unit = q.dtype
    q, k, v, go = (x.double().cpu() for x in (q, k, v, go))
    out, grads, group = torch.zeros_like(q), [torch.zeros_like(x) for x in (q, k, v)], q.shape[1] // k.shape[1]
    q0 = k0 = 0
    for n_q, n_k, ctx in zip(q_lens, k_lens, ctxs):
        rows, keys = slice(q0, q0 + n_q), slice(k0, k0 + n_k)
        q0, k0 = q0 + n_q, k0 + n_k
        i, j = ctx + torch.arange(n_q)[:, None], torch.arange(n_k)[None]
        seen = (j <= i) & (j >= i - (i + 1 if window_left is None else window_left))
        for h in range(q.shape[1]):
            qh, kh, vh, gh = q[rows, h], k[keys, h // group], v[keys, h // group], go[rows, h]
            prob = torch.softmax((scale * qh @ kh.T).masked_fill(~seen, float("-inf")), -1)
            out[rows, h] = (prob @ vh).to(unit).double()
            ds = prob * (gh @ vh.T - (gh * out[rows, h]).sum(-1, keepdim=True))
            grads[0][rows, h] = scale * ds @ kh
            grads[1][keys, h // group] += scale * ds.T @ qh
            grads[2][keys, h // group] += prob.T @ gh
    return out.to(unit).to(DEV), grads


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("window_left", [None, 33, 100])
@pytest.mark.parametrize("hq,hkv,d", [(4, 2, 64), (4, 1, 128), (2, 2, 128), (4, 2, 192), (3, 3, 256)])
@pytest.mark.parametrize("parts,dq_rows", [("1w", "16"), ("1", "16"), ("2", "32"), ("4s", "16"), ("4", "32")])
def test_queries_behind_cached_keys_on_the_matrix_core_kernels(dtype, window_left, hq, hkv, d, parts, dq_rows, monkeypatch):
    """Contexts (fewer queries than keys) in every form of the dq and dkv kernels: queries that start inside a tile, at its edge
    and one off it, in the first and in later blocks of keys, keys behind the last query's position, fewer keys than positions,
    a sequence of keys alone.  The bar, in the 2-norm: P and dS are rounded to the inputs' type, by half a unit in the last
    place at most; one unit (wide heads do not round them: their own bar)."""
    if d > 128 and parts not in ("1", "2"):
        pytest.skip("wide heads have two shapes")
    monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)
    g = torch.Generator().manual_seed(d + hq)
    q_lens, ctxs = [70, 1, 0, 161, 33, 40, 5], [45, 200, 7, 96, 0, 129, 31]
    k_lens = [n + c + more for n, c, more in zip(q_lens, ctxs, (3, 0, 2, 40, 0, -5, 0))]
    cu, cu_k = (torch.tensor([0] + list(torch.tensor(x).cumsum(0)), dtype=torch.int32, device=DEV) for x in (q_lens, k_lens))
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=DEV)
    q, go = (torch.randn(sum(q_lens), hq, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    k, v = (torch.randn(sum(k_lens), hkv, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    out, want = _with_contexts(q, k, v, go, q_lens, k_lens, ctxs, window_left, d**-0.5)
    got = _c_backward(go, q, k, v, out, cu, torch.float32, d**-0.5, -1 if window_left is None else window_left, cu_k, ctx)
    unit = 4e-6 if d > 128 else 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    for x, ref, name in zip(got, want, ("dq", "dk", "dv")):
        err = ((x.cpu().double() - ref).norm() / ref.norm()).item()
        assert err <= unit, f"{name} {dtype} {hq}/{hkv} d={d} window={window_left}: {err:.3g}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("query_start,window_left", [(0, None), (7, None), (3, 5)])
def test_dense_backward(dtype, query_start, window_left):
    g = torch.Generator().manual_seed(11 + query_start)
    b, h, sq, d = 3, 4, 21, 64
    sk = query_start + sq + 4  # keys behind the last query's position exist and must get zero gradient
    q = torch.randn(b, h, sq, d, generator=g).to(dtype)
    k = torch.randn(b, h, sk, d, generator=g).to(dtype)
    v = torch.randn(b, h, sk, d, generator=g).to(dtype)
    go = torch.randn(b, h, sq, d, generator=g).to(dtype)
    qd, kd, vd = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    out = ops.areno_causal_attention(qd, kd, vd, query_start=query_start, window_left=window_left)
    out.backward(go.to(DEV))
    qf, kf, vf = (x.float().requires_grad_(True) for x in (q, k, v))
    want = ar.ref_attention(qf, kf, vf, query_start, ar.window_left_arg(window_left), d**-0.5)
    want.backward(go.float())
    for got, ref, name in ((qd.grad, qf.grad, "dq"), (kd.grad, kf.grad, "dk"), (vd.grad, vf.grad, "dv")):
        _close(got, ref, REL[dtype], f"dense {name} {dtype} start={query_start} window={window_left}")
    assert float(kd.grad[:, :, query_start + sq :].abs().max()) == 0.0


def test_backward_is_deterministic_and_refuses_other_head_dims():
    g = torch.Generator().manual_seed(2)
    cu = torch.tensor([0, 40, 90], dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(90, h, 128, generator=g).to(torch.bfloat16).to(DEV) for h in (8, 2, 2, 8))
    grads = []
    for _ in range(2):
        qd, kd, vd = (x.clone().requires_grad_(True) for x in (q, k, v))
        ops.areno_varlen_causal_attention(qd, kd, vd, cu).backward(go)
        grads.append((qd.grad, kd.grad, vd.grad))
    for a, b_ in zip(*grads):
        assert torch.equal(a, b_), "no atomics: two runs must agree bit for bit"
    # head dims the backward kernels do not cover (not a multiple of 8, or above 256) are refused by name
    for d in (20, 264):
        qx = torch.randn(10, 2, d, device=DEV, dtype=torch.float32, requires_grad=True)
        cux = torch.tensor([0, 10], dtype=torch.int32, device=DEV)
        out = ops.areno_varlen_causal_attention(qx, qx.detach(), qx.detach(), cux)
        with pytest.raises(RuntimeError, match=f"head_dim {d}"):
            out.sum().backward()


@pytest.mark.parametrize("kv,window_left", [("bf16", None), ("bf16", 11), ("fp32", None), ("int8", None)])
def test_decode_backward_recomputes_like_the_reference(kv, window_left):
    """The decode op under autograd (``_ArenoPagedCausalAttentionDecode.backward``, areno/accel/attention.py:245-264 in
    the reference): gradients of q and of the cache tensors as they stand after the append, none for the update rows;
    compared with autograd through the CPU oracle's decode on the same (appended) cache.  Quantized caches (this
    build's own) give a gradient for q only."""
    from areno_amd import workloads
    from tests.gpu_util import dequant_cpu, gpu_quantize

    act = torch.float32 if kv == "fp32" else torch.bfloat16
    lengths = torch.tensor([0, 5, 16, 37, 70])
    w = workloads.make_decode_workload("decode-backward", seed=61, batch=5, hq=8, hkv=2, d=64, bs=16, kv=kv, lengths=lengths,
                                       device=DEV, act_dtype=act, quantize_fn=gpu_quantize, pool_slack=0.5)  # fmt: skip
    q = w.q.clone().requires_grad_(True)
    quantized = w.k_scale is not None
    kc, vc = w.k_cache, w.v_cache
    if not quantized:
        kc, vc = kc.clone().requires_grad_(True), vc.clone().requires_grad_(True)
    out = ops.areno_paged_causal_attention_decode(q, w.k_update, w.v_update, kc, vc, w.block_table, w.cache_seqlens,
                                                  window_left=window_left, softmax_scale=w.softmax_scale,
                                                  k_scale=w.k_scale, v_scale=w.v_scale)  # fmt: skip
    assert out.requires_grad
    g = torch.Generator().manual_seed(9)
    grad_out = torch.randn(out.shape, generator=g).to(out.dtype)
    out.backward(grad_out.to(DEV))

    # the oracle on the cache after the append, in fp32 on the CPU
    k_ref, v_ref = (dequant_cpu(kc.detach(), w.k_scale), dequant_cpu(vc.detach(), w.v_scale))
    q_ref = w.q.detach().cpu().float().requires_grad_(True)
    k_ref, v_ref = k_ref.requires_grad_(True), v_ref.requires_grad_(True)
    want = ar.ref_paged_decode(q_ref, k_ref, v_ref, w.block_table.cpu(), w.cache_seqlens.cpu(),
                               -1 if window_left is None else window_left, w.softmax_scale)  # fmt: skip
    want.backward(grad_out.float())
    rel = REL[act]
    _close(q.grad, q_ref.grad, rel, "dq")
    if quantized:
        assert w.k_update.grad is None
    else:
        _close(kc.grad, k_ref.grad, rel, "dk_cache")
        _close(vc.grad, v_ref.grad, rel, "dv_cache")
        live = set(w.block_table.cpu().flatten().tolist())
        untouched = [b for b in range(kc.shape[0]) if b not in live]
        assert float(kc.grad[untouched].abs().max()) == 0.0, "pages no row lists must get no gradient"


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 128), (torch.float16, 64), (torch.bfloat16, 96), (torch.float32, 64)])
def test_gradients_in_the_input_dtype_are_the_fp32_gradients_rounded_once(dtype, d):
    """The extension's backward with fp32 gradients (the reference launchers' contract) and with gradients in the
    inputs' dtype (what the autograd functions ask for): the second is the first cast, bit for bit, on the
    matrix-core kernels (head dims 64 / 128) and on the vector-ALU ones (96; fp32 inputs)."""
    from areno_amd.accel.attention import _extension

    g = torch.Generator().manual_seed(d)
    lens = [70, 1, 129, 300]
    t, hq, hkv = sum(lens), 6, 2
    cu = torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32, device=DEV)
    q, go = (torch.randn(t, hq, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    k, v = (torch.randn(t, hkv, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    wide = _extension().areno_attention_backward(go, q, k, v, out, cu, None, None, -1, d**-0.5, False)
    typed = _extension().areno_attention_backward(go, q, k, v, out, cu, None, None, -1, d**-0.5, True)
    for a, b, name in zip(wide, typed, ("dq", "dk", "dv")):
        assert a.dtype == torch.float32 and b.dtype == dtype
        assert torch.equal(a.to(dtype), b), f"{name} {dtype} d={d}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d,parts,dq_rows", [(64, "1w", "16"), (64, "4s", "32"), (128, "1", "32"), (128, "2", "16"), (192, "1", "16"), (192, "2", "16"), (256, "1", "16"), (256, "2", "16")])
def test_gradients_in_the_inputs_type_are_the_fp32_ones_rounded_in_every_form(dtype, d, parts, dq_rows, monkeypatch):
    """The kernels' stores in either type, rows behind the last sequence (zeros) included: bit for bit the same sums, rounded
    once."""
    monkeypatch.setenv("ARENO_BACKWARD_PARTS", parts)
    monkeypatch.setenv("ARENO_BACKWARD_DQ_ROWS", dq_rows)
    g = torch.Generator().manual_seed(d)
    cu = torch.tensor([0, 33, 33, 170], dtype=torch.int32, device=DEV)
    q, k, v, go = (torch.randn(203, h, d, generator=g).to(dtype).to(DEV) for h in (4, 2, 2, 4))
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    wide, narrow = (_c_backward(go, q, k, v, out, cu, t, d**-0.5) for t in (torch.float32, dtype))
    for w, n, name in zip(wide, narrow, ("dq", "dk", "dv")):
        assert w[:170].abs().max() > 0 and torch.equal(w.to(dtype), n), f"{name} {dtype} d={d} parts={parts}"


def _small_varlen(dtype=torch.bfloat16):
    g = torch.Generator().manual_seed(5)
    q, k, v = (torch.randn(49, h, 64, generator=g).to(dtype).to(DEV).requires_grad_(True) for h in (8, 2, 2))
    return q, k, v, torch.tensor([0, 40, 49], dtype=torch.int32, device=DEV)


def _through_the_python_class(q, k, v, cu):
    return ops._VarlenCausalAttention.apply(q, k, v, cu, -1, 64**-0.5)


def test_varlen_autograd_node_is_that_of_the_python_class():
    """The extension's node and the Python class: the same gradients with every subset of inputs that want one, saved-tensor
    hooks that see the same tensors, recomputation, non-contiguous inputs, no graph without a gradient to give."""
    from torch.utils.checkpoint import checkpoint

    q, k, v, cu = _small_varlen()
    weight = torch.randn(49, 8, 64, device=DEV, dtype=torch.bfloat16)
    want = torch.autograd.grad(_through_the_python_class(q, k, v, cu), (q, k, v), weight)
    for wanted in ((0,), (1, 2), (0, 1, 2)):
        args = [x.detach().requires_grad_(i in wanted) for i, x in enumerate((q, k, v))]
        out = ops.areno_varlen_causal_attention(*args, cu)
        grads = torch.autograd.grad(out, [args[i] for i in wanted], weight)
        assert all(torch.equal(a, want[i]) for a, i in zip(grads, wanted))

    def packed_by(op):
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.clone()), t.cpu())[1], lambda t: t.to(DEV)):
            out = op(q, k, v, cu)
        grads = torch.autograd.grad(out, (q, k, v), weight)
        return seen, grads

    (seen, grads), (seen_class, _) = packed_by(ops.areno_varlen_causal_attention), packed_by(_through_the_python_class)
    assert len(seen) == len(seen_class) and all(torch.equal(a, b) for a, b in zip(seen, seen_class))
    assert all(torch.equal(a, b) for a, b in zip(grads, want))

    def layer(a, b, c):
        return ops.areno_varlen_causal_attention(a * 1, b * 1, c * 1, cu)  # (the recomputation stops as soon as it has what was saved)

    grads = torch.autograd.grad(checkpoint(layer, q, k, v, use_reentrant=False), (q, k, v), weight)
    assert all(torch.equal(a, b) for a, b in zip(grads, want))
    wide = torch.randn(49, 8, 128, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    part = wide[..., ::2]
    grad = torch.autograd.grad(ops.areno_varlen_causal_attention(part, k, v, cu), wide, weight)[0]
    assert torch.equal(grad, torch.autograd.grad(_through_the_python_class(part, k, v, cu), wide, weight)[0])
    with torch.no_grad():
        assert not ops.areno_varlen_causal_attention(q, k, v, cu).requires_grad
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    with torch.no_grad():
        q.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        out.backward(weight)
    q, k, v, cu = _small_varlen()
    out = ops.areno_varlen_causal_attention(q, k, v, cu)
    out.backward(weight)
    with pytest.raises(RuntimeError, match="second time"):
        out.backward(weight)


def test_varlen_calls_that_no_node_of_its_own_takes():
    """Forward-mode tangents and vmap are refused as the Python class refuses them; a hook's exception stays itself."""
    q, k, v, cu = _small_varlen()
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(q.detach(), torch.ones_like(q))
        with pytest.raises(RuntimeError):
            ops.areno_varlen_causal_attention(dual, k, v, cu)
    with pytest.raises(RuntimeError, match="vmap"):
        torch.vmap(lambda x: ops.areno_varlen_causal_attention(x, k, v, cu))(torch.stack([q.detach(), q.detach()]))

    class Own(Exception):
        pass

    def refuse(t):
        raise Own

    with torch.autograd.graph.saved_tensors_hooks(refuse, lambda t: t), pytest.raises(Own):
        ops.areno_varlen_causal_attention(q, k, v, cu)
