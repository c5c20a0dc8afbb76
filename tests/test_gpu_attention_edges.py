"""The attention kernel at the edges of its block loop, against float64 softmax attention
(plain numpy on the host).

Tolerance, as in test_gpu_attention.py: bf16 probabilities and one bf16 rounding of the
output, normwise max <= 1e-2 and mean <= 4e-3."""
import numpy as np
import pytest
import torch

from genet5_amd import attention
from genet5_amd.attention import alibi_slopes

pytestmark = pytest.mark.gpu


def reference(q, k, v, cu, scale, slopes):
    q, k, v = (t.double().cpu().numpy() for t in (q, k, v))
    out = np.zeros_like(q)
    rep = q.shape[1] // k.shape[1]
    for a, b in zip(cu[:-1], cu[1:]):
        pos = np.arange(b - a, dtype=np.float64)
        dist = np.abs(pos[:, None] - pos[None, :])
        for h in range(q.shape[1]):
            s = q[a:b, h] @ k[a:b, h // rep].T * scale
            if slopes is not None:
                s = s - slopes[h] * dist
            p = np.exp(s - s.max(axis=1, keepdims=True))
            out[a:b, h] = p @ v[a:b, h // rep] / p.sum(axis=1, keepdims=True)
    return out


def inputs(T, H, seed, dev, scale=1.0):
    g = torch.Generator(device="cpu").manual_seed(seed)
    return [(torch.randn(T, H, 64, generator=g) * s).to(torch.bfloat16).to(dev)
            for s in (scale, scale, 1.0)]


def check(got, ref, what):
    err = np.abs(got.double().cpu().numpy() - ref)
    mx, mean = err.max() / np.abs(ref).max(), err.mean() / np.abs(ref).mean()
    print(f"  {what}: max_rel={mx:.2e} mean_rel={mean:.2e}", flush=True)
    assert mx <= 1e-2 and mean <= 4e-3, (what, mx, mean)


@pytest.mark.parametrize("use_alibi", [False, True])
@pytest.mark.parametrize("softmax_scale", [0.125, 0.5, 0.0, -0.125])
def test_block_edges(cuda_device, use_alibi, softmax_scale):
    """Lengths around the 32-query, 64-key and 128-query edges, in one packed call, with
    scales that the fast path takes (a negative one on negated queries) and one, zero, that
    only the exact path does."""
    lens = [1, 31, 32, 33, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 257]
    cu = np.concatenate([[0], np.cumsum(lens)]).tolist()
    q, k, v = inputs(cu[-1], 4, 3, cuda_device)
    slopes = alibi_slopes(4) if use_alibi else None
    cu_t = torch.tensor(cu, dtype=torch.int32, device=cuda_device)
    sl = torch.tensor(slopes, device=cuda_device) if use_alibi else None
    print(f"attention edges alibi={use_alibi} scale={softmax_scale}", flush=True)
    # max_seqlen past 2,048 makes the kernel use the key bounds (a larger grid only)
    for max_len in (max(lens), 2200):
        out = attention.attn_varlen_fwd(q, k, v, cu_t, max_len, softmax_scale, sl)
        torch.cuda.synchronize()
        check(out, reference(q, k, v, cu, softmax_scale, slopes), f"max_seqlen={max_len}")


def test_negative_slopes(cuda_device):
    cu = [0, 200, 330]
    q, k, v = inputs(cu[-1], 2, 5, cuda_device)
    slopes = [-0.02, 0.3]
    out = attention.attn_varlen_fwd(q, k, v, torch.tensor(cu, dtype=torch.int32, device=cuda_device),
                                    200, 0.125, torch.tensor(slopes, device=cuda_device))
    torch.cuda.synchronize()
    check(out, reference(q, k, v, cu, 0.125, slopes), "negative slope")


@pytest.mark.parametrize("softmax_scale", [0.125, -0.125, 0.0])
@pytest.mark.parametrize("slopes", [[-0.02, -0.3, 0.3, -1e-4], [0.0, -5.0, 1e30, -1e30]])
def test_slopes_of_either_sign_over_many_blocks(cuda_device, slopes, softmax_scale):
    """Whole blocks before and after the queries with a bias that grows with the distance,
    and slopes that leave the bias chunk's range (2^60 scale), where the exact path serves."""
    cu = [0, 700, 829]
    q, k, v = inputs(cu[-1], 4, 13, cuda_device)
    print(f"slopes {slopes} scale {softmax_scale}", flush=True)
    out = attention.attn_varlen_fwd(q, k, v, torch.tensor(cu, dtype=torch.int32, device=cuda_device),
                                    700, softmax_scale, torch.tensor(slopes, device=cuda_device))
    torch.cuda.synchronize()
    check(out, reference(q, k, v, cu, softmax_scale, slopes), f"{slopes} {softmax_scale}")


@pytest.mark.parametrize("scale", [1.0, 3.0])
def test_positions_past_8192(cuda_device, scale):
    """Long distances in the bias chunk's constant, both loops: a nearly flat slope keeps
    the far keys in every row."""
    L = 8192 * 2 + 77
    q, k, v = inputs(L, 2, 7, cuda_device, scale)
    slopes = [1e-4, 3e-5]
    cu = [0, L]
    out = attention.attn_varlen_fwd(q, k, v, torch.tensor(cu, dtype=torch.int32, device=cuda_device),
                                    L, 0.125, torch.tensor(slopes, device=cuda_device))
    torch.cuda.synchronize()
    rows = np.array([0, 33, 8191, 8192, 8250, 16383, L - 1])
    qd, kd, vd = (t.double().cpu().numpy() for t in (q, k, v))
    ref = np.zeros((len(rows), 2, 64))
    for h in range(2):
        s = qd[rows, h] @ kd[:, h].T * 0.125 - slopes[h] * np.abs(rows[:, None] - np.arange(L))
        p = np.exp(s - s.max(axis=1, keepdims=True))
        ref[:, h] = p @ vd[:, h] / p.sum(axis=1, keepdims=True)
    check(out[torch.from_numpy(rows).to(cuda_device)], ref, f"scale={scale}")


def test_other_sequences_nan_and_inf_stay_out(cuda_device):
    """A partial last block's missing keys are not read from the next sequence: NaN keys and
    infinite values there leave this one's output unchanged, bit for bit."""
    cu = [0, 70, 140, 333]
    q, k, v = inputs(cu[-1], 2, 9, cuda_device)
    cu_t = torch.tensor(cu, dtype=torch.int32, device=cuda_device)
    sl = torch.tensor([0.5, 0.01], device=cuda_device)
    want = attention.attn_varlen_fwd(q, k, v, cu_t, 193, 0.125, sl)
    k2, v2 = k.clone(), v.clone()
    for a, b in ((0, 70), (140, 333)):
        k2[a:b] = float("nan")
        v2[a:b] = float("inf")
    got = attention.attn_varlen_fwd(q, k2, v2, cu_t, 193, 0.125, sl)
    torch.cuda.synchronize()
    assert torch.equal(got[70:140].view(torch.int16), want[70:140].view(torch.int16))
    # an infinite value in a sequence's own last row reaches its rows as an infinity
    v3 = v.clone()
    v3[139, :, 0] = float("inf")
    own = attention.attn_varlen_fwd(q, k, v3, cu_t, 193, 0.125, None)
    torch.cuda.synchronize()
    assert torch.isinf(own[70:140, :, 0]).all() and torch.isfinite(own[70:140, :, 1:]).all()


def test_wide_token_strides(cuda_device):
    """Token strides too large for 32-bit offsets inside a 64-key tile (2^24 elements)."""
    T, stride = 70, 1 << 24
    q, k, v = inputs(T, 1, 11, cuda_device)
    buf = torch.empty((T * stride,), dtype=torch.bfloat16, device=cuda_device)
    kw = buf.as_strided((T, 1, 64), (stride, 64, 1))
    vw = buf.as_strided((T, 1, 64), (stride, 64, 1), storage_offset=64)
    kw.copy_(k)
    vw.copy_(v)
    cu_t = torch.tensor([0, T], dtype=torch.int32, device=cuda_device)
    got = attention.attn_varlen_fwd(q, kw, vw, cu_t, T, 0.125)
    want = attention.attn_varlen_fwd(q, k, v, cu_t, T, 0.125)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
