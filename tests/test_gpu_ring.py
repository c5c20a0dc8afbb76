"""The grouped GEMM's ring kernel (few rows: tiles of 1 to 4 blocks of 32 rows by 128
columns) and its launches of few persistent tiles against many persistent 256-row tiles,
which serve the launches with many rows.

Every accumulator takes its k in one order whatever the tile, so the two must agree bit
for bit; the persistent kernel is checked against float32 products elsewhere
(test_gpu_gemm.py), and one expert is checked here too."""
import pytest
import torch

from genet5_amd import ops

pytestmark = pytest.mark.gpu


def _offsets(counts, dev):
    off = [0]
    for c in counts:
        off.append(off[-1] + c)
    return off, torch.tensor(off, dtype=torch.int32, device=dev)


# The tile that the launch takes on 256 CUs (blocks of 32 rows, workgroups per CU) stands
# after each case: every form of the kernel has one.
@pytest.mark.parametrize("K,n_out,counts", [
    (128, 128, [1, 0, 31, 32, 33]),         # 1, two: the smallest, two k-steps, one n-tile
    (192, 256, [0, 5, 64, 65]),             # 1, two: odd k-step count
    (768, 768, [6, 0, 9, 4, 1, 12, 7, 0]),  # 1, two
    (3072, 768, [97, 96, 0, 128, 31, 64, 65, 129, 1, 95, 100, 90, 97, 97, 97]),  # 2, two
    (1024, 768, [257, 255, 256, 288, 289, 1, 0, 320]),  # 2, two
    (768, 384, [1137]),                     # 1, two: one expert, an odd number of n-tiles
    (256, 2304, [4550]),                    # persistent: one expert in the larger launch too
    (192, 768, [137, 96, 97, 0, 128, 129, 192, 193, 31, 160, 161, 95, 288, 289, 33]),  # 3, one
    (3072, 768, [137, 96, 97, 0, 128, 129, 192, 193, 31, 160, 161, 95, 288, 289, 33]),  # 3, one
    (256, 768, [256, 255, 257, 0, 1, 128, 129, 300, 511, 512, 385, 320, 290, 230, 270]),  # 4, one
    (128, 768, [375, 384, 385, 0, 31, 33, 512, 513, 400, 390, 700, 640, 641, 128, 129]),  # 4, two
    (768, 2304, [2048]),                    # 4, two: one expert
    # persistent tiles with less than one per CU (whole ones, n-halves), three and two
    # fragment slots, 256 and 128 columns
    (192, 768, [800, 769, 0, 1023, 1024, 1025, 700, 1, 900, 850, 760, 513, 640, 1100, 1300]),
    (448, 256, [9000, 8000, 7000, 9500, 1, 0, 4000, 257]),
    (384, 640, [9000, 1, 0, 257, 300]),
])
@pytest.mark.parametrize("packed", [False, True])
def test_ring_equals_persistent_tiles(cuda_device, K, n_out, counts, packed):
    print(f"ring K={K} n_out={n_out} counts={counts} packed={packed}", flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(K + n_out + len(counts))
    rows = sum(counts)
    # one more expert with so many rows that the launch leaves the ring kernel
    big = -(-(768 * 256 * 256) // n_out)
    E = len(counts)
    off, t_off = _offsets(counts, cuda_device)
    _, t_off_big = _offsets(counts + [big], cuda_device)
    b = (torch.randn(E + 1, n_out, K, device=cuda_device, generator=g) / K ** 0.5).bfloat16()
    if packed:
        a = torch.randn(ops.packed_rows(rows + big, E + 1) + ops.ROW_PAD, K, device=cuda_device,
                        generator=g).bfloat16()
        small = ops.grouped_gemm_padded(a[:ops.packed_rows(rows, E) + ops.ROW_PAD], 0, rows, t_off,
                                        b[:E])
        large = ops.grouped_gemm_padded(a, 0, rows + big, t_off_big, b)
    else:
        a = torch.randn(rows + big + ops.ROW_PAD, K, device=cuda_device, generator=g).bfloat16()
        small = ops.grouped_gemm(a[:rows + ops.ROW_PAD], rows, t_off, b[:E])
        large = ops.grouped_gemm(a, rows + big, t_off_big, b)
    torch.cuda.synchronize()
    assert torch.equal(small.view(torch.int16), large[:rows].view(torch.int16))
    if not packed:
        e = max(range(E), key=lambda i: counts[i])
        ref = a[off[e]:off[e + 1]].float() @ b[e].float().t()
        err = (small[off[e]:off[e + 1]].float() - ref).abs()
        # one bf16 rounding (2^-9 relative, half an ulp) of an fp32 sum of K products of
        # about N(0, 1/K): K fp32 roundings of partial sums of about 1
        assert (err <= ref.abs() * 2.0 ** -8 + K * 2.0 ** -24 * 4).all()


@pytest.mark.parametrize("n,d,F,E,k,p", [
    (1, 768, 3072, 16, 2, 0.1),      # two rows in all
    (130, 768, 3072, 16, 2, 0.0),    # one block per expert
    (777, 768, 3072, 16, 2, 0.1),    # up to four blocks, the last partial
    (1000, 256, 1024, 8, 2, 0.1),    # three-block tiles
    (96, 128, 128, 4, 1, 0.0),       # the smallest d and F: two k-steps, two n-tiles
])
def test_ring_gate_up_equals_persistent_tiles(cuda_device, n, d, F, E, k, p):
    """The gate|up products of a few tokens (ring kernel) equal the same tokens' rows in a
    batch that takes the persistent tiles, bit for bit: h, and where the training forward
    keeps them (d and F multiples of 256) the SwiGLU factors, under one dropout mask (it is
    keyed on the token and slot)."""
    print(f"ring gate|up n={n} d={d} F={F} E={E} k={k} p={p}", flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(n + d)
    # (past ring_wide's rows: d = 128's two n-tiles stay below half the CUs up to 32,768)
    big = {128: 40000, 256: 24000, 768: 6000}[d]
    r = lambda *s, std=1.0: (torch.randn(*s, device=cuda_device, generator=g) * std).bfloat16()
    x, wr = r(big, d), r(E, d, std=0.05)
    wgu, wd = r(E, 2 * F, d, std=0.02), r(E, d, F, std=0.02)
    train = d % 256 == 0 and F % 256 == 0
    rows = []
    for m in (n, big):
        if train:
            out = ops.moe_forward_train(x[:m], wr, wgu, wd, k, dropout=(p, 77) if p else None,
                                        return_h=True, factors=True)
            inv, ops_rows = out[6][:n * k].long(), (out[9], out[8])
            rows.append([t[inv] for t in ops_rows])
        idx, _, _, off, perm, inv = ops.route(x[:m], wr, k)
        _, h = ops.expert_swiglu(x[:m], perm, off, wgu, wd, k, return_h=True)
        rows.append([h[inv[:n * k].long()]])
    torch.cuda.synchronize()
    half = len(rows) // 2
    for small, large in zip(rows[:half], rows[half:]):
        for a, b in zip(small, large):
            assert torch.equal(a.view(torch.int16), b.view(torch.int16))


@pytest.mark.parametrize("counts", [[0, 1, 31, 32, 33, 64, 0, 129], [383, 0, 97, 2],
                                    [0, 0, 0, 5]])
@pytest.mark.parametrize("kmax", [0, 384])
def test_ring_dh_swiglu_equals_staged(cuda_device, counts, kmax):
    """The dh product with the SwiGLU backward of a few rows (ring kernel): the staged dh
    times the factors in fp32, bit for bit, zeros in every padding row that the weight
    gradient reads and nothing written after them."""
    import ctypes

    from genet5_amd import _lib
    d, F, E = 256, 512, len(counts)
    print(f"ring dh counts={counts} kmax={kmax}", flush=True)
    g = torch.Generator(device=cuda_device).manual_seed(sum(counts) + kmax)
    rows = sum(counts)
    off, t_off = _offsets(counts, cuda_device)
    wrows = [max(384, -(-c // 192) * 192) for c in counts]
    starts = [e * kmax if kmax else sum(wrows[:e]) for e in range(E)]
    prows = E * kmax if kmax else ops.packed_rows(rows, E)
    dy = torch.randn(prows + ops.ROW_PAD, d, device=cuda_device, generator=g).bfloat16()
    wdt = (torch.randn(E, F, d, device=cuda_device, generator=g) * 0.05).bfloat16()
    fac = torch.randn(rows, 2 * F, device=cuda_device, generator=g).bfloat16()
    got = torch.full((prows + ops.ROW_PAD, 2 * F), 7.0, device=cuda_device).bfloat16()
    shape = _lib.make_shape(rows, d, F, E, 1, _lib.DTYPE_BF16)
    _lib.call("g5moe_dh_swiglu_backward", ops._ptr(dy), kmax, ops._ptr(t_off), ops._ptr(wdt),
              ops._ptr(fac), ops._ptr(got), ctypes.byref(shape), ops._stream(cuda_device))
    dh = ops.grouped_gemm_padded(dy, kmax, rows, t_off, wdt).float()
    want = torch.full_like(got, 7.0)
    fv = fac.view(rows, F // 32, 2, 32).float()
    prod = (dh.view(rows, F // 32, 1, 32) * fv).reshape(rows, 2 * F).bfloat16()
    for e in range(E):
        want[starts[e]:starts[e] + wrows[e]] = 0
        want[starts[e]:starts[e] + counts[e]] = prod[off[e]:off[e + 1]]
    torch.cuda.synchronize()
    # values: a zero product may carry either sign
    assert torch.equal(got.float(), want.float())
