"""The grouped GEMM's ring kernel (few rows: tiles of 1 to 4 blocks of 32 rows by 128
columns) against the persistent 256-row tiles, which serve the launches with many rows.

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


@pytest.mark.parametrize("K,n_out,counts", [
    (128, 128, [1, 0, 31, 32, 33]),                    # the smallest: two k-steps, one n-tile
    (192, 256, [0, 5, 64, 65]),                        # odd k-step count
    (768, 768, [6, 0, 9, 4, 1, 12, 7, 0]),             # one block per tile
    (3072, 768, [97, 96, 0, 128, 31, 64, 65, 129, 1, 95, 100, 90, 97, 97, 97]),
    (1024, 768, [257, 255, 256, 288, 289, 1, 0, 320]),  # three- and four-block tiles
    (768, 384, [1137]),                                # one expert, an odd number of n-tiles
    (256, 2304, [4550]),
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
