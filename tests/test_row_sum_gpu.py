"""GPU: the sum of a row's squares and the reciprocal RMS at the row lengths and magnitudes where their code changes."""
import pytest
import torch

from oracle import eager

from helpers import check_against_oracle, run_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vpt", [1, 2, 4])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float64])
def test_every_number_of_block_sums(cuda_device, dtype, vpt):
    """Every number of 512-float blocks up to the longest row, with no floats beside the chains, one vector, nearly three
    vectors and scalars left over, and a last block of one and of fifteen steps; alone and several rows to a workgroup."""
    vec, longest = 16 // dtype.itemsize, 16384 // dtype.itemsize
    lengths = sorted({n for b in range(1, longest // 512 + 1) for n in (512 * b, 512 * b - vec, 512 * b - 8, 512 * b - 480, 512 * b - 456)}
                     | {vec, 32 - vec, 32, 64})
    for n in lengths:
        print("case", dtype, vpt, n, flush=True)
        p, r, g = eager.make_inputs(2, 7, n, dtype, 1.0, seed=n)
        want = eager.reduce_rms(p, r, g, 1e-6, "none")
        for rpb in (0, 5):
            check_against_oracle(run_hip(p, r, g, 1e-6, "none", vecs_per_thread=vpt, rows_per_block=rpb), want, "none", gamma=g, eps=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_reciprocal_rms_at_the_ends_of_its_fast_path(cuda_device, dtype):
    """Means of squares around 2^-60 and 2^100, where the plain divisions and square root take over, far beyond both, and a mean that
    vanishes beside eps."""
    for k in (-62, -31, -30, -29, 0, 49, 50, 51, 55):
        for eps in (0.0, 1e-6):
            print("case", dtype, k, eps, flush=True)
            p, r, g = eager.make_inputs(2, 16, 1000, torch.float32, 1.0, seed=90 + k)
            p, r, g = (p * 2.0 ** k).to(dtype), (r * 2.0 ** k).to(dtype), g.to(dtype)
            check_against_oracle(run_hip(p, r, g, eps, "none"), eager.reduce_rms(p, r, g, eps, "none"), "none", gamma=g, eps=eps)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32, torch.float64])
def test_reciprocal_rms_of_the_hardest_means(cuda_device, dtype):
    """Means whose root lies just below a power of two or whose reciprocal lies next to the middle of two floats.  The row's own
    squares vanish beside eps, which is the mean."""
    x = (torch.arange(1024, dtype=torch.float64) / 1024 + 1) * 2.0 ** -14
    r, g = x.to(dtype).expand(3, -1).contiguous(), torch.ones(1024, dtype=dtype)
    for bits in (0x407ffffe, 0x407fffff, 0x3f8d8936, 0x3f9fb52d, 0x3f9fb52f):
        for k in (0, 9, 20):
            eps = float(torch.tensor([bits], dtype=torch.int32).view(torch.float32)) * 4.0 ** k
            print("case", dtype, hex(bits), k, flush=True)
            p = torch.zeros((2, 3, 1024), dtype=dtype)
            check_against_oracle(run_hip(p, r, g, eps, "none"), eager.reduce_rms(p, r, g, eps, "none"), "none", gamma=g, eps=eps)


def test_reciprocal_rms_of_a_row_just_below_two(cuda_device):
    r = torch.tensor([[2.0, 2.0, 2.0, 2.0 - 2.0 ** -22]])
    p, g = torch.zeros((2, 1, 4)), torch.ones(4)
    want = eager.reduce_rms(p, r, g, 0.0, "none")
    assert want["norm_out"][0, 0].item() == 1.0 + 2.0 ** -23
    check_against_oracle(run_hip(p, r, g, 0.0, "none"), want, "none", gamma=g, eps=0.0)
