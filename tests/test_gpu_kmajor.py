"""The K-major 256x256 kernel at the edges of its stages, tiles and schedule,
against the oracle (2e-2 * sqrt(max(K, 512) / 512), as in test_gpu_gemm) and,
where no tile is split, bitwise against the 128x128 tile (every output is the
same fp32 sum in the same K order)."""
import pytest
import torch

import grouped_gemm as gg
from test_gpu_gemm import assert_parity, covered_rows, kmajor_copy, log, make_inputs

pytestmark = pytest.mark.gpu

# (counts, K, N): K below, at and past one, two and three 64-deep stages, and
# not a multiple of a stage; rows and columns below, at and past a tile; a
# last chunk of C's rows that is not 16 bytes; more tiles than workers.
CASES = [
    ([1, 0, 3], 8, 2),
    ([255, 257], 64, 256),
    ([256, 0, 1], 72, 258),
    ([513, 40], 128, 250),
    ([300, 0, 20], 136, 512),
    ([17, 512], 192, 770),
    ([600, 31, 0, 257], 328, 264),
]


@pytest.mark.parametrize("case", range(len(CASES)))
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kmajor_256_edges(cuda_device, case, dtype):
    counts, k, n = CASES[case]
    a, b, offs = make_inputs(counts, k, n, dtype, cuda_device, seed=300 + case, extra_rows=3)
    b_km = kmajor_copy(b, 0)
    mask = torch.from_numpy(covered_rows(offs)).to(cuda_device)
    want = gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(128, 128), use_atomic_queue=False)
    for queue, atomic, workers in (("device", False, None), ("device", True, 3), ("device", False, 2),
                                   ("prebuilt", True, 5)):
        log(f"kmajor edges case={case} {dtype} queue={queue} atomic={atomic} workers={workers}")
        c = gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(256, 256), queue=queue,
                                       use_atomic_queue=atomic, num_sms=workers)
        torch.cuda.synchronize()
        assert torch.equal(c[: mask.numel()][mask], want[: mask.numel()][mask]), (queue, atomic)
    assert_parity(c, a, b, offs, k)


@pytest.mark.parametrize("parts,workers", [(2, 16), (3, 16), (4, 16)])
def test_kmajor_split_last_round(cuda_device, parts, workers):
    """Tiles of a short last round summed as 2, 3 or 4 parts of K (at least
    1024 of K each): within the tolerance of the oracle, the same bits on
    every call whichever part comes last, and in a second round after whole
    tiles."""
    k, n = 1024 * parts + 200, 512
    tiles = workers // parts  # split as many ways as fit
    for extra in (0, workers):  # a whole round before the split one
        counts = [256 * ((tiles + extra) // 2) - 5]
        a, b, offs = make_inputs(counts, k, n, torch.bfloat16, cuda_device, seed=parts, extra_rows=1)
        b_km = kmajor_copy(b, 0)
        outs = []
        for _ in range(3):
            log(f"kmajor split parts={parts} extra={extra}")
            outs.append(gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(256, 256), num_sms=workers))
        torch.cuda.synchronize()
        assert torch.equal(outs[0][: counts[0]], outs[1][: counts[0]])
        assert torch.equal(outs[0][: counts[0]], outs[2][: counts[0]])
        assert_parity(outs[0], a, b, offs, k)
