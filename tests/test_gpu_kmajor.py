"""The K-major 256x256 kernel at the edges of its stages, tiles and schedule,
against the oracle (2e-2 * sqrt(max(K, 512) / 512), as in test_gpu_gemm) and,
where no tile is split, bitwise against the 128x128 tile (every output is the
same fp32 sum in the same K order)."""
import pytest
import torch

import expert_mlp as mlp
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


@pytest.mark.parametrize("case", range(len(CASES) + 1))
def test_kmajor_256_one_worker(cuda_device, case):
    """Every tile on one worker, its loads running on from tile to tile: short
    K keeps the four-wave kernel there (two tiles a worker), and K of less
    than a stage, too."""
    counts, k, n = (CASES + [([1, 0, 3], 8, 258)])[case]
    a, b, offs = make_inputs(counts, k, n, torch.bfloat16, cuda_device, seed=400 + case, extra_rows=3)
    b_km = kmajor_copy(b, 0)
    mask = torch.from_numpy(covered_rows(offs)).to(cuda_device)
    want = gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(128, 128), use_atomic_queue=False)
    for queue, atomic in (("device", False), ("device", True), ("prebuilt", True)):
        log(f"kmajor one worker case={case} queue={queue} atomic={atomic}")
        c = gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(256, 256), queue=queue,
                                       use_atomic_queue=atomic, num_sms=1)
        torch.cuda.synchronize()
        assert torch.equal(c[: mask.numel()][mask], want[: mask.numel()][mask]), (queue, atomic)


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


def _fused(a, b, offs, activation, block, workers, atomic):
    out = b.shape[2] // 2 if activation == "swiglu" else b.shape[2]
    return mlp._grouped_gemm_ex(a, b, offs, mlp._EPILOGUES[activation], out, workers, block, atomic)


# N: whole tiles; a last tile whose columns end inside a wave's half; C's rows
# not whole 16-byte chunks (GELU only: SwiGLU's N is a multiple of 64).
@pytest.mark.parametrize("activation,n", [("gelu", 512), ("gelu", 320), ("gelu", 516), ("swiglu", 512),
                                          ("swiglu", 320), ("swiglu", 704)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_kmajor_fused_epilogues(cuda_device, activation, n, dtype):
    """The activations on several tiles a worker (the next tile's loads behind
    the stores), several stages of K and a part of one: bitwise the 128x128
    tile's."""
    counts, k = [300, 0, 257, 1, 200], 1032
    a, b, offs = make_inputs(counts, k, n, dtype, cuda_device, seed=n, extra_rows=1)
    b_km = kmajor_copy(b, 16)
    rows = sum(counts)
    want = _fused(a, b_km, offs, activation, 128, None, False)
    for atomic, workers in ((False, 2), (True, 3), (True, 1)):
        log(f"kmajor fused {activation} n={n} {dtype} atomic={atomic} workers={workers}")
        got = _fused(a, b_km, offs, activation, 256, workers, atomic)
        torch.cuda.synchronize()
        assert torch.equal(got[:rows], want[:rows]), (atomic, workers)


@pytest.mark.parametrize("activation,n", [("none", 320), ("none", 516), ("gelu", 512), ("gelu", 516),
                                          ("swiglu", 320)])
@pytest.mark.parametrize("tiles,k", [(8, 2248), (5, 3272), (4, 4160)])  # halves, thirds, quarters of K
def test_kmajor_split_epilogues(cuda_device, activation, n, tiles, k):
    """Tiles summed in parts of K under every epilogue, with columns that do
    not fill the tile.  The whole tile's sum and the parts' differ by fp32
    rounding (about 1e-5 of unit-scale sums, at most 1e-4 after the
    activation), so the bf16 results differ by a rounding at most."""
    workers, counts = 16, [256 * (tiles // 2) - 5]
    a, b, offs = make_inputs(counts, k, n, torch.bfloat16, cuda_device, seed=tiles, extra_rows=1)
    b_km = kmajor_copy(b, 0)

    def run(block, num_sms, atomic):
        if activation == "none":
            return gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(block, block), num_sms=num_sms,
                                              use_atomic_queue=atomic)[: counts[0]]
        return _fused(a, b_km, offs, activation, block, num_sms, atomic)[: counts[0]]

    log(f"kmajor split {activation} n={n} tiles={tiles} k={k}")
    want = run(128, None, False)
    outs = [run(256, workers, True) for _ in range(3)]
    torch.cuda.synchronize()
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    torch.testing.assert_close(outs[0].float(), want.float(), rtol=2.0 ** -7, atol=1e-4)


@pytest.mark.parametrize("experts", [64, 65, 129, 1000, 2048])
def test_kmajor_finds_the_expert(cuda_device, experts):
    """Device-derived tiles of more experts than a wave has lanes, empty ones
    among them, more than one m-tile in a few."""
    gen = torch.Generator().manual_seed(experts)
    counts = torch.randint(0, 6, (experts,), generator=gen)
    counts[torch.randint(0, experts, (3,), generator=gen)] = 300
    counts[-1] = 2
    k, n = 72, 258
    a, b, offs = make_inputs(counts.tolist(), k, n, torch.bfloat16, cuda_device, seed=experts)
    b_km = kmajor_copy(b, 0)
    want = gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(128, 128), use_atomic_queue=False)
    for atomic in (False, True):
        log(f"kmajor experts={experts} atomic={atomic}")
        got = gg.persistent_grouped_gemm(a, b_km, offs, kernel_tile=(256, 256), num_sms=3, use_atomic_queue=atomic)
        torch.cuda.synchronize()
        assert torch.equal(got, want), atomic
