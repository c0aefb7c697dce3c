"""The plane GEMM (launches of 8 rows and more on a frozen weight) at the edges of its tiles: row counts around 16-row
fragments and 32/64/128-row tiles, output widths around the 16-column fragments and the 128/256-column tiles,
contractions of one slab, an odd number of slabs and long enough to be split, and rank-r terms of one, two and three
32-rank steps, against the same product in float64.

Bars: a product of two ~22-bit operands (modes 3 and 5) is off by ~2^-22 per term plus the fp32 accumulation, 2e-6
over these lengths; two planes on one side (modes 2 and 4) leave the other's fp16 rounding, as one pass does: 2^-11
per term, averaging to ~3e-4 of the row, 1e-3. The rank term is bf16 hi/lo, 2^-16 of its own size (here about a tenth
of the output)."""
import numpy as np
import pytest

from oracle import binding as o

pytestmark = pytest.mark.gpu

Q8_0, Q4_K, Q6_K = 8, 12, 14
BAR = {1: 1e-3, 2: 1e-3, 3: 2e-6, 4: 1e-3, 5: 2e-6}


@pytest.fixture(scope="module")
def gpu():
    from hos_amd import Gpu
    g = Gpu(0)
    yield g
    g.close()


# (dx, type, rows, cols, t): forward output width rows over a contraction of cols, dX the other way round
SHAPES = [
    (False, Q8_0, 16, 32, 64),       # one fragment, one slab
    (False, Q8_0, 48, 288, 8),       # fewer rows than a fragment has, more steps than the small kernel has waves
    (True, Q4_K, 1152, 256, 33),     # the longest contraction of the small kernel
    (False, Q8_0, 40, 96, 65),       # a ragged 16-column block, three slabs
    (False, Q4_K, 129, 256, 127),
    (False, Q6_K, 257, 512, 129),    # one column past a 256-column tile
    (True, Q8_0, 32, 32, 64),
    (True, Q8_0, 96, 160, 333),      # a contraction of three slabs (no 64-deep ones)
    (True, Q4_K, 4096, 256, 70),     # long enough to split
    (True, Q8_0, 2080, 288, 1031),
    (False, Q8_0, 1000, 2048, 2050),
]


@pytest.mark.parametrize("passes", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("shape", SHAPES)
def test_plane_gemm_edges(gpu, shape, passes):
    dx, ty, rows, cols, t = shape
    print(f"plane gemm {shape} passes {passes}", flush=True)
    rng = np.random.default_rng(rows * 7 + cols + t)
    raw = o.quantize(rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(0.05), ty)
    w = o.dequant(raw, ty, rows * cols).reshape(rows, cols).astype(np.float64)
    x = rng.standard_normal((t, rows if dx else cols)).astype(np.float32)
    gpu.set_gemm_passes(passes)
    gpu.upload_quant(0x77, raw, ty, rows, cols)
    y = gpu.qgemm_dx(0x77, x, cols) if dx else gpu.qgemm_fwd(0x77, x, rows)
    want = x.astype(np.float64) @ (w if dx else w.T)
    gpu.evict(0x77)
    gpu.set_gemm_passes(1)
    err = np.linalg.norm(y - want) / np.linalg.norm(want)
    assert err <= BAR[passes], err
    # every element, not only the norm: a row or column gone wrong would be off by about its own size
    assert np.abs(y - want).max() <= 0.05 * np.sqrt((want ** 2).mean())


@pytest.mark.parametrize("rank,ldu", [(1, 1), (8, 56), (16, 17), (31, 40), (33, 33), (48, 64), (96, 96)])
@pytest.mark.parametrize("which", [0, 1])
def test_plane_gemm_rank_term(gpu, which, rank, ldu):
    rows, cols, t = 288, 224, 141
    print(f"plane gemm rank {rank} ldu {ldu} which {which}", flush=True)
    rng = np.random.default_rng(rank * 3 + which)
    raw = o.quantize(rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(0.05), Q8_0)
    w = o.dequant(raw, Q8_0, rows * cols).reshape(rows, cols).astype(np.float64)
    n, c = (rows, cols) if which == 0 else (cols, rows)
    x = rng.standard_normal((t, c)).astype(np.float32)
    u = rng.standard_normal((t, ldu)).astype(np.float32) * np.float32(0.1)
    lf = rng.standard_normal((rank, n)).astype(np.float32) * np.float32(0.1)
    gpu.set_gemm_passes(3)
    gpu.upload_quant(0x78, raw, Q8_0, rows, cols)
    xd, ud, ld, out = gpu.to_dev(x), gpu.to_dev(u), gpu.to_dev(lf), gpu.empty_dev((t, n))
    gpu.op("qgemm_lora_dev", which, 0x78, xd, t, ud, ldu, ld, n, 1, rank, 1.5, out)
    y = out.get()
    base = x.astype(np.float64) @ (w.T if which == 0 else w)
    term = 1.5 * (u[:, :rank].astype(np.float64) @ lf.astype(np.float64))
    for a in (xd, ud, ld, out):
        a.free()
    gpu.evict(0x78)
    gpu.set_gemm_passes(1)
    err = np.linalg.norm(y - (base + term))
    assert err <= 2e-6 * np.linalg.norm(base) + 2e-5 * np.linalg.norm(term)


# contractions of one, nine and fifteen slabs, of two splits, of four with a short last one, and outputs past 512
# workgroups of 16 rows
@pytest.mark.parametrize("n,c", [(32, 64), (576, 576), (96, 960), (576, 1536), (64, 2240), (1536, 576)])
@pytest.mark.parametrize("which,rank", [(0, 0), (1, 0), (0, 16), (1, 33)])
def test_chain_sums_are_the_dequantizing_kernels(gpu, which, rank, n, c):
    """Under 8 rows the dequantizing kernel runs; 64 rows have its tiles and splits: equal bit for bit."""
    print(f"chain {n} x {c} which {which} rank {rank}", flush=True)
    t = 64
    rng = np.random.default_rng(n + c + rank)
    rows, cols = (n, c) if which == 0 else (c, n)
    raw = o.quantize(rng.standard_normal((rows, cols)).astype(np.float32) * np.float32(0.05), Q8_0)
    x = rng.standard_normal((t, c)).astype(np.float32)
    u = rng.standard_normal((t, max(rank, 1))).astype(np.float32)
    lf = rng.standard_normal((max(rank, 1), n)).astype(np.float32)
    gpu.set_gemm_passes(3)
    gpu.upload_quant(0x79, raw, Q8_0, rows, cols)

    def product(i, j):
        if rank == 0:
            return gpu.qgemm_dx(0x79, x[i:j], cols) if which else gpu.qgemm_fwd(0x79, x[i:j], rows)
        xd, ud, ld, out = gpu.to_dev(x[i:j].copy()), gpu.to_dev(u[i:j].copy()), gpu.to_dev(lf), gpu.empty_dev((j - i, n))
        gpu.op("qgemm_lora_dev", which, 0x79, xd, j - i, ud, rank, ld, n, 1, rank, 1.5, out)
        y = out.get()
        for a in (xd, ud, ld, out):
            a.free()
        return y

    y = product(0, t)
    parts = np.concatenate([product(i, min(i + 7, t)) for i in range(0, t, 7)])
    gpu.evict(0x79)
    gpu.set_gemm_passes(1)
    np.testing.assert_array_equal(y, parts)
