"""The tile GEMM (prompts) at the edges of its tiles, K slices and K groups:
every tile shape, ragged rows and columns, odd block counts, split and
unsplit, on both combines and under graph replay."""
import numpy as np
import pytest

from parity import check_parity, exact_f64
from rdlquant import synth

pytestmark = pytest.mark.gpu

# smallest (one block, one column), both sides of a 64-row x tile and a 64-column
# weight tile, odd block counts (blocks 2 bytes past a dword, the matrix ending
# inside one), K in 16 / 8 / 4 / 2 slices with a ragged last one, 256 x 128 tiles,
# and rows longer than one workgroup's registers hold (k > 16384)
# (the rows before 257 with k <= 2048 stay on the small-tile kernel)
SHAPES = [(65, 1, 32), (65, 1, 4096), (65, 65, 2080), (129, 63, 4128), (128, 1024, 4096), (80, 4096, 2080),
          (257, 130, 96), (257, 6000, 544), (300, 14400, 96), (513, 4097, 288), (2049, 65, 32), (70, 40, 16416)]


@pytest.mark.parametrize("kind,dtype", [("q4", 2), ("q8", 8)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_tiles(rq, orc, gpu, kind, dtype, m, n, k):
    print(f"case {kind} tiles m={m} n={n} k={k}", flush=True)
    x = synth.activations(m, k, m + n + k)
    w = synth.weights(dtype, n, k, m + n)
    got = getattr(rq, f"matmul_f32_{kind}")(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 24).astype(int))
    want = orc.matmul(kind, x[rows], w, len(rows), k, n, threads=16)
    check_parity(got[rows].reshape(-1), want, exact_f64(orc, kind, x[rows], w, len(rows), k, n))


@pytest.mark.parametrize("m,n,k", [(128, 1024, 4096), (100, 4096, 1024)])
def test_split_tiles_combines_and_replays_agree(rq, gpu, m, n, k):
    # the XCD-local and the agent-coherent combine and a captured call give the
    # same bits, call after call (the counters return to zero)
    import torch
    print(f"case split tiles m={m} n={n} k={k}", flush=True)
    w = rq.Weight.upload(synth.q4_0_weights(n, k, 5), rq.DTYPE_Q4_0, n, k)
    x = torch.from_numpy(synth.activations(m, k, 6)).to(gpu)

    def product(stream):
        y = torch.full((m, n), np.nan, device=gpu)
        w.forward_dev(x.data_ptr(), m, y.data_ptr(), rq.MODE_FLOAT, stream)
        return y

    main = torch.cuda.current_stream().cuda_stream
    want = product(main)
    try:
        rq.set_gemm_combine(rq.COMBINE_COHERENT)
        coherent = [product(main) for _ in range(3)]
    finally:
        rq.set_gemm_combine(rq.COMBINE_AUTO)
    local = [product(main) for _ in range(3)]
    torch.cuda.synchronize()
    g, side, y = torch.cuda.CUDAGraph(), torch.cuda.Stream(), torch.empty(m, n, device=gpu)
    with torch.cuda.graph(g, stream=side):
        w.forward_dev(x.data_ptr(), m, y.data_ptr(), rq.MODE_FLOAT, side.cuda_stream)
    for got in coherent + local:
        assert torch.equal(got, want)
    for _ in range(3):
        y.fill_(np.nan)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        product(main)
        torch.cuda.synchronize()
    w.free()
