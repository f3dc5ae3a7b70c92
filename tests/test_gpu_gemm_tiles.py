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
SHAPES = [(65, 1, 32), (65, 65, 96), (129, 63, 1056), (128, 1024, 4096), (66, 200, 4128), (80, 4096, 2080),
          (130, 6000, 544), (200, 14400, 96), (513, 4097, 288), (70, 40, 16416)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_q4_0_tiles(rq, orc, gpu, m, n, k):
    print(f"case q4_0 tiles m={m} n={n} k={k}", flush=True)
    x = synth.activations(m, k, m + n + k)
    w = synth.q4_0_weights(n, k, m + n)
    got = rq.matmul_f32_q4(x, w, m, k, n).reshape(m, n)
    rows = np.unique(np.linspace(0, m - 1, 24).astype(int))
    want = orc.matmul("q4", x[rows], w, len(rows), k, n, threads=16)
    check_parity(got[rows].reshape(-1), want, exact_f64(orc, "q4", x[rows], w, len(rows), k, n))


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
