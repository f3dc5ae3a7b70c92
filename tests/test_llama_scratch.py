"""The decoder's GEMM work memory covers every product its prompt chunks run,
by the sizes the launches use (no device: sizes only)."""
import itertools

import pytest

from rdlquant import llama as L

Q4_0, Q4_1, Q8_0, Q4_K, Q6_K = 2, 3, 8, 12, 14


def matrices(c, t):
    """(type, out, in) of a layer's matrices, joined as the model joins them."""
    q, kv = c.n_heads * c.head_dim, c.n_kv_heads * c.head_dim
    tq, tk, tv, to, tg, tu, td = (t.get((s, 0), Q4_0) for s in (L.WQ, L.WK, L.WV, L.WO, L.W_GATE, L.W_UP, L.W_DOWN))
    out = [(to, c.dim, q), (td, c.dim, c.ffn_dim)]
    if tq == tk == tv:
        out.append((tq, q + 2 * kv, c.dim))
    elif tq == tk:
        out += [(tq, q + kv, c.dim), (tv, kv, c.dim)]
    else:
        out += [(tq, q, c.dim), (tk, kv, c.dim), (tv, kv, c.dim)]
    return out + ([(tg, 2 * c.ffn_dim, c.dim)] if tg == tu else [(tg, c.ffn_dim, c.dim), (tu, c.ffn_dim, c.dim)])


TYPES = [{}, {(L.WV, 0): Q6_K}, {(L.WV, 0): Q8_0, (L.W_DOWN, 0): Q4_1}, {(L.WK, 0): Q8_0, (L.W_UP, 0): Q4_1},
         {(s, 0): Q4_K for s in (L.WQ, L.WK, L.WO, L.W_GATE, L.W_UP)}, {(s, 0): Q6_K for s in (L.W_GATE, L.W_UP)}]


# dim, heads, KV heads, head_dim, FFN: wide and narrow [Wq; Wk] beside wide and narrow FFNs
@pytest.mark.parametrize("dim,heads,kv,hd,ffn", [
    (2048, 16, 8, 128, 8192), (8192, 64, 16, 128, 14336), (6144, 48, 48, 128, 16384), (6144, 48, 48, 128, 8192),
    (1024, 8, 8, 128, 2560), (4096, 32, 8, 128, 14336), (4096, 32, 32, 128, 11008), (512, 8, 2, 64, 1024),
    (256, 64, 64, 256, 256), (16384, 2, 1, 256, 16384), (256, 4, 1, 64, 16384)])
@pytest.mark.parametrize("types", TYPES, ids=range(len(TYPES)))
def test_scratch_covers_every_chunk(rq, dim, heads, kv, hd, ffn, types):
    for mb in (1, 5, 33, 64, 128, 300, 1100):
        c = L.LlamaConfig(dim=dim, n_layers=1, n_heads=heads, n_kv_heads=kv, head_dim=hd, ffn_dim=ffn, vocab=64,
                          max_seq=64, max_batch=mb)
        have = L.gemm_scratch_bytes(c, types)
        rows = sorted({*range(1, min(mb, 80) + 1), *(m for m in (128, 255, 256, 300, 1023, 1024, mb) if m <= mb)})
        for (t, n, k), m, mode in itertools.product(matrices(c, types), rows, (rq.MODE_FLOAT, rq.MODE_NATIVE)):
            need = L.product_scratch_bytes(t, m, n, k, mode)
            assert need <= have, (mb, m, t, n, k, mode, need, have)


def test_scratch_queries_reject_what_create_rejects(rq):
    with pytest.raises(rq.InvalidData):
        L.gemm_scratch_bytes(L.LlamaConfig(dim=33, n_layers=1))
    with pytest.raises(rq.QuantError):
        L.gemm_scratch_bytes(L.LlamaConfig(dim=96, n_layers=1, head_dim=96, n_heads=1, n_kv_heads=1, ffn_dim=256),
                             {(L.WQ, 0): Q6_K})
    with pytest.raises(rq.QuantError):
        L.product_scratch_bytes(5, 8, 64, 64)
