"""Decode calls with more 128-column tiles than CUs (blocks of half the waves, two per CU): within one ulp
of the exact product of the unrounded weights at a ragged width, the gated epilogue included through its own
tests' shapes; a row-exact launch equals lone calls bit for bit."""
import numpy as np
import pytest
import torch

from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K,N,G", [(1, 256, 32776, 128), (1, 288, 65544, 32), (2, 256, 33000, 64), (16, 128, 65536, 128),
                                     (20, 96, 32776, 32), (3, 64, 65672, 64)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_more_tiles_than_cus(M, K, N, G, dt):
    from litevllm_amd import ops
    print(f"many tiles M={M} K={K} N={N} G={G} {dt}", flush=True)
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K)
    t = {k: torch.from_numpy(v).to(DEV) for k, v in p.items() if isinstance(v, np.ndarray)}
    x = t["x"].to(dt)
    w = (t["qweight"], t["scales"], t["qzeros"], G)
    y = ops.gemm(x, *w, layout="autoawq")
    ye = x.double().cpu().numpy() @ O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], G, out_dtype="float32").astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if dt == torch.float16 else 7))
    assert (np.abs(y.double().cpu().numpy() - ye) / ulp).max() <= 1.0
    if M <= 3:
        rows = ops.gemm_rows_exact(x, *w, layout="autoawq")
        for m in range(M):
            assert torch.equal(rows[m:m + 1], ops.gemm(x[m:m + 1], *w, layout="autoawq"))
