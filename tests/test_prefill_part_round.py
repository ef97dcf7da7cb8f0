"""Prefill calls whose last round of 256-column blocks is a part round, at row-tile counts that do not divide the
CUs (3, 5, 7): the rest of the columns runs as 128-column blocks.  Every output within one ulp (of max(|y|, 1))
of the float64 product with the weights rounded once."""
import numpy as np
import pytest
import torch

from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K,N,G", [(520, 128, 25608, 128), (768, 96, 22792, 32), (1100, 64, 14600, 64), (1700, 64, 9992, 64)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_part_round_at_odd_row_tiles(M, K, N, G, dt):
    from litevllm_amd import ops
    print(f"part round M={M} K={K} N={N} G={G} {dt}", flush=True)
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K)
    t = {k: torch.from_numpy(v).to(DEV) for k, v in p.items() if isinstance(v, np.ndarray)}
    x = t["x"].to(dt)
    y = ops.gemm(x, t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq")
    half = "float16" if dt == torch.float16 else "bfloat16"
    w = O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], G, out_dtype=half)
    w = O.bf16_bits_to_f32(w) if half == "bfloat16" else w
    ye = x.double().cpu().numpy() @ w.astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if dt == torch.float16 else 7))
    assert (np.abs(y.double().cpu().numpy() - ye) / ulp).max() <= 1.0


@pytest.mark.parametrize("K", [480, 512])
def test_part_round_from_k_512_on(K):
    """Both sides of the K from which such row-tile counts take the part round."""
    test_part_round_at_odd_row_tiles(768, K, 23048, 32, torch.float16)
