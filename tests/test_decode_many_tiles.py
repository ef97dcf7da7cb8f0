"""Decode calls with more 128-column tiles than CUs (blocks of half the waves, two per CU): within one ulp
of the exact product of the unrounded weights at a ragged width, with several groups a wave and several DMA
instructions of staged activations, and through the gated epilogue; a row-exact launch equals lone calls bit for
bit."""
import numpy as np
import pytest
import torch

from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K,N,G", [(1, 256, 32776, 128), (1, 5376, 32776, 128), (1, 4128, 33800, 32), (2, 4096, 32776, 64),
                                     (1, 288, 65544, 32), (2, 256, 33000, 64), (16, 128, 65536, 128),
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


@pytest.mark.parametrize("M,K,I,G", [(1, 256, 16392, 128), (1, 5376, 16456, 32), (2, 576, 16392, 64), (8, 256, 20488, 128),
                                     (17, 1056, 16392, 32), (24, 512, 32776, 128)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_gated_epilogue_with_more_tiles_than_cus(M, K, I, G, dt):
    from litevllm_amd import ops
    print(f"gated many tiles M={M} K={K} I={I} G={G} {dt}", flush=True)
    pg, pu = (make_awq_problem(M=M, K=K, N=I, group_size=G, seed=s) for s in (M, M + 1))
    t = lambda a: torch.from_numpy(a).to(DEV)
    x = torch.from_numpy(pg["x"]).to(dt)
    y = ops.gate_up_act(x.to(DEV), t(pg["qweight"]), t(pu["qweight"]), t(pg["scales"]), t(pu["scales"]), G,
                        gate_qzeros=t(pg["qzeros"]), up_qzeros=t(pu["qzeros"]), activation="silu", layout="autoawq",
                        decode_layout="stream")
    wg, wu = (O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], G, out_dtype="float32") for p in (pg, pu))
    xd = x.double().numpy()
    g, u = xd @ wg.astype(np.float64), xd @ wu.astype(np.float64)
    ye = g / (1.0 + np.exp(-g)) * u
    # the gate's and the up product's fp32 sums each carry their own error into the product
    e32 = 2.0 ** -23 * np.sqrt(K) * (np.abs(xd) @ np.abs(wg) * np.abs(u) + np.abs(xd) @ np.abs(wu) * np.abs(g))
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if dt == torch.float16 else 7))
    assert (np.abs(y.double().cpu().numpy() - ye) <= ulp + e32).all()
