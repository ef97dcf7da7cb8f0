"""The prefill stream kernel's stage loop at its steady state: many 64-row stages, groups of one to several stage
pairs, a K that ends on half a stage, both block widths.  Calls of few columns reach it through the C entry
without a workspace (their middle-batch plan needs one).  Every output within one ulp (of max(|y|, 1)) of the
float64 product with the weights rounded once."""
import numpy as np
import pytest
import torch

from litevllm_amd import _lib as L
from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


@pytest.mark.parametrize("M,K,N,G", [(200, 2048, 512, 128), (300, 2048, 264, 256), (300, 2080, 520, 32), (257, 4160, 136, 64),
                                     (130, 4096, 520, 1024), (300, 1024, 24576, 128), (512, 1056, 24584, 32), (300, 1152, 24584, 64)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_many_stages(M, K, N, G, dt):
    from litevllm_amd import ops
    print(f"prefill stages M={M} K={K} N={N} G={G} {dt}", flush=True)
    lib = L.load()
    assert lib.awq_w4a16_gemm_kernel(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM, 0, None, None) == L.KERNEL_PREFILL_STREAM
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K, with_bias=True)
    t = {k: torch.from_numpy(p[k]).to(DEV) for k in ("qweight", "scales", "qzeros", "bias")}
    x = torch.from_numpy(p["x"]).to(dt)
    xd, qk, y = x.to(DEV), ops.pack_decode_stream(t["qweight"]), torch.empty((M, N), dtype=dt, device=DEV)
    code = L.DTYPE_F16 if dt == torch.float16 else L.DTYPE_BF16
    rc = lib.awq_w4a16_gemm(xd.data_ptr(), K, qk.data_ptr(), t["scales"].data_ptr(), t["qzeros"].data_ptr(), t["bias"].data_ptr(),
                            y.data_ptr(), N, M, N, K, G, 0, L.LAYOUT_DECODE_STREAM, code, L.DTYPE_F16, L.DTYPE_F16, None, 0,
                            int(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    half = "float16" if dt == torch.float16 else "bfloat16"
    w = O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], G, out_dtype=half)
    w = O.bf16_bits_to_f32(w) if half == "bfloat16" else w
    ye = x.double().numpy() @ w.astype(np.float64) + p["bias"].astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if dt == torch.float16 else 7))
    assert (np.abs(y.double().cpu().numpy() - ye) / ulp).max() <= 1.0
