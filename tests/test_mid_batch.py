"""The middle-batch GEMM (17 rows to a few hundred, ``awq_mid_kernel.h``) through ``ops.gemm``, at the edges
of its tiles: row tiles of 32 to 128 rows, a partial column tile, K that ends inside a stage, K ranges,
shares without work.  Every output within one ulp (of max(|y|, 1)) of the float64 product with the weights
that the path multiplies: unrounded up to 64 rows, rounded once to the activation dtype above; bitwise
the same on a second call."""
import numpy as np
import pytest
import torch

from kernel_paths import decode_serves
from oracle import awq_oracle as O
from oracle.gen import make_awq_problem

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _expected(p, x, sc, G, zp, half, bias=None):
    M, N = x.shape[0], p["qweight"].shape[1] * 8
    out = "float32" if decode_serves(M, N, G) else half
    w = O.dequant_awq(p["qweight"], sc.float().numpy(), p["qzeros"] if zp else None, G, out_dtype=out, zero_point=zp)
    w = O.bf16_bits_to_f32(w) if out == "bfloat16" else w
    y = x.double().numpy() @ w.astype(np.float64)
    return y if bias is None else y + bias.double().numpy()


@pytest.mark.parametrize("M,K,N,G", [
    (17, 2048, 136, 64), (25, 1024, 8, 128), (32, 4096, 264, 128), (33, 544, 520, 32), (48, 1088, 1000, 64),
    (49, 2080, 264, 32), (64, 3072, 1024, 128), (65, 512, 2056, 128), (80, 96, 24, 32), (97, 1088, 136, 64),
    (128, 2080, 520, 32), (129, 2048, 1024, 256), (200, 1408, 392, 128), (400, 1024, 264, 64)])
@pytest.mark.parametrize("act,sdt,zp", [(torch.float16, torch.float16, True), (torch.float16, torch.float16, False),
                                        (torch.float16, torch.bfloat16, True), (torch.bfloat16, torch.float16, True),
                                        (torch.bfloat16, torch.bfloat16, False)])
def test_mid_batch_vs_oracle(M, K, N, G, act, sdt, zp):
    from litevllm_amd import ops
    print(f"mid batch M={M} K={K} N={N} G={G} {act} scales={sdt} zp={zp}", flush=True)
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K + N, with_bias=True)
    x, sc = torch.from_numpy(p["x"]).to(act), torch.from_numpy(p["scales"]).to(sdt)
    b = torch.from_numpy(p["bias"])
    qz = torch.from_numpy(p["qzeros"]).to(DEV) if zp else None
    args = (x.to(DEV), torch.from_numpy(p["qweight"]).to(DEV), sc.to(DEV), qz, G)
    y, y2 = (ops.gemm(*args, bias=b.to(DEV), layout="autoawq") for _ in range(2))
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    ye = _expected(p, x, sc, G, zp, "float16" if act == torch.float16 else "bfloat16", b)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if act == torch.float16 else 7))
    err = np.abs(y.double().cpu().numpy() - ye) / ulp
    assert err.max() <= 1.0, float(err.max())


@pytest.mark.parametrize("M", [40, 200])
def test_mid_batch_strides_capture_and_scratch(M):
    """Strided rows in and out, replays of a captured call, the allocation-free entry point, and a
    workspace that does not hold the plan's K ranges (the decode kernels up to 64 rows where it holds theirs,
    the prefill kernel above)."""
    from litevllm_amd import _lib as L
    from litevllm_amd import ops
    K, N, G = 2048, 512, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M)
    t = {k: torch.from_numpy(v).to(DEV) for k, v in p.items() if isinstance(v, np.ndarray)}
    call = lambda x, out=None: ops.gemm(x, t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq", out=out)
    y = call(t["x"])
    xb = torch.zeros((M, K + 64), dtype=torch.float16, device=DEV)
    xb[:, :K] = t["x"]
    ob = torch.full((M, N + 64), 7.0, dtype=torch.float16, device=DEV)
    call(xb[:, :K], ob[:, :N])
    assert torch.equal(ob[:, :N], y) and bool((ob[:, N:] == 7.0).all())
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        yg = call(t["x"])
    for _ in range(3):
        yg.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(yg, call(t["x"]))
    lib = L.load()
    qk = ops.pack_decode_stream(t["qweight"])
    ws = int(lib.awq_w4a16_gemm_workspace_bytes(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM))
    assert ws > 65536  # K ranges
    out = torch.empty_like(y)
    head = (t["x"].data_ptr(), K, qk.data_ptr(), t["scales"].data_ptr(), t["qzeros"].data_ptr(), None, out.data_ptr(), N, M, N, K,
            G, 0, L.LAYOUT_DECODE_STREAM, L.DTYPE_F16, L.DTYPE_F16, L.DTYPE_NONE)
    st = int(torch.cuda.current_stream().cuda_stream)
    small = torch.zeros(ws - 4, dtype=torch.uint8, device=DEV)
    assert lib.awq_w4a16_gemm(*head, small.data_ptr(), ws - 4, st) == 0
    # other kernels, the same products in another order
    assert float((out.float() - y.float()).abs().max()) <= 2 * float(y.float().abs().max()) * 2.0 ** -10
    # without one: 64 rows and K = 2048 need ranges on the decode kernels too
    assert lib.awq_w4a16_gemm(*head, None, 0, st) == (L.ERR_WORKSPACE if M <= 64 else 0)
    assert lib.awq_w4a16_gemm_noalloc(*head, st) == 0
    if M <= 64:
        assert torch.equal(out, y)
    else:  # the prefill kernel: the same products in another order
        assert float((out.float() - y.float()).abs().max()) <= 2 * float(y.float().abs().max()) * 2.0 ** -10


@pytest.mark.parametrize("M", [32, 57])
def test_mid_batch_without_workspace_where_decode_needs_none(M):
    """K = 1504: the plan cuts K, the decode kernels' plan does not, so a call without a workspace runs."""
    from litevllm_amd import _lib as L
    from litevllm_amd import ops
    K, N, G = 1504, 512, 32
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M)
    t = {k: torch.from_numpy(v).to(DEV) for k, v in p.items() if isinstance(v, np.ndarray)}
    lib, qk = L.load(), ops.pack_decode_stream(t["qweight"])
    assert int(lib.awq_w4a16_gemm_workspace_bytes(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM)) > 65536
    out = torch.empty((M, N), dtype=torch.float16, device=DEV)
    rc = lib.awq_w4a16_gemm(t["x"].data_ptr(), K, qk.data_ptr(), t["scales"].data_ptr(), t["qzeros"].data_ptr(), None, out.data_ptr(),
                            N, M, N, K, G, 0, L.LAYOUT_DECODE_STREAM, L.DTYPE_F16, L.DTYPE_F16, L.DTYPE_NONE, None, 0,
                            int(torch.cuda.current_stream().cuda_stream))
    assert rc == 0
    ye = _expected(p, t["x"].cpu(), t["scales"].cpu(), G, True, "float16")
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - 10)
    assert (np.abs(out.double().cpu().numpy() - ye) / ulp).max() <= 1.0


@pytest.mark.parametrize("M,K,N", [(20, 1024, 264), (25, 1056, 136), (32, 2080, 264), (40, 1024, 520), (64, 2048, 1000)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_outlier_and_infinite_activations_in_groups_of_32(M, K, N, dt):
    """Groups of 32: the operands are q - z themselves, so an activation far above its row's others adds nothing
    where q == z, and an infinite one gives +-inf wherever q != z and NaN (0 * inf) only where q == z."""
    from litevllm_amd import ops
    print(f"outliers M={M} K={K} N={N} {dt}", flush=True)
    G = 32
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K + N)
    x = torch.from_numpy(p["x"]).to(dt)
    x[::2, 100] = 2e4
    x[1, 40], x[3, 41] = float("inf"), float("-inf")
    w = tuple(torch.from_numpy(p[k]).to(DEV) for k in ("qweight", "scales", "qzeros")) + (G,)
    y = ops.gemm(x.to(DEV), *w, layout="autoawq").double().cpu().numpy()
    with np.errstate(invalid="ignore"):  # 0 * inf
        ye = _expected(p, x, torch.from_numpy(p["scales"]), G, True, "float16")
    fin = np.isfinite(ye)
    assert np.array_equal(y[~fin], ye[~fin], equal_nan=True)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye[fin]), 1.0))) - (10 if dt == torch.float16 else 7))
    assert (np.abs(y[fin] - ye[fin]) / ulp).max() <= 1.0


# (M, K, N, G) on either side of the line from which 17 .. 32 rows leave the decode kernels
DECODE_SIDE = [(17, 544, 256, 32), (24, 1504, 512, 32), (32, 1504, 1032, 32), (20, 1024, 4096, 128), (27, 1280, 512, 128), (32, 1024, 264, 64), (32, 1024, 2560, 32),
               (32, 2048, 6152, 32), (32, 4096, 3080, 32), (32, 8192, 136, 32), (29, 2048, 24576, 64), (27, 2048, 24576, 128),
               (32, 2048, 32776, 128), (30, 2560, 34816, 128)]
MID_SIDE = [(17, 1536, 264, 64), (25, 1248, 1024, 32), (17, 2048, 4096, 128), (28, 1280, 512, 128), (25, 4096, 3072, 32), (32, 2048, 6144, 32),
            (30, 2048, 24576, 64), (28, 2048, 24576, 128), (31, 2560, 34816, 128), (33, 544, 256, 32)]


@pytest.mark.parametrize("shape,mid", [(s, False) for s in DECODE_SIDE] + [(s, True) for s in MID_SIDE])
def test_rows_from_which_the_kernel_takes_a_call(shape, mid):
    """Each shape on the kernel that measured faster, and its outputs as test_mid_batch_vs_oracle holds them."""
    from litevllm_amd import _lib as L
    from litevllm_amd import ops
    M, K, N, G = shape
    print(f"mid or decode {shape}", flush=True)
    ws = int(L.load().awq_w4a16_gemm_workspace_bytes(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM))
    route = L.load().awq_w4a16_gemm_kernel(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM, ws, None, None)
    assert route == (L.KERNEL_MID if mid else L.KERNEL_DECODE)
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K)
    x = torch.from_numpy(p["x"]).to(torch.bfloat16)
    w = tuple(torch.from_numpy(p[k]).to(DEV) for k in ("qweight", "scales", "qzeros")) + (G,)
    y = ops.gemm(x.to(DEV), *w, layout="autoawq", decode_layout="stream" if M <= 32 else None).double().cpu().numpy()
    ye = _expected(p, x, torch.from_numpy(p["scales"]), G, True, "bfloat16")
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - 7)
    assert (np.abs(y - ye) / ulp).max() <= 1.0


# (M, K, N, G, rows of a row tile, K ranges): every instantiation above 64 rows, one row past the tile below where
# that selects it, ragged columns, K that ends inside a stage or unit, several row tiles, K ranges
ROW_TILES = [
    (65, 544, 16656, 32, 80, 1), (65, 576, 16664, 64, 80, 1), (75, 640, 16776, 128, 80, 1), (200, 2080, 2752, 32, 80, 3),
    (400, 4096, 520, 128, 80, 8), (81, 1056, 16656, 32, 96, 1), (96, 576, 16656, 64, 96, 1), (81, 768, 16664, 256, 96, 1),
    (97, 1056, 16656, 32, 112, 1), (97, 1088, 16664, 64, 112, 1), (111, 1152, 16656, 128, 112, 1), (100, 4160, 5480, 32, 112, 5),
    (113, 1088, 16656, 64, 128, 1), (128, 1152, 16664, 128, 128, 1), (113, 1280, 16656, 256, 128, 1), (120, 8192, 5480, 128, 128, 4)]


@pytest.mark.parametrize("M,K,N,G,tile,ranges", ROW_TILES)
def test_row_tiles_above_64_rows(M, K, N, G, tile, ranges):
    import ctypes
    from litevllm_amd import _lib as L
    from litevllm_amd import ops
    print(f"row tiles M={M} K={K} N={N} G={G} tile={tile} ranges={ranges}", flush=True)
    t, r = ctypes.c_int32(), ctypes.c_int32()
    ws = int(L.load().awq_w4a16_gemm_workspace_bytes(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM))
    assert L.load().awq_w4a16_gemm_kernel(M, N, K, G, 0, L.LAYOUT_DECODE_STREAM, ws, t, r) == L.KERNEL_MID
    assert (t.value, r.value) == (tile, ranges)
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K)
    qw, qz = (torch.from_numpy(p[k]).to(DEV) for k in ("qweight", "qzeros"))
    for act, sdt in ((torch.float16, torch.float16), (torch.bfloat16, torch.float16), (torch.float16, torch.bfloat16)):
        if sdt == torch.bfloat16 and K > 1200:  # the operand path alone: the short shapes do
            continue
        x, sc = torch.from_numpy(p["x"]).to(act), torch.from_numpy(p["scales"]).to(sdt)
        y = ops.gemm(x.to(DEV), qw, sc.to(DEV), qz, G, layout="autoawq").double().cpu().numpy()
        ye = _expected(p, x, sc, G, True, "float16" if act == torch.float16 else "bfloat16")
        ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if act == torch.float16 else 7))
        assert (np.abs(y - ye) / ulp).max() <= 1.0, (act, sdt)
