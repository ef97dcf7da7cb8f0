"""GPU parity: HIP kernels (through the C ABI) against the CPU oracle.

Bars (stated per test):
  * dequantized weights: bit-exact (uint16 patterns / fp32 values equal);
  * GEMM outputs vs the exact oracle (float64 sum of exact products with the weights the
    serving kernel uses, see ``_w_used``): every element within 1 fp16 ulp of the exact
    value (ulp taken at max(|y|, 1), see ``oracle.awq_oracle.fp16_ulp``), i.e. fp32
    accumulation plus one final rounding;
  * GEMM outputs vs the reference's own CPU path (dequant + F.linear): elementwise
    |d| <= max(2e-2, 1 ulp(|ref|)) and mean relative error sum|d|/sum|ref| <= 1e-3.
    The 2e-2 bound alone is below one fp16 ulp for |y| >= 32 (one rounding flip
    between two fp32 summation orders already exceeds it), hence the ulp clause.
"""
import numpy as np
import pytest
import torch

from oracle import awq_oracle as O
from oracle import ref_cpu as R
from oracle.gen import make_awq_problem
from kernel_paths import decode_serves

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _lib():
    from litevllm_amd import ops
    return ops


def _to_dev(p):
    return {k: (torch.from_numpy(v).to(DEV) if isinstance(v, np.ndarray) else v) for k, v in p.items()}


def _note(msg):
    print(msg, flush=True)


def _w_used(p, M, G, zp=True, half="float16"):
    """Dequantized [K, N] weights as the kernel serving the call multiplies them: the skinny
    kernels (M <= 32, and 32-row chunks of them a little above) feed the MFMA the exact
    integers q - z and scale each group's fp32 sum, so their weights enter unrounded, as in the
    reference's M = 1 branch (awq_fused_gemm.py:1966-1971); the prefill kernels round them to
    the activation dtype first, as the reference's tl.dot branch does (1973-1976)."""
    N = int(p["qweight"].shape[1]) * 8
    out = "float32" if decode_serves(M, N, G) else half
    w = O.dequant_awq(p["qweight"], p["scales"], p["qzeros"] if zp else None, G, out_dtype=out, zero_point=zp)
    return O.bf16_bits_to_f32(w) if out == "bfloat16" else w


def _check_vs_exact(y, ye, what):
    rep = O.error_report(y, ye)
    assert rep["max_ulp"] <= 1.0, (what, rep)
    return rep


def _check_vs_ref(y, yr, what):
    y = np.asarray(y, dtype=np.float64)
    yr = np.asarray(yr, dtype=np.float64)
    d = np.abs(y - yr)
    bound = np.maximum(2e-2, O.fp16_ulp(yr, floor=2.0 ** -14))
    assert (d <= bound).all(), (what, float(d.max()), float((d / bound).max()))
    mrel = float(d.sum() / max(np.abs(yr).sum(), 1e-30))
    assert mrel <= 1e-3, (what, mrel)


# ------------------------------------------------------------------ dequant
@pytest.mark.parametrize("layout", ["autoawq", "kn_seq", "ref"])
@pytest.mark.parametrize("zp", [True, False])
@pytest.mark.parametrize("out_dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("scale_dtype", [torch.float16, torch.bfloat16])
def test_dequant_bit_exact(layout, zp, out_dtype, scale_dtype):
    ops = _lib()
    _note(f"dequant layout={layout} zp={zp} out={out_dtype} scales={scale_dtype}")
    rng = np.random.default_rng(11)
    K, N, G = 512, 384, 64
    W = rng.integers(0, 16, size=(K, N), dtype=np.int32)
    Z = rng.integers(0, 16, size=(K // G, N), dtype=np.int32)
    S = (np.abs(rng.standard_normal((K // G, N))) * 0.02 + 1e-4).astype(np.float32)
    S_t = torch.from_numpy(S).to(scale_dtype)
    S_np = S_t.float().numpy()                     # the exact scale values used
    # expected: one rounding of the exact product, by layout orientation
    exact = (W.reshape(K // G, G, N) - (Z[:, None, :] if zp else 8)).astype(np.float64) * S_np[:, None, :].astype(np.float64)
    exact = exact.reshape(K, N)
    if layout == "autoawq":
        qw, qz, sc = O.pack_awq(W), O.pack_awq(Z), S_t
    elif layout == "kn_seq":
        qw, qz, sc = O.pack_ref(W), O.pack_ref(Z), S_t
    else:
        qw, qz = O.pack_ref(np.ascontiguousarray(W.T)), O.pack_ref(np.ascontiguousarray(Z.T))
        sc = S_t.t().contiguous()
        exact = exact.T
    out = ops.dequant(torch.from_numpy(qw).to(DEV), sc.to(DEV),
                      torch.from_numpy(qz).to(DEV) if zp else None, G, layout=layout,
                      out_dtype=out_dtype).cpu()
    want = torch.from_numpy(np.ascontiguousarray(exact)).to(out_dtype)
    assert torch.equal(out.view(torch.int16) if out_dtype != torch.float32 else out.view(torch.int32),
                       want.view(torch.int16) if out_dtype != torch.float32 else want.view(torch.int32))


def test_dequant_matches_numpy_oracle_config0():
    ops = _lib()
    p = make_awq_problem(M=1, K=2048, N=5632, group_size=128, seed=0)
    t = _to_dev(p)
    w = ops.dequant(t["qweight"], t["scales"], t["qzeros"], 128, layout="autoawq").cpu().numpy()
    w_ref = O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], 128)
    assert np.array_equal(w.view(np.uint16), w_ref.view(np.uint16))


def test_repack_ref_to_autoawq_on_device():
    ops = _lib()
    p = make_awq_problem(M=1, K=1024, N=512, group_size=128, seed=1)
    qr, zr, sr = O.repack_awq_to_ref(p["qweight"], p["qzeros"], p["scales"])
    qw, sc, qz = ops.repack_ref_to_autoawq(torch.from_numpy(qr).to(DEV), torch.from_numpy(sr).to(DEV),
                                           torch.from_numpy(zr).to(DEV), 128)
    assert np.array_equal(qw.cpu().numpy(), p["qweight"])
    assert np.array_equal(qz.cpu().numpy(), p["qzeros"])
    assert np.array_equal(sc.cpu().numpy(), p["scales"])


# ------------------------------------------------------------------ GEMM shapes
SHAPES = [
    # (M, K, N, G)  -- skinny (M <= 32) and prefill kernels, partial column tiles
    (1, 256, 512, 128), (1, 2048, 5632, 128), (2, 512, 4096, 128), (3, 1024, 1000 // 8 * 8, 64),
    (5, 512, 264, 32), (8, 4096, 1024, 128), (16, 1024, 2048, 128), (17, 512, 520, 128),
    (32, 2048, 1536, 128), (33, 512, 512, 128), (64, 1024, 768, 64), (100, 512, 2056, 128),
    (256, 1024, 1024, 128), (300, 2048, 512, 128),
    # M = 5 .. 8 with two 16-column tiles per CU: the narrow kernel under auto
    (6, 4096, 6144, 128), (8, 2048, 8192, 64),
    # one tile per CU over a long K (M <= 4 up to K = 14336, M <= 8 up to 8192): narrow too
    (4, 8192, 4096, 128), (8, 8192, 2048, 64),
    # three and four 16-column tiles per CU (M <= 2, K <= 4096): narrow under auto
    (1, 2048, 12288, 128), (2, 4096, 16384, 64), (3, 2048, 16384, 64), (5, 2048, 12288, 128),
    # group size 32 in the prefill kernel: two groups per 64-row stage, and K % 64 == 32
    (40, 2080, 520, 32), (64, 1024, 1024, 32), (300, 96, 264, 32),
    # group size 256: four stages per group in the prefill kernel (constants once per pair of
    # stages), also for M <= 32, which the decode kernels do not take at this group size
    (8, 1024, 512, 256), (48, 1024, 520, 256), (300, 2048, 264, 256),
]


@pytest.mark.parametrize("M,K,N,G", SHAPES)
@pytest.mark.parametrize("stream", [None, False])
def test_gemm_autoawq_vs_oracle(M, K, N, G, stream):
    ops = _lib()
    _note(f"gemm autoawq M={M} K={K} N={N} G={G} stream={stream}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M * 7 + N)
    t = _to_dev(p)
    y = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq",
                 decode_stream=stream).cpu().numpy()
    w = _w_used(p, M, G)                                                 # [K, N]
    _check_vs_exact(y, O.linear_exact(p["x"], w.T), f"M={M} K={K} N={N}")
    qr, zr, sr = O.repack_awq_to_ref(p["qweight"], p["qzeros"], p["scales"]) if (K // G) % 8 == 0 else (None,) * 3
    if qr is not None:
        yr = R.awq_linear_cpu(torch.from_numpy(p["x"]), torch.from_numpy(qr), torch.from_numpy(sr),
                              torch.from_numpy(zr), G).numpy()
        _check_vs_ref(y, yr, f"M={M} K={K} N={N}")


@pytest.mark.parametrize("M,K,N,G", [(128, 2048, 8192, 128), (256, 4096, 1024, 64), (384, 1024, 2056, 128),
                                     (200, 512, 512, 32), (300, 2080, 520, 32)])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_prefill_k_ranges(M, K, N, G, dt):
    """Calls of 128 .. 384 rows over few columns, whose K is cut in ranges (the middle-batch kernel's:
    fp32 partials summed in range order by a second launch; K % 64 == 32 ends on a half stage):
    within 1 ulp of the exact oracle on the fp16-rounded weights, bias added once, bitwise
    reproducible."""
    ops = _lib()
    _note(f"prefill k ranges M={M} K={K} N={N} G={G} {dt}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + K + G)
    t = _to_dev(p)
    x = t["x"].to(dt)
    b = torch.randn(N, generator=torch.Generator().manual_seed(N)).to(dt)
    y = ops.gemm(x, t["qweight"], t["scales"], t["qzeros"], G, bias=b.to(DEV), layout="autoawq")
    y2 = ops.gemm(x, t["qweight"], t["scales"], t["qzeros"], G, bias=b.to(DEV), layout="autoawq")
    torch.cuda.synchronize()
    assert torch.equal(y, y2)
    half = "float16" if dt == torch.float16 else "bfloat16"
    w = _w_used(p, M, G, half=half)
    xe = x.float().cpu().numpy()
    ye = O.linear_exact(xe, w.T, b.float().double().numpy())
    yv = y.float().cpu().numpy()
    if dt == torch.float16:
        _check_vs_exact(yv, ye, f"M={M} K={K} N={N} G={G}")
    else:  # one bf16 rounding of the fp32 sum: |d| <= 1 bf16 ulp of max(|y|, 1)
        ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - 7)
        assert (np.abs(yv - ye) <= ulp).all(), float((np.abs(yv - ye) / ulp).max())


@pytest.mark.parametrize("M,layout", [(1, None), (4, None), (16, None), (1, "stream"), (16, "stream"),
                                      (64, None), (512, None)])
def test_gemm_strided_rows(M, layout):
    """Activation rows at a stride past K (read in place through lda, as the reference's kernel
    takes stride_am, awq_fused_gemm.py:1074) and output rows at a stride past N (ldc): the same
    bits as contiguous rows on the narrow, stream and prefill kernels, nothing written past N."""
    ops = _lib()
    K, N, G = 1024, 2048, 128
    _note(f"gemm strided rows M={M} layout={layout}")
    t = _to_dev(make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + 3))
    y = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq", decode_layout=layout)
    xb = torch.zeros((M, K + 64), dtype=torch.float16, device=DEV)
    xb[:, :K] = t["x"]
    ob = torch.full((M, N + 64), 7.0, dtype=torch.float16, device=DEV)
    ys = ops.gemm(xb[:, :K], t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq", decode_layout=layout,
                  out=ob[:, :N])
    torch.cuda.synchronize()
    assert ys.data_ptr() == ob.data_ptr()
    assert torch.equal(ys, y), (M, layout)
    assert bool((ob[:, N:] == 7.0).all())


@pytest.mark.parametrize("M", [1, 7, 40])
@pytest.mark.parametrize("bias_dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_gemm_bias(M, bias_dtype):
    ops = _lib()
    _note(f"gemm bias M={M} {bias_dtype}")
    K, N, G = 1024, 768, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=5)
    t = _to_dev(p)
    b = torch.randn(N, generator=torch.Generator().manual_seed(3)).to(bias_dtype)
    y = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, bias=b.to(DEV), layout="autoawq").cpu().numpy()
    w = _w_used(p, M, G)
    _check_vs_exact(y, O.linear_exact(p["x"], w.T, b.double().numpy()), f"bias M={M}")


@pytest.mark.parametrize("M,K,N", [(1, 1024, 512), (9, 512, 1024), (24, 512, 256), (128, 1024, 512)])
def test_gemm_bf16_activations(M, K, N):
    ops = _lib()
    _note(f"gemm bf16 M={M} K={K} N={N}")
    G = 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=9)
    t = _to_dev(p)
    xb = torch.from_numpy(p["x"]).to(torch.bfloat16)
    y = ops.gemm(xb.to(DEV), t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq").float().cpu().numpy()
    # decode path: unrounded weights; prefill: rounded once to bf16 from the exact product
    # (fused path, awq_fused_gemm.py:1966-1976)
    wb = _w_used(p, M, G, half="bfloat16")
    ye = xb.double().numpy() @ wb.astype(np.float64)
    # one bf16 rounding of the fp32 sum: |d| <= 1 bf16 ulp of max(|y|, 1)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - 7)
    assert (np.abs(y - ye) <= ulp).all(), float((np.abs(y - ye) / ulp).max())


@pytest.mark.parametrize("act,sdt", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float16),
                                     (torch.float16, torch.bfloat16), (torch.float16, torch.float16)])
@pytest.mark.parametrize("M,G", [(1, 128), (1, 64), (1, 32), (4, 128), (17, 32), (32, 64)])
@pytest.mark.parametrize("stream", ["stream", "narrow", False])
@pytest.mark.parametrize("zp", [True, False])
def test_decode_dtype_combinations(act, sdt, M, G, stream, zp):
    """Every activation / scale dtype pair through the decode kernel, stream copy or AutoAWQ
    layout, with and without zero points: within one ulp of the output dtype (at max(|y|, 1))
    of the exact sum over unrounded weights (q - z) * s, s taken in its own dtype."""
    ops = _lib()
    K, N = 2048, 1040
    _note(f"decode dtypes act={act} scales={sdt} M={M} G={G} stream={stream} zp={zp}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M * 31 + G)
    sc = torch.from_numpy(p["scales"]).to(sdt)
    xa = torch.from_numpy(p["x"]).to(act)
    qz = torch.from_numpy(p["qzeros"]).to(DEV) if zp else None
    y = ops.gemm(xa.to(DEV), torch.from_numpy(p["qweight"]).to(DEV), sc.to(DEV), qz, G, layout="autoawq",
                 decode_stream=stream is not False, decode_layout=stream or None).float().cpu().numpy()
    w = O.dequant_awq(p["qweight"], sc.float().numpy(), p["qzeros"] if zp else None, G, out_dtype="float32",
                      zero_point=zp)
    ye = xa.double().numpy() @ w.astype(np.float64)
    ulp = 2.0 ** (np.floor(np.log2(np.maximum(np.abs(ye), 1.0))) - (10 if act == torch.float16 else 7))
    err = np.abs(y - ye) / ulp
    assert err.max() <= 1.0, float(err.max())


@pytest.mark.parametrize("M,K,N,G", [(1, 1024, 512, 32), (4, 512, 256, 128), (64, 512, 512, 64),
                                     (48, 1056, 256, 32)])
def test_gemm_symmetric(M, K, N, G):
    ops = _lib()
    _note(f"gemm symmetric M={M} K={K} N={N} G={G}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=13)
    t = _to_dev(p)
    y = ops.gemm(t["x"], t["qweight"], t["scales"], None, G, layout="autoawq").cpu().numpy()
    w = _w_used(p, M, G, zp=False)
    _check_vs_exact(y, O.linear_exact(p["x"], w.T), "symmetric")


def test_gemm_kn_seq_layout():
    ops = _lib()
    M, K, N, G = 3, 512, 512, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=17)
    W = O.unpack_awq(p["qweight"])
    Z = O.unpack_awq(p["qzeros"])
    qw, qz = O.pack_ref(W), O.pack_ref(Z)
    y = ops.gemm(torch.from_numpy(p["x"]).to(DEV), torch.from_numpy(qw).to(DEV),
                 torch.from_numpy(p["scales"]).to(DEV), torch.from_numpy(qz).to(DEV), G,
                 layout="kn_seq").cpu().numpy()
    w = _w_used(p, M, G)
    _check_vs_exact(y, O.linear_exact(p["x"], w.T), "kn_seq")


# ------------------------------------------------------------------ split-K
@pytest.mark.parametrize("M", [1, 8, 32])
def test_split_k_config2_bit_stable(M):
    """Config 2: K=12288, N=4096, split-K in {1, 4, 8}: each split is bitwise
    reproducible across calls, and every split is within the bars of the oracle."""
    ops = _lib()
    K, N, G = 12288, 4096, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=2)
    t = _to_dev(p)
    ye = O.linear_exact(p["x"], _w_used(p, M, G).T)
    qr, zr, sr = O.repack_awq_to_ref(p["qweight"], p["qzeros"], p["scales"])
    yr = R.awq_linear_cpu(torch.from_numpy(p["x"]), torch.from_numpy(qr), torch.from_numpy(sr),
                          torch.from_numpy(zr), G).numpy()
    for sk in (1, 4, 8):
        _note(f"split-K M={M} split={sk} (AutoAWQ layout read directly)")
        y1 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=sk, layout="autoawq", decode_stream=False)
        y2 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=sk, layout="autoawq", decode_stream=False)
        assert torch.equal(y1.view(torch.int16), y2.view(torch.int16)), f"split {sk} not bit-stable"
        _check_vs_exact(y1.cpu().numpy(), ye, f"split {sk}")
        # the reference's own CPU path (dequant + F.linear): max-abs / mean-relative bars
        _check_vs_ref(y1.cpu().numpy(), yr, f"config2 M={M} split {sk} vs reference CPU path")


@pytest.mark.parametrize("M,K,sk", [(1, 4096, 3), (4, 2080, 5), (16, 1024, 200)])
@pytest.mark.parametrize("stream", [True, False])
def test_split_k_uneven_ranges(M, K, sk, stream):
    """split_k follows the reference's ranges (ceil(ceil(K/64)/split_k) blocks of 64 rows each,
    awq_fused_gemm.py:1798-1800): uneven, a K that is not a multiple of 64, and more splits
    than 64-row blocks (the extra ranges are empty).  Bit-stable and within the oracle bar."""
    ops = _lib()
    N, G = 1024, 32
    _note(f"split-K uneven M={M} K={K} split={sk} stream={stream}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=K + sk)
    t = _to_dev(p)
    y1 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=sk, layout="autoawq", decode_stream=stream)
    y2 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=sk, layout="autoawq", decode_stream=stream)
    assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
    _check_vs_exact(y1.cpu().numpy(), O.linear_exact(p["x"], _w_used(p, M, G).T), f"split {sk}")


CONFIG12 = [(m, 4096, n) for m in (1, 4, 16) for n in (4096, 6144, 24576)] + [(m, 12288, 4096) for m in (1, 8, 32)]


@pytest.mark.parametrize("M,K,N", CONFIG12)
def test_forced_split1_matches_auto(M, K, N):
    """A forced ``split_k = 1`` (the whole K per block) runs the kernel "auto" runs wherever
    auto does not split K, so the two are bitwise equal there: every config-1 shape but
    M = 16, N = 6144, and config 2 at M = 1.  Where auto splits, split 1 takes the narrow
    kernel (N / 16 whole-K blocks): bit-stable and within 1 ulp of the exact oracle."""
    ops = _lib()
    G = 128
    auto_whole_k = ops._narrow_fits(M, N, K, 0) or ops._auto_splits(M, N, K) == 1
    _note(f"split 1 vs auto M={M} K={K} N={N} auto_whole_k={auto_whole_k}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M * 7 + N)
    t = _to_dev(p)
    ya = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=0, layout="autoawq")
    y1 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=1, layout="autoawq")
    y1b = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=1, layout="autoawq")
    assert torch.equal(y1.view(torch.int16), y1b.view(torch.int16)), "split 1 not bit-stable"
    if auto_whole_k:
        assert torch.equal(y1.view(torch.int16), ya.view(torch.int16)), "split 1 differs from auto"
    _check_vs_exact(y1.cpu().numpy(), O.linear_exact(p["x"], _w_used(p, M, G).T), f"split 1 M={M} N={N}")


# ------------------------------------------------------------------ benchmark configs
@pytest.mark.parametrize("M,N", [(m, n) for m in (1, 4, 16) for n in (4096, 6144, 24576)])
@pytest.mark.parametrize("stream", [None, False])
def test_config1_decode_sweep(M, N, stream):
    ops = _lib()
    _note(f"config1 M={M} N={N} stream={stream}")
    K, G = 4096, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=1)
    t = _to_dev(p)
    y = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq",
                 decode_stream=stream).cpu().numpy()
    w = _w_used(p, M, G)
    _check_vs_exact(y, O.linear_exact(p["x"], w.T), f"config1 M={M} N={N}")
    qr, zr, sr = O.repack_awq_to_ref(p["qweight"], p["qzeros"], p["scales"])
    yr = R.awq_linear_cpu(torch.from_numpy(p["x"]), torch.from_numpy(qr), torch.from_numpy(sr),
                          torch.from_numpy(zr), G).numpy()
    _check_vs_ref(y, yr, f"config1 M={M} N={N}")


@pytest.mark.parametrize("M,N", [(512, 12288), (512, 24576), (2048, 12288), (2048, 24576)])
def test_config3_prefill(M, N):
    """Full-size prefill: every output against a torch fp32 GEMM on the (bit-exact
    checked) dequantized weight, from both prefill kernels (the stream copy's, which serves
    these shapes, and the AutoAWQ tensor's); 128 sampled rows against the exact oracle."""
    ops = _lib()
    _note(f"config3 M={M} N={N}")
    K, G = 4096, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=3, outliers=True)
    t = _to_dev(p)
    y = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq")
    y_kn = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq", decode_stream=False)
    wd = ops.dequant(t["qweight"], t["scales"], t["qzeros"], G, layout="autoawq")     # [K, N]
    w = O.dequant_awq(p["qweight"], p["scales"], p["qzeros"], G)
    assert np.array_equal(wd.cpu().numpy().view(np.uint16), w.view(np.uint16))
    y32 = (t["x"].float() @ wd.float())
    ulp = torch.exp2(torch.floor(torch.log2(y32.abs().clamp_min(1.0))) - 10)
    for yy, what in ((y, "stream copy"), (y_kn, "AutoAWQ tensor")):
        d = (yy.float() - y32).abs()
        assert bool((d <= 1.0 * ulp + 1e-3 * y32.abs().clamp_min(1.0) * 2 ** -10).all()), (what, float((d / ulp).max()))
    rows = np.random.default_rng(0).choice(M, size=128, replace=False)
    ye = O.linear_exact(p["x"][rows], w.T)
    _check_vs_exact(y.cpu().numpy()[rows], ye, f"config3 M={M} N={N}")
    # 8 sampled rows against the reference's own CPU path (dequant + F.linear in fp16)
    r8 = rows[:8]
    qr, zr, sr = O.repack_awq_to_ref(p["qweight"], p["qzeros"], p["scales"])
    yr = R.awq_linear_cpu(torch.from_numpy(p["x"][r8]), torch.from_numpy(qr), torch.from_numpy(sr),
                          torch.from_numpy(zr), G).numpy()
    _check_vs_ref(y.cpu().numpy()[r8], yr, f"config3 M={M} N={N} vs reference CPU path")


# ------------------------------------------------------------------ decode stream layout
def _stream_layout_numpy(qw_kn):
    """The decode stream layout restated with numpy gathers: in the (tile t, k-step s) run, lane
    l = 16q + r owns word 16 t + r (zero past the last word) of rows 32 s + 8 q + j; its u32
    number v < 4 is lo16(row 2v) | lo16(row 2v+1) << 16 and number 4 + v the same of the high
    halves, stored at byte 1024 (n // 4) + 16 l + 4 (n % 4); runs tile-major."""
    K, NW = qw_kn.shape
    tiles = -(-NW // 16)
    pad = np.zeros((K, tiles * 16), dtype=np.uint32)
    pad[:, :NW] = qw_kn.view(np.uint32)
    v = pad.reshape(K // 32, 4, 4, 2, tiles, 16)            # [s, q, v, row parity, t, r]
    lo, hi = v & 0xFFFF, v >> 16
    plo = lo[:, :, :, 0] | (lo[:, :, :, 1] << 16)           # [s, q, v, t, r]
    phi = hi[:, :, :, 0] | (hi[:, :, :, 1] << 16)
    n = np.stack([plo, phi], axis=2)                         # [s, q, e, v, t, r]
    lane = n.transpose(4, 0, 2, 1, 5, 3)                     # [t, s, e, q, r, v]
    return np.ascontiguousarray(lane).reshape(-1).view(np.int32)


def _narrow_layout_numpy(qw):
    """Narrow decode layout: (tile t, quad c, lane 16 q + r, i) -> u32 holding column 16 t + r
    at rows 32 s + 8 q + j of k-step s = 4 c + i (zero past K), row j at bit 16 (j % 2) + 4 (j // 2)."""
    K, NW = qw.shape
    N = NW * 8
    tiles, KS = -(-N // 16), K // 32
    KQ = -(-KS // 4)
    pad = np.zeros((KQ * 128, tiles * 16), dtype=np.uint32)
    pad[:K, :N] = O.unpack_awq(qw)
    v = pad.reshape(KQ, 4, 4, 8, tiles, 16)                  # [c, i, q, j, t, r]
    out = np.zeros((tiles, KQ, 4, 16, 4), dtype=np.uint32)   # [t, c, q, r, i]
    for j in range(8):
        out |= v[:, :, :, j].transpose(3, 0, 2, 4, 1) << np.uint32((j & 1) * 16 + (j >> 1) * 4)
    return out.reshape(-1).view(np.int32)


@pytest.mark.parametrize("K,N", [(256, 4096), (128, 1000), (64, 520), (32, 8), (96, 24), (2816, 48)])
def test_pack_decode_narrow_layout(K, N):
    ops = _lib()
    rng = np.random.default_rng(K * 3 + N)
    qw = rng.integers(-2**31, 2**31 - 1, size=(K, N // 8), dtype=np.int64).astype(np.int32)
    got = ops.pack_decode_narrow(torch.from_numpy(qw).to(DEV)).cpu().numpy()
    assert np.array_equal(got, _narrow_layout_numpy(qw))


@pytest.mark.parametrize("M,K,N,G", [(1, 4096, 4096, 128), (1, 2048, 1000, 32), (4, 4096, 6144, 128),
                                     (16, 1024, 520, 64), (17, 2048, 1536, 128), (32, 512, 264, 32),
                                     (1, 14336, 4096, 128), (9, 96, 2056, 32)])
@pytest.mark.parametrize("zp", [True, False])
def test_gemm_decode_narrow_vs_oracle(M, K, N, G, zp):
    """The narrow layout (whole K per 16-column block): within 1 ulp of the exact oracle with
    unrounded weights, bias included, and bitwise stable across calls."""
    ops = _lib()
    _note(f"decode narrow M={M} K={K} N={N} G={G} zp={zp}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + 3 * N + K)
    t = _to_dev(p)
    qz = t["qzeros"] if zp else None
    b = torch.from_numpy(np.random.default_rng(M).standard_normal(N).astype(np.float32)).half()
    y = ops.gemm(t["x"], t["qweight"], t["scales"], qz, G, bias=b.to(DEV), layout="autoawq",
                 decode_stream=True, decode_layout="narrow")
    y2 = ops.gemm(t["x"], t["qweight"], t["scales"], qz, G, bias=b.to(DEV), layout="autoawq",
                  decode_stream=True, decode_layout="narrow")
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    w = _w_used(p, M, G, zp=zp)
    _check_vs_exact(y.cpu().numpy(), O.linear_exact(p["x"], w.T, b.double().numpy()), f"narrow M={M} N={N}")


@pytest.mark.parametrize("K,N", [(256, 4096), (128, 1000), (64, 520)])
def test_pack_decode_stream_layout(K, N):
    ops = _lib()
    rng = np.random.default_rng(K + N)
    qw = rng.integers(-2**31, 2**31 - 1, size=(K, N // 8), dtype=np.int64).astype(np.int32)
    got = ops.pack_decode_stream(torch.from_numpy(qw).to(DEV)).cpu().numpy()
    assert np.array_equal(got, _stream_layout_numpy(qw))


@pytest.mark.parametrize("M,K,N,G", [(1, 2048, 5632, 128), (4, 4096, 6144, 128), (16, 1024, 1000, 64),
                                     (3, 512, 520, 32), (32, 2048, 1536, 128), (24, 1024, 4096, 128)])
@pytest.mark.parametrize("zp", [True, False])
def test_gemm_decode_stream_vs_oracle(M, K, N, G, zp):
    """Decode-shaped calls through the stream copy: within 1 ulp of the exact oracle, and
    identical to an explicit stream call (cache hit path)."""
    ops = _lib()
    _note(f"decode stream M={M} K={K} N={N} G={G} zp={zp}")
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=M + N + K)
    t = _to_dev(p)
    qz = t["qzeros"] if zp else None
    y = ops.gemm(t["x"], t["qweight"], t["scales"], qz, G, layout="autoawq", decode_stream=True)
    y2 = ops.gemm(t["x"], t["qweight"], t["scales"], qz, G, layout="autoawq")
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
    w = _w_used(p, M, G, zp=zp)
    _check_vs_exact(y.cpu().numpy(), O.linear_exact(p["x"], w.T), f"stream M={M} N={N}")


@pytest.mark.parametrize("M", [1, 16, 32])
def test_decode_stream_split_k_bit_stable(M):
    ops = _lib()
    K, N, G = 12288, 4096, 128
    p = make_awq_problem(M=M, K=K, N=N, group_size=G, seed=21)
    t = _to_dev(p)
    ye = O.linear_exact(p["x"], _w_used(p, M, G).T)
    for sk in (1, 4, 8):
        _note(f"stream split-K M={M} split={sk}")
        y1 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=sk, layout="autoawq", decode_stream=True)
        y2 = ops.gemm(t["x"], t["qweight"], t["scales"], t["qzeros"], G, split_k=sk, layout="autoawq", decode_stream=True)
        assert torch.equal(y1.view(torch.int16), y2.view(torch.int16))
        _check_vs_exact(y1.cpu().numpy(), ye, f"stream split {sk}")
