"""Which weights a GEMM call multiplies, as the library dispatches it (``gemm_route`` in
``litevllm_amd/csrc/awq_capi.hip``): up to 64 rows the unrounded (q - z) * s (the decode kernels and the
middle-batch kernel's unrounded form), above the weights rounded once to the activation dtype (the
middle-batch kernel's rounded form and the prefill kernels), so a test's exact reference takes the matching
weights."""


def decode_serves(M: int, N: int, G: int) -> bool:
    """Whether the weights enter unrounded: up to 64 rows in groups of 32, 64 and 128 (N does not enter
    the rule)."""
    return int(G) in (32, 64, 128) and M <= 64
