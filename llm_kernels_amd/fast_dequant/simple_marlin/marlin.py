"""W4A16 GEMM entry point `mul` (reference fast_dequant/simple_marlin/test.py:25 ->
marlin_w4a16_gemm.cpp:23-111).  Same argument list and error behaviour (RuntimeError)."""
try:
    from ... import _lib
except ImportError:  # this directory itself is on sys.path (the reference's top-level module layout)
    import _lib


def mul(A, B, C, s, workspace, thread_k=-1, thread_n=-1, sms=-1, max_par=16):
    """C[M,N] (fp16, written in place) = A[M,K] (fp16) x dequant(B, s).

    B is the int32 [K/16, 2N] tensor and s the permuted fp16 [K/g, N] tensor from QuantUtils.pack;
    groupsize is inferred as K / s.size(0).  `workspace`, `thread_k`, `thread_n`, `sms` and `max_par`
    are accepted and ignored, as in the reference.
    """
    return _lib.host.marlin_mul(A, B, C, s)
