"""GPU: the matrix-core kernels for few rows of activations (short prompts through rfq_gemm_f16 and
rfq_gemm_f16_arranged) at the edges of their tiles: rows per operand (16), rows
per slice (128), weight rows per workgroup (16 and 32), 128-element units of k and their remainders, more and fewer units
than wavefronts; against the float64 contraction of the decoded weights."""
import numpy as np
import pytest

from helpers import assert_close
from rocmforge_amd import quantize as Q

pytestmark = pytest.mark.gpu

FORMATS = [Q.Q4_0, Q.Q8_0, Q.Q4_K, Q.Q6_K, Q.GGUF_Q4_0, Q.GGUF_Q8_0, Q.GGUF_Q4_K, Q.GGUF_Q6_K]
SHORT_BLOCKS = [Q.Q4_0, Q.Q8_0, Q.GGUF_Q4_0, Q.GGUF_Q8_0]

# Both operands are exact (integer codes; activations as given, float32 ones to 2^-22) and the sums are float32: a sum of k
# products of random sign is about sqrt(k) * 2^-24 of their typical size off, 4e-6 at k = 4096; max over the outputs.
TOL = 2e-5


def weights_of(oracle, fmt, w, n, k):
    return oracle.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64)


def shape_of(fmt, n, k):
    return n, k if fmt in SHORT_BLOCKS else (k + 255) // 256 * 256


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(1, 16, 256), (9, 17, 96), (16, 31, 288), (17, 640, 1056), (32, 33, 1024), (48, 8200, 512), (49, 64, 2080),
                                   (65, 100, 768), (96, 130, 1024), (128, 48, 992), (129, 5001, 1024), (160, 200, 1536)])
def test_prompts(fmt, m, n, k, oracle, cuda):
    import torch
    from rocmforge_amd import ops
    n, k = shape_of(fmt, n, k)
    w = Q.make_weights(fmt, n, k, seed=fmt + m)
    a = np.random.default_rng(m * n).standard_normal((m, k)).astype(np.float16)
    dw, da = torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda)
    want = a.astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T
    plain = ops.gemm_f16(fmt, dw, da, n, k, out_dtype=torch.float32)
    arranged = ops.gemm_f16_arranged(fmt, dw, ops.ArrangedA(da), n, out_dtype=torch.float32)
    for got, what in ((plain, "rows"), (arranged, "arranged")):
        assert_close(got.cpu().numpy(), want, f"{Q.NAMES[fmt]} {m}x{n}x{k} {what}", tol=TOL, plain_tol=2e-4)
    f16 = ops.gemm_f16(fmt, dw, da, n, k)
    assert torch.equal(f16, plain.half())
