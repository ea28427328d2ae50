"""GPU: the matrix-core kernels for few rows of activations (short prompts through rfq_gemm_f16 and
rfq_gemm_f16_arranged, decode batches of 2 to 8 through rfq_gemv) at the edges of their tiles: rows per operand (16), weight
rows per workgroup (16 and 32), 128-element units of k and their remainders, more and fewer units than wavefronts; against the float64 contraction of the decoded weights."""
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


BATCH_FORMATS = FORMATS + [Q.MXFP4, Q.MXFP6_E2M3]


@pytest.mark.parametrize("fmt", BATCH_FORMATS)
@pytest.mark.parametrize("m,n,k", [(2, 4200, 544), (3, 1029, 1024), (4, 3100, 3072), (5, 15, 256), (5, 17, 32), (6, 33, 96), (7, 5201, 480), (8, 64, 4128),
                                   (8, 13400, 768), (5, 200, 13824)])
def test_decode_batches(fmt, m, n, k, oracle, cuda):
    import torch
    from rocmforge_amd import ops
    if fmt in FORMATS:
        n, k = shape_of(fmt, n, k)
    w = Q.make_weights(fmt, n, k, seed=fmt + m)
    x = np.random.default_rng(m * n).standard_normal((m, k)).astype(np.float32)
    got = ops.gemv(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), n, k)
    want = x.astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T
    assert_close(got.cpu().numpy(), want, f"{Q.NAMES[fmt]} {m}x{n}x{k}", tol=TOL, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.GGUF_Q4_K, Q.Q6_K, Q.MXFP4])
def test_decode_batch_of_any_magnitude(fmt, oracle, cuda):
    """The fp16 parts of x follow its magnitude: vectors of very different size, sizes that grow and shrink by powers of
    ten along k, zeros, subnormals; an infinity or a NaN changes its own vector's outputs and no other's: to NaN, or, for
    the formats and shapes that other batches multiply in float32 (here Q6_K and MXFP4), an infinity to the infinity of its
    product with the weight."""
    import torch
    from rocmforge_amd import ops
    m, n, k = 8, 48, 2048
    w = Q.make_weights(fmt, n, k, seed=5)
    rng = np.random.default_rng(6)
    x = rng.standard_normal((m, k))
    x[0] *= 1e30
    x[1] *= 1e-30
    x[2] *= 10.0 ** np.linspace(-8, 8, k)
    x[3] *= 10.0 ** np.linspace(8, -8, k)
    x[4, : k // 2] = 0
    x[5] = 0
    x[6] *= 1e-41
    x = x.astype(np.float32)
    dw = torch.from_numpy(w).to(cuda)
    got = ops.gemv(fmt, dw, torch.from_numpy(x).to(cuda), n, k).cpu().numpy().astype(np.float64)
    w64 = weights_of(oracle, fmt, w, n, k)
    want = x.astype(np.float64) @ w64.T
    for v in (0, 1, 2, 3, 4, 5, 7):
        assert_close(got[v], want[v], f"{Q.NAMES[fmt]} vector {v}", tol=TOL, plain_tol=2e-4)
    # (subnormal x: 2^-149 steps in the products' own sums)
    assert np.all(np.abs(got[6] - want[6]) <= 2e-5 * np.abs(want[6]).max() + 64 * 2.0 ** -149)
    for bad in (np.inf, -np.inf, np.nan):
        y = x.copy()
        y[2, 700] = bad
        again = ops.gemv(fmt, dw, torch.from_numpy(y).to(cuda), n, k).cpu().numpy().astype(np.float64)
        with np.errstate(invalid="ignore"):
            product = w64[:, 700] * bad if fmt in (Q.Q6_K, Q.MXFP4) else np.full(n, np.nan)
        assert np.array_equal(again[2], product, equal_nan=True)
        keep = [0, 1, 3, 4, 5, 6, 7]
        assert np.array_equal(again[keep], got[keep])


@pytest.mark.parametrize("fmt", [Q.MXFP4, Q.MXFP6_E2M3])
def test_mx_exponents_beyond_the_clamp(fmt, oracle, cuda):
    """Blocks whose exponent byte is 1..127 (the reference clamps value * 2^e) beside -128 and ordinary ones."""
    import torch
    from rocmforge_amd import ops
    m, n, k = 8, 64, 1024
    w = Q.make_weights(fmt, n, k, seed=9).copy()
    blocks = w.reshape(-1, Q.BLOCK_BYTES[fmt])
    rng = np.random.default_rng(10)
    blocks[:, 0] = rng.choice(np.array([-128, -3, -1, 0, 1, 2, 3, 4, 5, 6, 127], np.int8), blocks.shape[0]).view(np.uint8)
    blocks[:, 1:] = rng.integers(0, 256, blocks[:, 1:].shape, dtype=np.uint8)
    x = rng.standard_normal((m, k)).astype(np.float32)
    got = ops.gemv(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), n, k)
    want = x.astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T
    assert_close(got.cpu().numpy(), want, Q.NAMES[fmt], tol=TOL, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", BATCH_FORMATS)
@pytest.mark.parametrize("m,n,k", [(2, 40, 256), (4, 1025, 768), (5, 16, 1280), (8, 5377, 1024)])
def test_norm_taken_along(fmt, m, n, k, oracle, cuda):
    import torch
    from rocmforge_amd import ops
    w = Q.make_weights(fmt, n, k, seed=fmt + m)
    rng = np.random.default_rng(m * n)
    x, nw = rng.standard_normal((m, k)).astype(np.float32) * 3, (1 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    got = ops.rms_norm_gemv(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), torch.from_numpy(nw).to(cuda), 1e-5, n, k)
    x64 = x.astype(np.float64)
    xn = x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-5) * nw
    assert_close(got.cpu().numpy(), xn @ weights_of(oracle, fmt, w, n, k).T, f"{Q.NAMES[fmt]} {m}x{n}x{k}", tol=TOL, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", BATCH_FORMATS)
@pytest.mark.parametrize("m,hidden,inter,norm", [(2, 256, 512, True), (3, 768, 1792, False), (3, 256, 6912, True), (5, 512, 6912, True), (8, 768, 2304, True)])
def test_gate_and_up_in_one_launch(fmt, m, hidden, inter, norm, oracle, cuda):
    import torch
    from rocmforge_amd import ops
    gate, up = Q.make_weights(fmt, inter, hidden, seed=fmt), Q.make_weights(fmt, inter, hidden, seed=fmt + 1)
    down = Q.make_weights(Q.Q8_0, hidden, inter, seed=3)
    rng = np.random.default_rng(m)
    x, nw = rng.standard_normal((m, hidden)).astype(np.float32), (1 + 0.1 * rng.standard_normal(hidden)).astype(np.float32)
    dev = [torch.from_numpy(t).to(cuda) for t in (gate, up, down, x, nw)]
    got = ops.mlp_swiglu(fmt, dev[0], dev[1], Q.Q8_0, dev[2], dev[3], dev[4] if norm else None, 1e-5, hidden, inter)
    xn = x.astype(np.float64)
    if norm:
        xn = xn / np.sqrt((xn * xn).mean(axis=1, keepdims=True) + 1e-5) * nw
    g, u = (xn @ weights_of(oracle, fmt, t, inter, hidden).T for t in (gate, up))
    h = g * (u / (1 + np.exp(-u)))
    want = h @ weights_of(oracle, Q.Q8_0, down, hidden, inter).T
    # (the product of two float32 sums, contracted once more: the errors of both add up)
    assert_close(got.cpu().numpy(), want, f"{Q.NAMES[fmt]} {m}x{hidden}x{inter}", tol=3 * TOL, plain_tol=6e-4)


@pytest.mark.parametrize("fmt", BATCH_FORMATS)
@pytest.mark.parametrize("m,n,k", [(4, 4000, 3072), (5, 96, 13824), (8, 256, 4096), (8, 96, 1024)])
@pytest.mark.parametrize("outlier", [False, True])
def test_decode_batches_keep_float32_precision(fmt, m, n, k, outlier, oracle, cuda):
    """The 2-norm of the error: two fp16 parts keep 23 bits of x (errors of 2^-23 in a quarter of the values: 4e-8 rms), a
    unit's sum of up to eight products rounds to 24 bits eight times (2.5e-8 rms each, partial sums growing like sqrt: 5e-8),
    the matrix instruction as often again; together below 1e-7, and what a float32 kernel reaches is 1.1e-7 to 1.3e-7.  It
    holds beside a value 2^14 times the others whose weights are zero, in the same unit and in those that follow."""
    import torch
    from rocmforge_amd import ops
    w = Q.make_weights(fmt, n, k, seed=fmt + m).copy()
    x = np.random.default_rng(m * n).standard_normal((m, k)).astype(np.float32)
    if outlier:
        w.reshape(n, -1)[:, : Q.BLOCK_BYTES[fmt]] = 0              # (a block of zero bytes decodes to zeros in every layout)
        x[:, 5] = 2.0 ** 14
    got = ops.gemv(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), n, k).cpu().numpy().astype(np.float64)
    want = x.astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T
    error = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert np.linalg.norm(error) / np.sqrt(m) <= 1.3e-7, (Q.NAMES[fmt], error)


@pytest.mark.parametrize("first", [120.5, 121.5, 122.5, 123.5, 126.5])
def test_decode_batch_up_to_the_largest_value(first, oracle, cuda):
    """The largest finite float after smaller ones of 2^first in the same wavefront's earlier unit (eight wavefronts take the
    128-element units in turn)."""
    import torch
    from rocmforge_amd import ops
    m, n, k = 5, 32, 2048
    w = Q.make_weights(Q.Q4_0, n, k, seed=3).copy()
    blocks = w.reshape(-1, 20)
    blocks[:, :4] = np.frombuffer(np.float32(1e-4).tobytes(), np.uint8)
    x = np.random.default_rng(1).standard_normal((m, k)).astype(np.float32)
    x[:, 3] = 2.0 ** first
    x[:, 1024 + 9] = np.finfo(np.float32).max
    got = ops.gemv(Q.Q4_0, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), n, k).cpu().numpy()
    want = x.astype(np.float64) @ weights_of(oracle, Q.Q4_0, w, n, k).T
    assert np.all(np.abs(got - want) <= 1e-6 * np.abs(want) + 1e-7 * np.abs(want).max())


@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.Q8_0])
@pytest.mark.parametrize("scale", [1e-37, 1e31, 1e33, 1e36])
def test_decode_batch_with_scales_of_any_size(fmt, scale, oracle, cuda):
    """The block scales of a 128-element unit near both ends of float32 against x that takes the results back to ordinary
    sizes, beside ordinary units of the same row."""
    import torch
    from rocmforge_amd import ops
    m, n, k = 6, 40, 1024
    w = Q.make_weights(fmt, n, k, seed=8).copy()
    blocks = w.reshape(n, k // 32, -1)
    blocks[:, 4:8, :4] = np.frombuffer(np.float32(scale).tobytes(), np.uint8)
    x = np.random.default_rng(2).standard_normal((m, k)).astype(np.float32)
    x[:, 4 * 32 : 8 * 32] /= np.float32(scale)
    got = ops.gemv(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), n, k).cpu().numpy()
    want = x.astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T
    assert_close(got, want, f"{Q.NAMES[fmt]} scale {scale}", tol=TOL, plain_tol=2e-4)
    x[2, 5 * 32 + 3] = 3e38                                        # (that vector's results lie beyond float32 or are large; the rest of its unit is lost beside it)
    again = ops.gemv(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(x).to(cuda), n, k).cpu().numpy()
    assert np.array_equal(np.delete(again, 2, 0), np.delete(got, 2, 0))
    with np.errstate(over="ignore"):
        large = (x[2].astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T).astype(np.float32)
    assert not np.isnan(again[2]).any() and np.array_equal(np.isinf(again[2]), np.isinf(large))
    assert np.array_equal(np.sign(again[2][np.isinf(large)]), np.sign(large[np.isinf(large)]))


@pytest.mark.parametrize("fmt,n,k,kept", [(Q.MXFP6_E2M3, 8400, 1024, True), (Q.MXFP6_E2M3, 40, 4096, True), (Q.Q6_K, 4096, 4096, True),
                                          (Q.Q6_K, 64, 9216, True), (Q.Q6_K, 1024, 9216, False), (Q.MXFP4, 1024, 9216, False),
                                          (Q.MXFP4, 64, 544, True), (Q.Q4_K, 256, 1024, True), (Q.Q4_K, 256, 1280, False), (Q.Q8_0, 256, 1024, False)])
@pytest.mark.parametrize("m", [5, 8])
def test_an_infinity_in_a_decode_batch(fmt, n, k, kept, m, oracle, cuda):
    """kept: the product of an infinity and a weight that is not zero stays an infinity (one of zero is NaN; Q4_K multiplies
    code and min apart, either of which may be zero, and adds the two); else all of that vector's results are NaN."""
    import torch
    from rocmforge_amd import ops
    w = Q.make_weights(fmt, n, k, seed=4)
    w64 = weights_of(oracle, fmt, w, n, k)
    x = np.random.default_rng(5).standard_normal((m, k)).astype(np.float32)
    dw = torch.from_numpy(w).to(cuda)
    got = ops.gemv(fmt, dw, torch.from_numpy(x).to(cuda), n, k).cpu().numpy()
    for at, bad in ((3, np.inf), (k - 1, -np.inf)):
        y = x.copy()
        y[m - 2, at] = bad
        again = ops.gemv(fmt, dw, torch.from_numpy(y).to(cuda), n, k).cpu().numpy()
        assert np.array_equal(np.delete(again, m - 2, 0), np.delete(got, m - 2, 0))
        with np.errstate(invalid="ignore"):
            product = w64[:, at] * bad
        if not kept:
            assert np.isnan(again[m - 2]).all()
        elif fmt != Q.Q4_K:
            assert np.array_equal(again[m - 2], product.astype(np.float32), equal_nan=True)
        else:
            inf = np.isinf(again[m - 2])
            assert inf.any() and np.array_equal(again[m - 2][inf], product[inf].astype(np.float32)) and np.isnan(again[m - 2][~inf]).all()


@pytest.mark.parametrize("fmt", [Q.Q8_0, Q.Q4_K, Q.MXFP6_E2M3])
@pytest.mark.parametrize("m", [3, 8])
def test_norm_of_vectors_whose_squares_overflow(fmt, m, oracle, cuda):
    """Finite x whose float32 sum of squares is infinite is zero after the norm (x / infinity), and so are its results, alone
    and as gate and up projection; with an infinity or a NaN in x the vector's results are NaN; the others keep theirs."""
    import torch
    from rocmforge_amd import ops
    n, k = 512, 1024
    w, up = Q.make_weights(fmt, n, k, seed=1), Q.make_weights(fmt, n, k, seed=2)
    down = Q.make_weights(Q.Q8_0, k, n, seed=3)
    x = np.random.default_rng(3).standard_normal((m, k)).astype(np.float32)
    dev = [torch.from_numpy(t).to(cuda) for t in (w, up, down, np.ones(k, np.float32))]

    def both(x):
        dx = torch.from_numpy(x).to(cuda)
        return (ops.rms_norm_gemv(fmt, dev[0], dx, dev[3], 1e-5, n, k).cpu().numpy(),
                ops.mlp_swiglu(fmt, dev[0], dev[1], Q.Q8_0, dev[2], dx, dev[3], 1e-5, k, n).cpu().numpy())
    ordinary = both(x)
    y = x.copy()
    y[1] *= np.float32(3e37)
    for got, before in zip(both(y), ordinary):
        assert np.all(got[1] == 0) and np.array_equal(np.delete(got, 1, 0), np.delete(before, 1, 0))
    for bad in (np.inf, -np.inf, np.nan):
        y[1, 700] = bad
        for got, before in zip(both(y), ordinary):
            assert np.isnan(got[1]).all() and np.array_equal(np.delete(got, 1, 0), np.delete(before, 1, 0))


@pytest.mark.parametrize("fmt", SHORT_BLOCKS)
@pytest.mark.parametrize("k", [800, 832, 864, 896])
@pytest.mark.parametrize("m,n", [(7, 72), (40, 9000)])
def test_an_infinity_in_the_last_group_of_a_prompt_row(fmt, k, m, n, oracle, cuda):
    """Rows that end inside a 128-element unit: what the kernel reads again to fill the unit is not multiplied, so that an
    infinity among it does not become NaN: every output is the infinity's product with its weight."""
    import torch
    from rocmforge_amd import ops
    w = Q.make_weights(fmt, n, k, seed=6)
    a = np.random.default_rng(7).standard_normal((m, k)).astype(np.float16)
    a[m // 2, k - 2] = -np.inf
    dw, da = torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda)
    with np.errstate(invalid="ignore"):
        product = (weights_of(oracle, fmt, w, n, k)[:, k - 2] * -np.inf).astype(np.float32)
    plain = ops.gemm_f16(fmt, dw, da, n, k, out_dtype=torch.float32).cpu().numpy()
    arranged = ops.gemm_f16_arranged(fmt, dw, ops.ArrangedA(da), n, out_dtype=torch.float32).cpu().numpy()
    for got in (plain, arranged):
        assert np.array_equal(got[m // 2], product, equal_nan=True)
        assert np.isfinite(np.delete(got, m // 2, 0)).all()


@pytest.mark.parametrize("m", [2, 5, 8])
def test_norm_and_projection_over_their_own_input(m, cuda):
    """rfq_rms_norm_gemv with the result written over x, and with x as its own scratch (then x holds the normalised rows):
    the calls whose norm has to be a step of its own."""
    import ctypes as C
    import torch
    from rocmforge_amd import _lib, ops
    n = k = 1024
    p = lambda t: C.c_void_p(t.data_ptr())
    w = torch.from_numpy(Q.make_weights(Q.Q8_0, n, k, seed=1)).to(cuda)
    gen = torch.Generator(device="cpu").manual_seed(2)
    x, nw = torch.randn((m, k), generator=gen).to(cuda), torch.randn(k, generator=gen).to(cuda)
    want = ops.rms_norm_gemv(Q.Q8_0, w, x, nw, 1e-5, n, k).cpu().numpy()
    xn = ops.rms_norm(x, nw, 1e-5)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for y, scratch in (("x", "own"), ("own", "x")):
        into = x.clone()
        own = torch.zeros((m, k), device=cuda)
        _lib.check(_lib.lib().rfq_rms_norm_gemv(Q.Q8_0, p(w), w.numel(), p(into), p(nw), 1e-5, p(into if y == "x" else own), m, n, k,
                                                p(into if scratch == "x" else own), stream))
        assert_close((into if y == "x" else own).cpu().numpy(), want, f"result over {y}, scratch {scratch}", tol=TOL, plain_tol=2e-4)
        if scratch == "x":
            assert torch.equal(into, xn)


@pytest.mark.parametrize("m,k,dtype", [(9, 1024, "f16"), (100, 1024, "f16"), (40, 2048, "f32")])
def test_prompt_over_its_own_activations(m, k, dtype, cuda):
    """The output in the activations' memory (n * size of an output = k * 2): read whole before it is written."""
    import ctypes as C
    import torch
    from rocmforge_amd import _lib, ops
    n = k if dtype == "f16" else k // 2
    out_dtype = torch.float16 if dtype == "f16" else torch.float32
    p = lambda t: C.c_void_p(t.data_ptr())
    w = torch.from_numpy(Q.make_weights(Q.GGUF_Q4_K, n, k, seed=1)).to(cuda)
    a = torch.randn((m, k), generator=torch.Generator(device="cpu").manual_seed(2)).to(cuda).half()
    want = ops.gemm_f16(Q.GGUF_Q4_K, w, a, n, k, out_dtype=out_dtype).float().cpu().numpy()
    into = a.clone()
    _lib.check(_lib.lib().rfq_gemm_f16(Q.GGUF_Q4_K, p(w), w.numel(), p(into), p(into), _lib.F16 if dtype == "f16" else _lib.F32, m, n, k,
                                       C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    got = into.view(out_dtype)[:, :n].float().cpu().numpy()
    assert_close(got, want, f"{m}x{n}x{k} {dtype}", tol=2e-5 if dtype == "f32" else 2.0 ** -10, plain_tol=None)


@pytest.mark.parametrize("fmt", BATCH_FORMATS)
@pytest.mark.parametrize("m,n,k", [(3, 3100, 3072), (6, 130, 1056), (8, 40, 13824)])
def test_decode_batches_at_any_address(fmt, m, n, k, oracle, cuda):
    """x on a 4-byte boundary and, where the blocks are whole dwords, weights at any byte: the same kernel and the same bits
    as on a 16-byte boundary; elsewhere other kernels take the unaligned weights."""
    import torch
    from rocmforge_amd import _lib, ops
    if fmt in FORMATS:
        n, k = shape_of(fmt, n, k)
    w = torch.from_numpy(Q.make_weights(fmt, n, k, seed=fmt)).to(cuda)
    x = torch.randn((m, k), generator=torch.Generator(device="cpu").manual_seed(m)).to(cuda)
    kernel = lambda: _lib.lib().rfq_bench_last_gemv_kernel().decode()
    want = ops.gemv(fmt, w, x, n, k)
    assert kernel().startswith("gemv_skinny_kernel")
    space = torch.empty(m * k + 4, device=cuda)
    for off in (1, 2, 3):
        moved = space[off : off + m * k].view(m, k)
        moved.copy_(x)
        assert moved.data_ptr() % 16 == 4 * off
        assert torch.equal(ops.gemv(fmt, w, moved, n, k), want) and kernel().startswith("gemv_skinny_kernel")
    space = torch.empty(w.numel() + 4, dtype=torch.uint8, device=cuda)
    windows = fmt in (Q.GGUF_Q4_0, Q.GGUF_Q8_0, Q.GGUF_Q6_K, Q.MXFP4, Q.MXFP6_E2M3)
    for off in (2,) if windows else (1, 2, 3):
        moved = space[off : off + w.numel()]
        moved.copy_(w)
        got = ops.gemv(fmt, moved, x, n, k)
        assert kernel().startswith("gemv_skinny_kernel") != windows
        assert_close(got.cpu().numpy(), want.cpu().numpy(), f"{Q.NAMES[fmt]} weights off by {off}", tol=TOL, plain_tol=2e-4)
        assert windows or torch.equal(got, want)


def kernel_name():
    from rocmforge_amd import _lib
    return _lib.lib().rfq_bench_last_gemv_kernel().decode()


@pytest.mark.parametrize("fmt", FORMATS)
def test_every_prompt_kernel(fmt, oracle, cuda):
    """Every form of the fp16 kernel that the dispatch can pick (16-row operands, row tiles of W; rows or arranged), at
    ragged sizes: that it is the one taken, its results, and that both orders of the activations give the same bits."""
    import torch
    from rocmforge_amd import ops
    most = 4 if fmt in (Q.Q4_0, Q.GGUF_Q4_0) else 8
    forms = [((1, 1), 13, 1003), ((2, 1), 24, 4001), ((3, 1), 37, 4090), ((4, 1), 61, 4001), ((6, 1), 90, 4090), ((6, 1), 75, 4001),
             ((1, 2), 12, 9001), ((2, 2), 24, 9001), ((3, 2), 41, 8999), ((4, 2), 60, 9001), ((4, 2) if most == 4 else (6, 2), 105 if most == 4 else 90, 8200),
             ((4, 2) if most == 4 else (8, 2), 121, 8200)]
    k = 544 if fmt in SHORT_BLOCKS else 512
    w = Q.make_weights(fmt, 9001, k, seed=fmt)
    dw = torch.from_numpy(w).to(cuda)
    w64 = weights_of(oracle, fmt, w, 9001, k)
    for form, m, n in forms:
        a = np.random.default_rng(m).standard_normal((m, k)).astype(np.float16)
        da, part = torch.from_numpy(a).to(cuda), dw[: Q.packed_bytes(fmt, n * k)]
        want = a.astype(np.float64) @ w64[:n].T
        plain = ops.gemm_f16(fmt, part, da, n, k, out_dtype=torch.float32)
        name = kernel_name()
        assert name.startswith(f"gemm_skinny_kernel<{Q.NAMES[fmt]},{form[0]},{form[1]},") and "arranged" not in name, (name, form, m, n)
        arranged = ops.gemm_f16_arranged(fmt, part, ops.ArrangedA(da), n, out_dtype=torch.float32)
        base = ",".join(name[:-1].split(",")[:4]) + ",arranged"
        assert kernel_name() in [base + how for how in (">", ",turned>", ",full>")]
        assert torch.equal(plain, arranged)
        assert_close(plain.cpu().numpy(), want, f"{Q.NAMES[fmt]} {m}x{n}x{k} {form}", tol=TOL, plain_tol=2e-4)


# m, n, k; the forms that rows of these sizes take on a part of 256 CUs (16-row operands, row tiles of W, slices, then how they are
# fetched) with their formats, "" all others; arranged activations where not the same tiles, "arranged".
FETCHES = [
    (17, 40, 8224, {"1,1,2,pairs,deep": ""}, {"1,1,2,arranged,turned": "Q8_0 GGUF_Q8_0"}),
    (9, 300, 2048, {"1,1,1,pairs,deep": ""}, {}),
    (29, 3000, 8448, {"2,1,1": "GGUF_Q4_0 GGUF_Q4_K", "2,1,1,pairs,deep": ""}, {"2,1,1,arranged,turned": "Q8_0"}),
    (17, 3000, 4096, {"2,1,1,pairs,deep": ""}, {}),
    (33, 4090, 1056, {"3,1,1": "GGUF_Q8_0", "3,1,1,pairs": ""}, {}),
    (33, 4090, 4096, {"3,1,1,pairs,deep": "GGUF_Q8_0", "3,1,1,pairs": ""}, {}),
    (9, 5000, 256, {"1,2,1,pairs,deep": "Q4_K", "1,2,1,pairs": ""}, {}),
    (9, 5000, 4096, {"1,2,1,pairs,deep": "Q4_0 Q4_K Q6_K GGUF_Q4_K", "1,2,1,pairs": ""}, {}),
    (17, 5000, 4128, {"2,2,1,pairs,deep": "Q4_0 Q4_K Q6_K GGUF_Q4_K", "2,2,1,pairs": ""}, {"2,2,1,arranged,turned": "Q8_0"}),
    (20, 8193, 8192, {"2,2,1,pairs,full": ""}, {"2,2,1,arranged,turned": "Q8_0", "2,2,1,arranged,full": "GGUF_Q4_K"}),
    (33, 8225, 416, {"3,2,1,full": "Q4_K", "3,2,1,pairs,full": ""}, {}),
    (56, 8250, 352, {"4,2,1,full": "Q4_0 Q6_K", "4,2,1,full,turned": "GGUF_Q4_0", "4,2,1": "Q8_0", "4,2,1,pairs": "GGUF_Q8_0", "4,2,1,pairs,full": ""}, {}),
    (60, 8208, 1280, {"4,2,1,full": "Q4_0 Q6_K", "4,2,1,full,turned": "GGUF_Q4_0", "4,2,1,pairs": "GGUF_Q8_0", "4,2,1,pairs,full": ""}, {}),
    (75, 8000, 224, {"3,2,2,pairs,full": "Q4_0 GGUF_Q4_0", "5,2,1,pairs": ""}, {"6,2,1,arranged": "GGUF_Q6_K"}),
    (80, 8300, 256, {"3,2,2,pairs,full": "Q4_0 GGUF_Q4_0", "5,2,1": "Q6_K", "6,2,1": "GGUF_Q6_K", "5,2,1,pairs": ""}, {}),
    (85, 8250, 192, {"3,2,2,pairs,full": "Q4_0 GGUF_Q4_0", "6,2,1": "Q6_K GGUF_Q6_K GGUF_Q8_0", "6,2,1,pairs": ""}, {}),
    (90, 8208, 1280, {"3,2,2,pairs,full": "Q4_0 GGUF_Q4_0", "6,2,1": "Q6_K GGUF_Q6_K", "6,2,1,pairs": ""}, {}),
    (96, 16400, 256, {"3,2,2,pairs,full": "Q4_0 GGUF_Q4_0", "6,2,1": "Q6_K GGUF_Q6_K GGUF_Q8_0", "6,2,1,pairs": ""}, {}),
    (150, 5001, 544, {"4,2,3,full": "Q4_0", "4,2,3,full,turned": "GGUF_Q4_0", "5,2,2": "Q6_K", "6,2,2": "GGUF_Q6_K", "5,2,2,pairs": ""}, {}),
]


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k,rows,others", FETCHES, ids=lambda v: str(v) if isinstance(v, int) else "")
def test_rows_in_pairs_of_groups(m, n, k, rows, others, fmt, oracle, cuda):
    """Rows fetched as pairs of groups and as single ones, one and two pairs ahead, with registers for one and two workgroups per CU;
    arranged activations with either operand turned, at the sizes where one form takes over from the other; last pairs of one group, and rows
    past the last that are not a multiple of eight: that it is the form taken, its results, and that both orders of the activations give
    the same bits."""
    import torch
    from rocmforge_amd import ops
    n, k = shape_of(fmt, n, k)
    w = Q.make_weights(fmt, n, k, seed=fmt)
    a = np.random.default_rng(m).standard_normal((m, k)).astype(np.float16)
    dw, da = torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda)
    label = Q.NAMES[fmt]
    form = next(f for f, formats in rows.items() if formats == "" or label in formats.split())
    got = ops.gemm_f16(fmt, dw, da, n, k, out_dtype=torch.float32)
    assert kernel_name() == f"gemm_skinny_kernel<{label},{form}>"
    arranged = ops.gemm_f16_arranged(fmt, dw, ops.ArrangedA(da), n, out_dtype=torch.float32)
    other = next((f for f, formats in others.items() if label in formats.split()), ",".join(form.split(",")[:3]) + ",arranged")
    assert kernel_name() == f"gemm_skinny_kernel<{label},{other}>"
    assert torch.equal(got, arranged)
    pick = np.unique(np.concatenate([np.arange(0, n, max(1, n // 61)), np.arange(n - 20, n)]))
    w64 = weights_of(oracle, fmt, w, n, k)[pick]
    assert_close(got.cpu().numpy()[:, pick], a.astype(np.float64) @ w64.T, f"{label} {m}x{n}x{k} {form}", tol=TOL, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", BATCH_FORMATS)
@pytest.mark.parametrize("norm", [False, True])
def test_every_decode_batch_kernel(fmt, norm, oracle, cuda):
    """Every form of the float32 kernel (row tiles of W, vectors) alone and with the norm: that it is the one taken, and its
    results."""
    import torch
    from rocmforge_amd import ops
    k = 768
    w = Q.make_weights(fmt, 13400, k, seed=fmt)
    dw = torch.from_numpy(w).to(cuda)
    w64 = weights_of(oracle, fmt, w, 13400, k)
    nw = (1 + 0.1 * np.random.default_rng(1).standard_normal(k)).astype(np.float32)
    for (tj, mv), m, n in [((1, 4), 4, 1101), ((2, 4), 3, 5401), ((2, 4), 4, 13399), ((1, 8), 5, 1101), ((2, 8), 8, 5401), ((4, 8), 7, 13399)]:
        x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32) * 3
        dx, part = torch.from_numpy(x).to(cuda), dw[: Q.packed_bytes(fmt, n * k)]
        x64 = x.astype(np.float64)
        if norm:
            got = ops.rms_norm_gemv(fmt, part, dx, torch.from_numpy(nw).to(cuda), 1e-5, n, k)
            x64 = x64 / np.sqrt((x64 * x64).mean(axis=1, keepdims=True) + 1e-5) * nw
        else:
            got = ops.gemv(fmt, part, dx, n, k)
        label = "MXFP6" if fmt == Q.MXFP6_E2M3 else Q.NAMES[fmt]
        assert kernel_name() == f"gemv_skinny_kernel<{label},{tj},{mv},{int(norm)}>"
        assert_close(got.cpu().numpy(), x64 @ w64[:n].T, f"{Q.NAMES[fmt]} {m}x{n}x{k}", tol=TOL, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(300, 96, 2048), (700, 200, 4096)])
def test_arranged_prompts_of_many_rows(fmt, m, n, k, oracle, cuda):
    """Arranged activations of 256 rows and more take the few-row kernel over narrow matrices (they cannot be split along k):
    slices of 16 rows and of more."""
    import torch
    from rocmforge_amd import ops
    w = Q.make_weights(fmt, n, k, seed=fmt)
    a = np.random.default_rng(m).standard_normal((m, k)).astype(np.float16)
    got = ops.gemm_f16_arranged(fmt, torch.from_numpy(w).to(cuda), ops.ArrangedA(torch.from_numpy(a).to(cuda)), n, out_dtype=torch.float32)
    assert kernel_name().startswith("gemm_skinny_kernel") != (fmt == Q.Q4_K)       # (Q4_K: as plain ones, which are split)
    # (Q4_K's tiled kernel multiplies q * scale rounded to fp16 once)
    assert_close(got.cpu().numpy(), a.astype(np.float64) @ weights_of(oracle, fmt, w, n, k).T, f"{Q.NAMES[fmt]} {m}x{n}x{k}",
                 tol=1e-3 if fmt == Q.Q4_K else TOL, plain_tol=None if fmt == Q.Q4_K else 2e-4)


@pytest.mark.parametrize("fmt", [Q.Q8_0, Q.GGUF_Q8_0])
@pytest.mark.parametrize("m,k", [(2, 1024), (4, 1024), (5, 4096), (8, 4096)])
def test_q8_0_batches_over_their_own_input(fmt, m, k, cuda):
    import torch
    from rocmforge_amd import ops
    w = torch.from_numpy(Q.make_weights(fmt, k, k, seed=1)).to(cuda)
    x = torch.randn((m, k), generator=torch.Generator(device="cpu").manual_seed(2)).to(cuda)
    want = ops.gemv(fmt, w, x, k, k)
    into = x.clone()
    ops.gemv(fmt, w, into, k, k, out=into)
    assert torch.equal(into, want)
