"""GPU parity: prefill GEMM for Q4_0 / Q8_0 / Q4_K / Q6_K (the reference's layouts
and the GGUF file layouts) on the fp16 matrix cores against the CPU oracle
(dequantise as the reference -- for the GGUF layouts, as ggml -- does, then the
reference's sequential fp32 matmul over the fp16 activations widened to f32)."""
import numpy as np
import pytest

from helpers import assert_close, error_report
from rocmforge_amd import quantize as Q

pytestmark = pytest.mark.gpu

FORMATS = [Q.Q4_0, Q.Q8_0, Q.Q4_K, Q.Q6_K, Q.GGUF_Q4_0, Q.GGUF_Q8_0, Q.GGUF_Q4_K, Q.GGUF_Q6_K]


def acts(m, k, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    return rng.standard_normal((m, k), dtype=np.float32).astype(np.float16)


def weights(fmt, n, k, seed):
    if fmt == Q.Q4_K and seed % 2:
        # a real min/max-free quantisation of N(0, 0.02) data (one-sided sub-blocks) next to the synthetic blocks
        rng = np.random.Generator(np.random.PCG64(seed))
        return Q.quantize_q4_k_onesided(rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    return Q.make_weights(fmt, n, k, seed=seed)


def gguf_q4_k_fused(w, n, k):
    """GGUF Q4_K values as the kernel forms them: (d * sc) * q - dmin * m as ONE fused multiply-add in f32
    (the float64 expression below is exact, so its f32 rounding is the fused result)."""
    b = np.frombuffer(bytes(w), np.uint8).reshape(-1, 144)
    d = b[:, 0:2].copy().view("<f2").astype(np.float32)
    dmin = b[:, 2:4].copy().view("<f2").astype(np.float32)
    s = b[:, 4:16].astype(np.uint32)
    sc = np.concatenate([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], axis=1).astype(np.float32)
    mn = np.concatenate([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], axis=1).astype(np.float32)
    qs = b[:, 16:].reshape(-1, 4, 32)
    q = np.stack([qs & 15, qs >> 4], axis=2).reshape(-1, 8, 32).astype(np.float64)
    d1 = (d * sc).astype(np.float32).astype(np.float64)[:, :, None]
    m1 = (dmin * mn).astype(np.float32).astype(np.float64)[:, :, None]
    return (d1 * q - m1).astype(np.float32).reshape(n, k)


def exact_weight_product(oracle, fmt, w, a, n, k):
    """The contraction of the decoded f32 weights with the fp16 activations, float64 sums: what the two-plane kernel
    is built to compute to 2^-22 per weight (hi = fp16(v), lo = fp16(v - hi))."""
    w32 = gguf_q4_k_fused(w, n, k) if fmt == Q.GGUF_Q4_K else oracle.dequantize(fmt, w, n * k).reshape(n, k)
    return a.astype(np.float64) @ w32.astype(np.float64).T


# The 256-byte Q4_K layout is contracted with q * scale as ONE fp16 operand (relative 2^-12 per weight) beside its exact
# integer mins; at the size of config 4 its plain relative error is 4.9e-4, at short k it can pass 1e-3 on outputs a
# tenth of the typical size, so for that format the small shapes are held to the first figure only.  Every other format
# runs two planes and is held to both.
def plain_tol_of(fmt, k):
    return None if fmt == Q.Q4_K and k < 4096 else 1e-3


def run(fmt, w, a, n, k, cuda, out_dtype):
    import torch
    from rocmforge_amd import ops
    out = ops.gemm_f16(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda), n, k, out_dtype=out_dtype)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k", [(1, 32, 256), (33, 70, 256), (300, 200, 512), (256, 128, 1024), (512, 259, 768)])
def test_small_shapes_fp32_out(fmt, m, n, k, oracle, cuda):
    import torch
    w, a = weights(fmt, n, k, 100 + fmt + m), acts(m, k, 200 + n)
    out = run(fmt, w, a, n, k, cuda, torch.float32).cpu().numpy()
    want = oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k)
    assert_close(out, want, f"{Q.NAMES[fmt]} {m}x{n}x{k}", plain_tol=plain_tol_of(fmt, k))
    # against the float64 contraction of the same weights only the fp32 summation order is left
    if fmt != Q.Q4_K:
        assert_close(out, exact_weight_product(oracle, fmt, w, a, n, k), f"{Q.NAMES[fmt]} {m}x{n}x{k} (float64 sums)", tol=2e-5,
                     plain_tol=2e-4)


def kernel_name():
    from rocmforge_amd import _lib
    return _lib.lib().rfq_bench_last_gemv_kernel().decode()


@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.Q8_0, Q.GGUF_Q4_0, Q.GGUF_Q8_0])
@pytest.mark.parametrize("m,kernel", [(40, "gemm_skinny_kernel"), (300, "gemm_kq_kernel")])
def test_k_not_a_multiple_of_the_stage(fmt, m, kernel, oracle, cuda):
    import torch
    n, k = 96, 96 + 64 * 3                                               # k % 64 == 32
    w, a = weights(fmt, n, k, 7), acts(m, k, 8)
    out = run(fmt, w, a, n, k, cuda, torch.float32).cpu().numpy()
    assert kernel_name().startswith(kernel)
    assert_close(out, oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k), "k tail")
    assert_close(out, exact_weight_product(oracle, fmt, w, a, n, k), "k tail (float64 sums)", tol=2e-5, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", FORMATS)
def test_ragged_tiles_of_few_rows(fmt, oracle, cuda):
    """Fewer than 256 rows over a matrix wide enough for the tiled kernel: one row tile, not full, and a ragged last column tile."""
    import torch
    m, n, k = 201, 14330, 2048
    w, a = weights(fmt, n, k, 71), acts(m, k, 72)
    out = run(fmt, w, a, n, k, cuda, torch.float32).cpu().numpy()
    assert kernel_name().startswith("gemm_kq_kernel")
    w64 = (gguf_q4_k_fused(w, n, k) if fmt == Q.GGUF_Q4_K else oracle.dequantize(fmt, w, n * k).reshape(n, k)).astype(np.float64)
    # (the 256-byte Q4_K layout rounds q * scale to fp16: errors of at most 2^-11 of it, evenly spread between two of its
    # codes' neighbours, 2^-11 / sqrt(12) = 1.4e-4 rms; the largest of three million normally distributed sums is 5.2 times that,
    # 7.4e-4 of what q * scale contributes, which the opposite mins leave up to twice the output's size: 1.5e-3)
    assert_close(out, a.astype(np.float64) @ w64.T, f"{Q.NAMES[fmt]} {m}x{n}x{k}", tol=1.5e-3 if fmt == Q.Q4_K else 2e-5,
                 plain_tol=None if fmt == Q.Q4_K else 2e-4)


@pytest.mark.parametrize("fmt", FORMATS)
def test_fp16_output_is_the_rounded_fp32_output(fmt, cuda):
    import torch
    m, n, k = 130, 264, 512
    w, a = weights(fmt, n, k, 31), acts(m, k, 32)
    f32 = run(fmt, w, a, n, k, cuda, torch.float32)
    f16 = run(fmt, w, a, n, k, cuda, torch.float16)
    assert torch.equal(f16, f32.to(torch.float16))                        # same accumulation, RNE cast


@pytest.mark.parametrize("fmt", [Q.Q4_K, Q.Q6_K, Q.GGUF_Q4_K, Q.GGUF_Q6_K])
def test_full_size_sampled(fmt, oracle, cuda):
    """M=512, K=4096, N=14336, fp16 in and out: sampled output columns against
    the oracle, and a checksum over every output:
    sum_n out[m, n] = A[m, :] . sum_n W[n, :]."""
    import torch
    m, n, k = 512, 14336, 4096
    w, a = Q.make_weights(fmt, n, k, seed=20260004), acts(m, k, 20260014)
    f32 = run(fmt, w, a, n, k, cuda, torch.float32)
    f16 = run(fmt, w, a, n, k, cuda, torch.float16)
    assert torch.equal(f16, f32.to(torch.float16))
    cols = np.array([0, 1, 31, 32, 127, 128, 4095, 7000, 14335])
    want = oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k, rows=cols)
    got = f32[:, torch.from_numpy(cols).to(cuda)].cpu().numpy()
    assert_close(got, want, "sampled fp32")
    print(f"{Q.NAMES[fmt]} 512x14336x4096, {cols.size} sampled columns, fp32 out: {error_report(got, want)}")
    got16 = f16[:, torch.from_numpy(cols).to(cuda)].float().cpu().numpy()
    assert_close(got16, want, "sampled fp16", tol=1e-3 + 2.0 ** -11)      # one fp16 rounding on top
    # every output against the float64 contraction of the decoded weights (a handful of weight rows gone wrong would
    # pass between the sampled columns and under the checksum): the exact forms to fp32 level, the 256-byte Q4_K
    # layout's single rounded operand to its 2^-12 per weight
    w64 = (gguf_q4_k_fused(w, n, k) if fmt == Q.GGUF_Q4_K else oracle.dequantize(fmt, w, n * k).reshape(n, k)).astype(np.float64)
    full = a.astype(np.float64) @ w64.T
    got_all = f32.cpu().numpy()
    rms = float(np.sqrt(np.mean(full * full)))
    per_row = np.max(np.abs(got_all - full), axis=0) / rms                  # worst output of each weight row
    print(f"{Q.NAMES[fmt]} all {m * n} outputs against float64: worst weight row {per_row.max():.2e} of rms(out), "
          f"median {np.median(per_row):.2e}")
    assert per_row.max() <= (1e-3 if fmt == Q.Q4_K else 2e-5), (Q.NAMES[fmt], int(np.argmax(per_row)), float(per_row.max()))
    del w64, full, got_all
    wsum = oracle.dequantize(fmt, w, n * k).reshape(n, k).astype(np.float64).sum(axis=0)
    check = f32.double().sum(dim=1).cpu().numpy()
    # each output carries the fp16 rounding of its weights (about 1e-4 rms, random sign): the sums of
    # 14336 of them agree to the same order; one wrong element would move a sum by about 1e-2
    assert_close(check, a.astype(np.float64) @ wsum, "row checksums", tol=1e-3)


@pytest.mark.parametrize("fmt", [Q.Q6_K, Q.GGUF_Q4_K, Q.GGUF_Q6_K, Q.Q8_0])
def test_one_plane_is_the_fp16_rounded_contraction(fmt, oracle, cuda):
    """RFQ_GEMM_ONE_PLANE: every weight as one fp16 operand.  Pinned by the float64 contraction of the weights rounded
    once to fp16; against the oracle its worst output lands at about 1e-3 of the typical output size (1.003e-3 for
    Q6_K here), which is why it is not the default."""
    import torch
    from rocmforge_amd import ops
    m, n, k = 300, 200, 512
    w, a = weights(fmt, n, k, 41), acts(m, k, 42)
    out = ops.gemm_f16(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda), n, k, out_dtype=torch.float32,
                       one_plane=True).cpu().numpy()
    w32 = gguf_q4_k_fused(w, n, k) if fmt == Q.GGUF_Q4_K else oracle.dequantize(fmt, w, n * k).reshape(n, k)
    rounded = a.astype(np.float64) @ w32.astype(np.float16).astype(np.float64).T
    assert_close(out, rounded, "one plane (rounded weights)", tol=2e-5, plain_tol=2e-4)
    assert_close(out, oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k), "one plane", tol=1.5e-3, plain_tol=None)
    two = ops.gemm_f16(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda), n, k, out_dtype=torch.float32).cpu().numpy()
    assert not np.array_equal(out, two)


@pytest.mark.parametrize("m,n,k,arranged,kernel", [(70, 140, 2048, False, "gemm_skinny_kernel<GGUF_Q4_K,"), (70, 140, 2048, True, "gemm_skinny_kernel<GGUF_Q4_K,"),
                                                   (300, 140, 2048, False, "gemm_kq_kernel<GGUF_Q4_K,codes of 64,2>"),
                                                   (700, 3700, 2048, True, "gemm_kq_kernel<GGUF_Q4_K,codes of 128,1,arranged>"),
                                                   (300, 14336, 2048, True, "gemm_kq_kernel<GGUF_Q4_K,codes of 192,1,arranged>"),
                                                   (512, 14336, 2048, False, "gemm_kq_kernel<GGUF_Q4_K,1,1>"),
                                                   (512, 14336, 2048, True, "gemm_kq_kernel<GGUF_Q4_K,1,1,arranged>"),
                                                   (511, 4000, 4096, False, "gemm_kq_kernel<GGUF_Q4_K,1,4>")])
def test_gguf_q4_k_super_block_scales_of_any_size(m, n, k, arranged, kernel, oracle, cuda):
    """GGUF_Q4_K is contracted with integer operands and the tiled kernels' accumulators run in units of the current super-block's
    d: super-blocks whose d is +0, -0, negative, or 2^+-8 times the neighbour's (also in a row's first and last block,
    and a whole row of zeros) must come out as the oracle's.  Each of the kernels, the special rows in front of a matrix wide
    enough for it: few rows, codes over row tiles that fit, whole tiles of 256 rows in one pass over k and in parts."""
    import torch
    from rocmforge_amd import ops
    special, nb = 140, k // 256
    w = weights(Q.GGUF_Q4_K, special, k, 51).copy()
    blocks = w.reshape(special, nb, 144)
    d = blocks[:, :, 0:2].copy().view("<f2")[..., 0]                      # [special, nb]
    rng = np.random.Generator(np.random.PCG64(52))
    d[0, :] = 0.0                                                         # a row without any scale (its mins remain)
    d[1, 0] = 0.0                                                         # zero first, later not
    d[2, nb - 1] = 0.0
    d[3, 3] = -0.0
    d[4, :] = -d[4, :]
    d[5, 1::2] *= np.float16(256.0)
    d[6, 1::2] /= np.float16(256.0)
    pick = rng.integers(0, nb, size=special)
    for r in range(7, special, 3): d[r, pick[r]] = 0.0
    for r in range(8, special, 5): d[r, pick[r]] *= np.float16(-64.0)
    blocks[:, :, 0:2] = d.astype("<f2")[..., None].view(np.uint8)
    dmin = blocks[:, :, 2:4].copy().view("<f2")[..., 0]
    dmin[9::4, 2] = 0.0
    dmin[10::7, :] = -dmin[10::7, :]
    blocks[:, :, 2:4] = dmin.astype("<f2")[..., None].view(np.uint8)
    a = acts(m, k, 53)
    wd = torch.from_numpy(w).to(cuda)
    if n > special:
        wide = torch.from_numpy(weights(Q.GGUF_Q4_K, n, k, 54)).to(cuda)
        wide[: wd.numel()] = wd
        wd = wide
    da = torch.from_numpy(a).to(cuda)
    if arranged:
        out = ops.gemm_f16_arranged(Q.GGUF_Q4_K, wd, ops.ArrangedA(da), n, out_dtype=torch.float32)
    else:
        out = ops.gemm_f16(Q.GGUF_Q4_K, wd, da, n, k, out_dtype=torch.float32)
    name = kernel_name()
    assert name == kernel or (kernel.endswith(",") and name.startswith(kernel)), name
    assert torch.isfinite(out).all()
    out = out[:, :special].cpu().numpy()
    want = oracle.qmatmul_nk(Q.GGUF_Q4_K, w, a.astype(np.float32), m, special, k)
    exact = exact_weight_product(oracle, Q.GGUF_Q4_K, w, a, special, k)
    for col in range(special):                                            # (each weight row against its own output size)
        assert_close(out[:, col], want[:, col], f"GGUF_Q4_K special super-block scales, weight row {col}")
        assert_close(out[:, col], exact[:, col], f"same (float64 sums), weight row {col}", tol=2e-5, plain_tol=2e-4)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("m,n,k,parts", [(300, 200, 2048, 2), (300, 130, 4096, 4), (257, 70, 8192, 8), (64, 130, 4096, 4), (33, 70, 8192, 8)])
def test_split_along_k(fmt, m, n, k, parts, oracle, cuda):
    """Few output tiles and a long k: the launch is split along k into whole super-blocks, the parts' f32 tiles are
    added in a fixed order: against the oracle, deterministic, and the fp16 output is the rounded fp32 output.  (Fewer than
    256 rows of such shapes go to the kernel for few rows, which does not split k, whatever rfq_gemm_f16_k_parts answers.)"""
    import torch
    from rocmforge_amd import _lib
    assert _lib.lib().rfq_gemm_f16_k_parts(m, n, k) == parts
    w, a = weights(fmt, n, k, 61 + fmt), acts(m, k, 62 + n)
    out = run(fmt, w, a, n, k, cuda, torch.float32)
    assert kernel_name().startswith("gemm_kq_kernel") == (m >= 256) and (m < 256 or kernel_name().endswith(f",{parts}>"))
    again = run(fmt, w, a, n, k, cuda, torch.float32)
    assert torch.equal(out, again)
    assert torch.equal(run(fmt, w, a, n, k, cuda, torch.float16), out.to(torch.float16))
    want = oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k)
    # (the 256-byte Q4_K layout here holds one-sided sub-blocks, mins of 0: its single fp16 operand q * scale then carries
    # the whole value and the plain figure is 4-7e-3 at any k, in one pass over k as in parts; held to the first figure)
    assert_close(out.cpu().numpy(), want, f"{Q.NAMES[fmt]} {m}x{n}x{k} in {parts} parts", plain_tol=None if fmt == Q.Q4_K else 1e-3)
    if fmt != Q.Q4_K:
        assert_close(out.cpu().numpy(), exact_weight_product(oracle, fmt, w, a, n, k), "same (float64 sums)", tol=2e-5, plain_tol=2e-4)
    else:
        w = weights(fmt, n, k, 62 + fmt)                                  # the synthetic blocks with integer mins: both figures
        out = run(fmt, w, a, n, k, cuda, torch.float32).cpu().numpy()
        assert_close(out, oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k), f"Q4_K synthetic blocks {m}x{n}x{k} in {parts} parts")


def test_k_parts_rule():
    from rocmforge_amd import _lib
    L = _lib.lib()
    assert L.rfq_gemm_f16_k_parts(512, 14336, 4096) == 1        # 224 tiles: the part is full
    assert L.rfq_gemm_f16_k_parts(512, 4096, 14336) == 4        # 64 tiles, 56 super-blocks: 4 x 14
    assert L.rfq_gemm_f16_k_parts(512, 4096, 4096) == 4
    assert L.rfq_gemm_f16_k_parts(512, 1024, 4096) == 4         # 16 tiles: k / parts stays >= 1024
    assert L.rfq_gemm_f16_k_parts(300, 384, 1024) == 1
    assert L.rfq_gemm_f16_k_parts(64, 128, 4128) == 1           # k not whole super-blocks
    assert L.rfq_gemm_f16_k_parts(0, 128, 4096) == 1


def test_weights_at_a_4_byte_offset_and_kept_temporary(oracle, cuda):
    """The weight loads need 4-byte alignment only; the per-stream temporary is
    reused by a smaller call after a larger one (and grown by a larger one).  256 rows and more: fewer take no temporary."""
    import torch
    from rocmforge_amd import ops
    fmt = Q.Q4_K
    outs = []
    for m, n, k in [(260, 128, 512), (400, 256, 1024), (260, 128, 512)]:
        w, a = weights(fmt, n, k, 6), acts(m, k, 7)
        buf = torch.zeros(w.size + 4, dtype=torch.uint8, device=cuda)
        buf[4:] = torch.from_numpy(w).to(cuda)
        out = ops.gemm_f16(fmt, buf[4:], torch.from_numpy(a).to(cuda), n, k, out_dtype=torch.float32)
        torch.cuda.synchronize()
        assert_close(out.cpu().numpy(), oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k), f"{m}x{n}x{k}", plain_tol=None)
        outs.append(out.cpu().numpy())
    assert np.array_equal(outs[0], outs[2])
    from rocmforge_amd import _lib
    assert kernel_name().startswith("gemm_kq_kernel")
    # one pass of a large call: its kept buffer (48 MiB) shows in the device's free memory once it is released
    big = torch.zeros((4096, 6144), dtype=torch.float16, device=cuda)
    ops.gemm_f16(Q.Q8_0, torch.zeros(Q.packed_bytes(Q.Q8_0, 128 * 6144), dtype=torch.uint8, device=cuda), big, 128, 6144)
    torch.cuda.synchronize()
    held = torch.cuda.mem_get_info()[0]
    assert _lib.lib().rfq_release_temporaries() == _lib.OK               # the next call allocates again
    assert torch.cuda.mem_get_info()[0] >= held + (40 << 20)
    w, a = weights(fmt, 128, 512, 6), acts(260, 512, 7)
    again = ops.gemm_f16(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda), 128, 512, out_dtype=torch.float32)
    torch.cuda.synchronize()
    assert np.array_equal(again.cpu().numpy(), outs[0])
    # a stream gives up its own buffer before it is destroyed; the default stream's stays
    side = torch.cuda.Stream()
    wd, ad = torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        on_side = ops.gemm_f16(fmt, wd, ad, 128, 512, out_dtype=torch.float32)
    side.synchronize()
    assert np.array_equal(on_side.cpu().numpy(), outs[0])
    import ctypes as C
    assert _lib.lib().rfq_release_stream_temporaries(C.c_void_p(side.cuda_stream)) == _lib.OK
    assert _lib.lib().rfq_release_stream_temporaries(C.c_void_p(side.cuda_stream)) == _lib.OK   # nothing left: still fine
    with torch.cuda.stream(side):
        on_side = ops.gemm_f16(fmt, wd, ad, 128, 512, out_dtype=torch.float32)      # allocates again
    side.synchronize()
    assert np.array_equal(on_side.cpu().numpy(), outs[0])
    assert np.array_equal(ops.gemm_f16(fmt, wd, ad, 128, 512, out_dtype=torch.float32).cpu().numpy(), outs[0])


def test_temporary_larger_than_the_kept_size(oracle, cuda):
    """m * k * 2 bytes above 64 MiB: the arranged activations go to a stream-ordered
    allocation that is released after the call."""
    import torch
    from rocmforge_amd import ops
    fmt, m, n, k = Q.Q4_K, 4096, 128, 8448
    w, a = weights(fmt, n, k, 8), acts(m, k, 9)
    out = ops.gemm_f16(fmt, torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda), n, k, out_dtype=torch.float32)
    torch.cuda.synchronize()
    cols = np.array([0, 5, 31, 32, 100, 127])
    want = oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k, rows=cols)
    assert_close(out[:, torch.from_numpy(cols).to(cuda)].cpu().numpy(), want, "large temporary")


def test_rejects_bad_arguments(cuda):
    import torch
    from rocmforge_amd import _lib, ops
    w = torch.zeros(Q.packed_bytes(Q.Q4_K, 64 * 256), dtype=torch.uint8, device=cuda)
    a = torch.zeros((4, 256), dtype=torch.float16, device=cuda)
    with pytest.raises(_lib.RfqError):
        ops.gemm_f16(Q.MXFP4, w, a, 64, 256)                              # MXFP goes through rfq_gemm_mx
    with pytest.raises(_lib.RfqError):
        ops.gemm_f16(Q.Q4_K, w[:-1], a, 64, 256)                          # byte count does not match the shape
    odd = torch.zeros(w.numel() + 1, dtype=torch.uint8, device=cuda)
    with pytest.raises(_lib.RfqError):
        ops.gemm_f16(Q.Q4_K, odd[1:], a, 64, 256)                         # weights not 4-byte aligned


@pytest.mark.parametrize("fmt", [Q.GGUF_Q4_0, Q.GGUF_Q8_0, Q.GGUF_Q6_K])
def test_gguf_blocks_at_a_2_byte_phase(fmt, oracle, cuda):
    """18-, 34- and 210-byte blocks sit at every 2-byte phase of a dword along a row; an odd number of
    blocks per row also moves each row's start by 2 bytes against the previous one."""
    import torch
    m, n = 48, 130
    k = 32 * 7 if fmt != Q.GGUF_Q6_K else 256 * 3
    w, a = weights(fmt, n, k, 41), acts(m, k, 42)
    out = run(fmt, w, a, n, k, cuda, torch.float32).cpu().numpy()
    assert_close(out, oracle.qmatmul_nk(fmt, w, a.astype(np.float32), m, n, k), f"{Q.NAMES[fmt]} odd block count")


# Activations arranged once for several projections: the same kernels, bit-identical results; nothing is
# allocated or kept, so the pair may be recorded into a graph without a call beforehand.
@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.Q8_0, Q.Q4_K, Q.Q6_K, Q.GGUF_Q4_K, Q.GGUF_Q6_K])
@pytest.mark.parametrize("m,n,k", [(64, 128, 512), (300, 259, 768), (33, 130, 1024), (512, 256, 4096)])
def test_arranged_activations_give_the_same_bits(fmt, m, n, k, cuda):
    import torch
    from rocmforge_amd import ops
    w = torch.from_numpy(weights(fmt, n, k, 31)).to(cuda)
    a = torch.from_numpy(acts(m, k, 32)).to(cuda)
    A = ops.ArrangedA(a)
    from rocmforge_amd import _lib
    split = _lib.lib().rfq_gemm_f16_k_parts(m, n, k) > 1      # rfq_gemm_f16 then adds k in parts: another order of the fp32 sums
    assert split == ((m, n, k) == (512, 256, 4096))
    for dt in (torch.float32, torch.float16):
        want = ops.gemm_f16(fmt, w, a, n, k, out_dtype=dt)
        got = ops.gemm_f16_arranged(fmt, w, A, n, out_dtype=dt)
        torch.cuda.synchronize()
        if split:
            assert_close(got.float().cpu().numpy(), want.float().cpu().numpy(), f"{Q.NAMES[fmt]} {m}x{n}x{k} {dt}",
                         tol=2e-5 if dt == torch.float32 else 2.0 ** -10, plain_tol=None)
        else:
            assert torch.equal(got, want), f"{Q.NAMES[fmt]} {m}x{n}x{k} {dt}"
    w2 = torch.from_numpy(weights(fmt, n, k, 33)).to(cuda)                  # a second projection of the same input
    if not split:
        assert torch.equal(ops.gemm_f16_arranged(fmt, w2, A, n), ops.gemm_f16(fmt, w2, a, n, k))


def test_arranged_activations_in_a_graph_and_bad_sizes(cuda):
    import ctypes as C
    import torch
    from rocmforge_amd import _lib, ops
    fmt, m, n, k = Q.Q4_K, 96, 256, 1024
    w = torch.from_numpy(weights(fmt, n, k, 41)).to(cuda)
    a = torch.from_numpy(acts(m, k, 42)).to(cuda)
    want = ops.gemm_f16(fmt, w, a, n, k)
    L = _lib.lib()
    nbytes = L.rfq_gemm_f16_arranged_bytes(m, k)
    assert nbytes == 3 * 16 * 4096 + 3 * 4 * 1024 and L.rfq_gemm_f16_arranged_bytes(m, 1020) == 0
    buf = torch.empty(nbytes, dtype=torch.uint8, device=cuda)
    out = torch.empty((m, n), dtype=torch.float16, device=cuda)
    side = torch.cuda.Stream()                                              # a stream the library has never seen
    side.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        s = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        _lib.check(L.rfq_gemm_f16_arrange(C.c_void_p(a.data_ptr()), m, k, C.c_void_p(buf.data_ptr()), nbytes, s))
        _lib.check(L.rfq_gemm_f16_arranged(fmt, C.c_void_p(w.data_ptr()), w.numel(), C.c_void_p(buf.data_ptr()), nbytes,
                                           C.c_void_p(out.data_ptr()), _lib.F16, m, n, k, s))
    for _ in range(3):
        out.zero_()
        buf.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    one = C.c_void_p(buf.data_ptr())
    assert L.rfq_gemm_f16_arrange(C.c_void_p(a.data_ptr()), m, k, one, nbytes - 1, None) == _lib.E_SIZE
    assert L.rfq_gemm_f16_arranged(fmt, C.c_void_p(w.data_ptr()), w.numel(), one, nbytes - 1, C.c_void_p(out.data_ptr()),
                                   _lib.F16, m, n, k, None) == _lib.E_SIZE
    assert L.rfq_gemm_f16_arranged(fmt, C.c_void_p(w.data_ptr()), w.numel(), one, nbytes, C.c_void_p(out.data_ptr()),
                                   _lib.BF16, m, n, k, None) == _lib.E_BADARG


# The kernel on integer codes, each of its row tiles at ragged sizes: one row, one column tile and more, k of one stage (128), of
# whole stages, of a stage with one group and of one with three, in one part and in several.  Codes and activations are
# exact, the sums float32: about sqrt(k) * 2^-24 of a typical output off.
@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.Q8_0, Q.GGUF_Q4_0, Q.GGUF_Q8_0, Q.GGUF_Q4_K])
@pytest.mark.parametrize("m,n,k,rows,parts", [(257, 15, 32, 64, 1), (300, 1000, 160, 64, 1), (257, 129, 128, 64, 1), (300, 12000, 224, 192, 1), (512, 14340, 256, 256, 1),
                                              (700, 3700, 384, 128, 1), (333, 4990, 3072, 192, 3), (511, 4000, 4096, 256, 4), (260, 40, 2048, 64, 2)])
def test_integer_code_tiles(fmt, m, n, k, rows, parts, oracle, cuda):
    import torch
    from rocmforge_amd import _lib, ops
    if fmt == Q.GGUF_Q4_K:
        k = (k + 255) // 256 * 256
    assert _lib.lib().rfq_gemm_f16_k_parts(m, n, k) == parts
    w, a = weights(fmt, n, k, 7), acts(m, k, 8)
    dw, da = torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda)
    out = ops.gemm_f16(fmt, dw, da, n, k, out_dtype=torch.float32)
    # (GGUF_Q4_K over whole tiles of 256 rows keeps the kernel laid out by hand)
    form = "1" if fmt == Q.GGUF_Q4_K and rows == 256 else f"codes of {rows}"
    assert kernel_name() == f"gemm_kq_kernel<{Q.NAMES[fmt]},{form},{parts}>"
    pick = np.unique(np.concatenate([np.arange(0, n, max(1, n // 97)), np.arange(max(0, n - 130), n)]))
    want = a.astype(np.float64) @ (gguf_q4_k_fused(w, n, k) if fmt == Q.GGUF_Q4_K else oracle.dequantize(fmt, w, n * k).reshape(n, k))[pick].astype(np.float64).T
    assert_close(out.cpu().numpy()[:, pick], want, f"{Q.NAMES[fmt]} {m}x{n}x{k}", tol=2e-5, plain_tol=2e-4)
    assert torch.equal(ops.gemm_f16(fmt, dw, da, n, k), out.half())


@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.Q8_0])
@pytest.mark.parametrize("scale", [1e-40, 1e30])
def test_integer_codes_under_scales_of_any_size(fmt, scale, oracle, cuda):
    """float32 block scales that fp16 operands could not carry."""
    import torch
    m, n, k = 260, 130, 256
    w = weights(fmt, n, k, 3).reshape(-1, Q.BLOCK_BYTES[fmt]).copy()
    w[:, :4] = (w[:, :4].copy().view("<f4") * np.float32(scale)).view(np.uint8)
    a = acts(m, k, 4)
    out = run(fmt, w.reshape(-1), a, n, k, cuda, torch.float32).cpu().numpy()
    want = a.astype(np.float64) @ oracle.dequantize(fmt, w.reshape(-1), n * k).reshape(n, k).astype(np.float64).T
    # (subnormal scales: a result is a sum of 8 products, each rounded to a multiple of 2^-149)
    assert np.abs(out - want).max() <= 2e-5 * np.abs(want).max() + 16 * 2.0 ** -149


@pytest.mark.parametrize("fmt", [Q.Q4_0, Q.Q8_0, Q.GGUF_Q4_0, Q.GGUF_Q8_0, Q.GGUF_Q4_K])
@pytest.mark.parametrize("m,n,k,rows,parts", [(257, 129, 32, 64, 1), (300, 1000, 160, 64, 1), (300, 12000, 224, 192, 1), (512, 14340, 352, 256, 1), (700, 3700, 96, 128, 1),
                                              (333, 4990, 3072, 192, 3)])
def test_infinities_and_nan_under_integer_codes(fmt, m, n, k, rows, parts, oracle, cuda):
    """An infinity or a NaN in a row of the activations, in its first group, between and in the last, which may end inside a stage of 128
    (there the padding's products must add nothing): the outputs of that row are the infinity's products with its weights (one of
    zero is NaN) or NaN, every other row keeps its bits.  GGUF_Q4_K multiplies the mins with sums of the activations, whose two
    fp16 parts an infinity leaves as infinity and NaN: NaN."""
    import torch
    from rocmforge_amd import ops
    if fmt == Q.GGUF_Q4_K:
        k = (k + 255) // 256 * 256
    w, a = weights(fmt, n, k, 9), acts(m, k, 10)
    dw = torch.from_numpy(w).to(cuda)
    clean = ops.gemm_f16(fmt, dw, torch.from_numpy(a).to(cuda), n, k, out_dtype=torch.float32).cpu().numpy()
    bad = {0: (0, np.inf), 17: (k // 2, -np.inf), 64: (k - 1, np.nan), m - 2: (max(0, k - 33), np.inf), m - 1: (k - 1, -np.inf)}
    for row, (at, value) in bad.items(): a[row, at] = value
    got = ops.gemm_f16(fmt, dw, torch.from_numpy(a).to(cuda), n, k, out_dtype=torch.float32).cpu().numpy()
    form = "1" if fmt == Q.GGUF_Q4_K and rows == 256 else f"codes of {rows}"
    assert kernel_name() == f"gemm_kq_kernel<{Q.NAMES[fmt]},{form},{parts}>"
    w32 = oracle.dequantize(fmt, w, n * k).reshape(n, k)
    for row, (at, value) in bad.items():
        with np.errstate(invalid="ignore"):
            want = np.full(n, np.nan, np.float32) if fmt == Q.GGUF_Q4_K else w32[:, at] * np.float32(value)
        assert np.array_equal(got[row], want, equal_nan=True), (row, at, value)
    others = np.setdiff1d(np.arange(m), list(bad))
    assert np.array_equal(got[others], clean[others])


@pytest.mark.parametrize("m,n,k,rows", [(800, 13824, 1024, "1"), (1024, 11008, 512, "1"), (1536, 22016, 256, "1"), (700, 3700, 1024, "codes of 128"), (2048, 6144, 256, "1"),
                                        (768, 11264, 256, "codes of 192")])
def test_gguf_q4_k_smaller_tiles_where_they_save_time(m, n, k, rows, cuda):
    """Three rounds of 128 rows (or seven of 192) cost more than two (six) of the 256-row kernel, two rounds of 192 less than two of
    256.  What the kernels give is checked on a few columns against float64 sums."""
    import torch
    from rocmforge_amd import ops
    w, a = weights(Q.GGUF_Q4_K, n, k, 11), acts(m, k, 12)
    dw, da = torch.from_numpy(w).to(cuda), torch.from_numpy(a).to(cuda)
    out = ops.gemm_f16(Q.GGUF_Q4_K, dw, da, n, k, out_dtype=torch.float32).cpu().numpy()
    assert kernel_name() == f"gemm_kq_kernel<GGUF_Q4_K,{rows},1>"
    A = ops.ArrangedA(da)
    assert np.array_equal(ops.gemm_f16_arranged(Q.GGUF_Q4_K, dw, A, n, out_dtype=torch.float32).cpu().numpy(), out)
    assert kernel_name() == f"gemm_kq_kernel<GGUF_Q4_K,{rows},1,arranged>"
    pick = np.unique(np.concatenate([np.arange(0, n, 997), np.arange(n - 3, n)]))
    part = w.reshape(n, -1)[pick].reshape(-1)
    assert_close(out[:, pick], a.astype(np.float64) @ gguf_q4_k_fused(part, len(pick), k).astype(np.float64).T, f"{m}x{n}x{k}", tol=2e-5, plain_tol=2e-4)
