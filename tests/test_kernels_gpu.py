"""Each HIP kernel alone against a plain torch float32 statement of the same operation
(tests/cpu_kernels.py), at sizes other than the engine's test models use, with sizes that are
no multiple of any tile.  Tolerances follow the reference's ladder for its CUDA kernels
(crates/synaptix-kernels-cuda/tests/*: float32 1e-5 .. 1e-4, bf16 around 1e-2 on O(1) data)."""
import itertools
import math

import pytest
import torch

import cpu_kernels as ref
from synaptix_amd.kernels import runtime as rt

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
F32, BF16, I32 = torch.float32, torch.bfloat16, torch.int32


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from synaptix_amd.kernels import ops as o
    return o


def rnd(shape, seed, dtype=F32, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


def close(got, want, atol, rtol=0.0, what=""):
    got, want = got.detach().cpu().to(F32), want.detach().cpu().to(F32)
    assert torch.isfinite(got).all(), f"{what}: non-finite values"
    err = (got - want).abs()
    bound = atol + rtol * want.abs()
    bad = err > bound
    assert not bad.any(), f"{what}: max abs err {err.max():.3e} (allowed {atol:.1e} + {rtol:.1e}|x|), {int(bad.sum())} values off"


# ----------------------------------------------------------------------------- rows

@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("V,H,N", [(100, 24, 7), (1000, 4100, 3)])
def test_embed(ops, dtype, V, H, N):
    table = rnd((V, H), 1, dtype)
    ids = torch.tensor([(i * 37 + V - 1) % V for i in range(N)], dtype=I32)
    out = torch.empty((N, H), dtype=F32, device=DEV)
    ops.embed(table.to(DEV), ids.to(DEV), out)
    assert torch.equal(out.cpu(), table[ids.long()].to(F32))  # a copy: exact


@pytest.mark.parametrize("out_dtype,gain_dtype", [(F32, F32), (BF16, BF16), (BF16, F32)])
@pytest.mark.parametrize("N,H", [(5, 72), (3, 4096), (2, 5000)])
def test_add_rmsnorm(ops, out_dtype, gain_dtype, N, H):
    eps = 1e-5
    resid, delta = rnd((N, H), 2), rnd((N, H), 3)
    gain = (1 + 0.1 * rnd((H,), 4)).to(gain_dtype)
    want_resid = resid.clone()
    want = torch.empty((N, H), dtype=out_dtype)
    ref.add_rmsnorm(want_resid, delta, gain, eps, want)
    r = resid.to(DEV)
    out = torch.empty((N, H), dtype=out_dtype, device=DEV)
    ops.add_rmsnorm(r, delta.to(DEV), gain.to(DEV), eps, out)
    close(r, want_resid, 1e-6, what="residual sum")
    close(out, want, 1e-5 if out_dtype == F32 else 2e-2, 1e-5 if out_dtype == F32 else 1e-2, "normed")
    # without a delta the residual stays; with rows only those rows are normed and nothing is written
    r2 = resid.to(DEV)
    ops.add_rmsnorm(r2, None, gain.to(DEV), eps, out)
    assert torch.equal(r2.cpu(), resid)
    rows = torch.tensor([N - 1, 0], dtype=I32)
    out2 = torch.empty((2, H), dtype=out_dtype, device=DEV)
    want2 = torch.empty((2, H), dtype=out_dtype)
    ref.add_rmsnorm(resid.clone(), delta, gain, eps, want2, rows)
    ops.add_rmsnorm(r2, delta.to(DEV), gain.to(DEV), eps, out2, rows.to(DEV))
    assert torch.equal(r2.cpu(), resid)
    close(out2, want2, 1e-5 if out_dtype == F32 else 2e-2, 1e-5 if out_dtype == F32 else 1e-2, "gathered rows")


def test_norm_gains_stored_as_a_difference_from_one(ops):
    """gain_offset = 1: the gain is 1 + w in every kernel that norms (rows with the residual sum, rows of any
    width, the q/k heads of prompts in both of their kernels, the q/k heads inside decode attention)."""
    eps = 1e-5
    for H, dt in ((72, F32), (4096, BF16)):
        resid, delta = rnd((3, H), 2), rnd((3, H), 3)
        w = (0.1 * rnd((H,), 4)).to(dt)
        want = torch.empty((3, H), dtype=F32)
        ref.add_rmsnorm(resid.clone(), delta, 1 + w.float(), eps, want)
        got = torch.empty((3, H), dtype=F32, device=DEV)
        ops.add_rmsnorm(resid.to(DEV), delta.to(DEV), w.to(DEV), eps, got, gain_offset=1.0)
        close(got, want, 1e-5, 1e-5, "add_rmsnorm with 1 + w")
        x = rnd((5, H), 5)
        ref.rmsnorm_rows(x, 1 + w.float(), eps, want2 := torch.empty((5, H)))
        got2 = torch.empty((5, H), dtype=F32, device=DEV)
        ops.rmsnorm_rows(x.to(DEV), w.to(DEV), eps, got2, gain_offset=1.0)
        close(got2, want2, 1e-5, 1e-5, "rmsnorm_rows with 1 + w")
    # q/k heads: head size 128 takes the 16-byte kernel, 48 the general one
    for nh, nkv, hd in ((4, 2, 128), (6, 2, 48)):
        N, width = 5, (nh + 2 * nkv) * hd
        table = torch.arange(2, dtype=I32).view(1, 2)
        tok_seq, tok_pos = torch.zeros(N, dtype=I32), torch.arange(60, 60 + N, dtype=I32)
        qkv = rnd((N, width), 6, BF16)
        qg, kg = (0.2 * rnd((hd,), 7)).to(BF16), (0.2 * rnd((hd,), 8)).to(BF16)
        ang = torch.arange(80, dtype=F32)[:, None] * (0.3 / (1 + torch.arange(hd // 2, dtype=F32)))[None, :]
        cos, sin = torch.cos(ang), torch.sin(ang)
        k_ref, v_ref = torch.zeros((2, nkv, 64, hd), dtype=BF16), torch.zeros((2, nkv, hd, 64), dtype=BF16)
        q_ref = torch.empty((N, nh * hd), dtype=BF16)
        ref.qk_norm_rope_kv_write(qkv, q_ref, k_ref, v_ref, table, tok_seq, tok_pos, (1 + qg.float()), (1 + kg.float()),
                                  eps, cos, sin, nh, nkv, hd)
        d = lambda t: t.to(DEV)
        kd, vd = torch.zeros_like(k_ref).to(DEV), dv(torch.zeros_like(v_ref))
        q = torch.empty((N, nh * hd), dtype=BF16, device=DEV)
        ops.qk_norm_rope_kv_write(d(qkv), q, kd, vd, d(table), d(tok_seq), d(tok_pos), d(qg), d(kg), eps, d(cos), d(sin),
                                  nh, nkv, hd, gain_offset=1.0)
        close(q, q_ref.float(), 2e-2, 1e-2, f"q heads of size {hd} with 1 + w")
        close(kd, k_ref.float(), 2e-2, 1e-2, f"k heads of size {hd} with 1 + w")
        # one more token through decode attention with the q/k/v intake
        one = rnd((1, width), 9, BF16)
        seq_len = torch.tensor([66], dtype=I32)
        q1 = torch.empty((1, nh * hd), dtype=BF16)
        ref.qk_norm_rope_kv_write(one, q1, k_ref, v_ref, table, torch.zeros(1, dtype=I32), seq_len - 1, 1 + qg.float(),
                                  1 + kg.float(), eps, cos, sin, nh, nkv, hd)
        want = torch.empty((1, nh * hd), dtype=F32)
        ref.attention_f32(q1.float(), k_ref.float(), v_ref.float(), table, torch.zeros(1, dtype=I32), seq_len - 1, want,
                          0.1, 0, nh, nkv, hd)
        # positions 0..59 of the pages hold zeros: they take part in the softmax on both sides alike
        out = torch.empty((1, nh * hd), dtype=BF16, device=DEV)
        work = torch.empty(nh * 2 * (hd + 2), dtype=F32, device=DEV)
        ops.attention_decode_fused_bf16(d(one), kd, vd, d(table), d(seq_len), out, work, 2, 0.1, 0, nh, nkv, hd, d(qg),
                                        d(kg), eps, d(cos), d(sin), gain_offset=1.0)
        close(out, want, 2e-2, 1e-2, f"decode attention, head size {hd}, gains 1 + w")


def test_an_unknown_activation_is_refused_before_any_launch(ops):
    x = torch.zeros((2, 64), dtype=BF16, device=DEV)
    out = torch.zeros((2, 32), dtype=BF16, device=DEV)
    with pytest.raises(Exception, match="activation 'gelu'"):
        ops.swiglu(x, out, "gelu")
    with pytest.raises(Exception, match="activation 'relu'"):
        ops.gemm_swiglu(x, torch.zeros((64, 64), dtype=BF16, device=DEV), out, "relu")
    from synaptix_amd.kernels.build import load_library
    lib = load_library("core")
    assert lib.syn_swiglu(None, None, 0, 2, 32, 7, None) != 0 and b"activation code 7" in lib.syn_last_error()


def test_rmsnorm_eps_sits_inside_the_root(ops):
    # tiny x: sqrt(mean + eps) and sqrt(mean) + eps differ by orders of magnitude
    x = torch.full((1, 64), 1e-4)
    gain = torch.ones(64)
    out = torch.empty((1, 64), device=DEV)
    ops.rmsnorm_rows(x.to(DEV), gain.to(DEV), 1e-6, out)
    want = 1e-4 / math.sqrt(1e-8 + 1e-6)
    close(out, torch.full((1, 64), want), 1e-6, what="eps inside the root")


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("R,D", [(9, 16), (5, 80), (3, 200)])
def test_rmsnorm_rows(ops, dtype, R, D):
    x, gain = rnd((R, D), 5, dtype), (1 + 0.1 * rnd((D,), 6)).to(dtype)
    want = torch.empty_like(x)
    ref.rmsnorm_rows(x, gain, 1e-6, want)
    out = torch.empty((R, D), dtype=dtype, device=DEV)
    ops.rmsnorm_rows(x.to(DEV), gain.to(DEV), 1e-6, out)
    close(out, want, 1e-5 if dtype == F32 else 2e-2, 0 if dtype == F32 else 1e-2)


def test_rmsnorm_reference_vector(ops):
    """The vector of crates/synaptix-ops/tests/rms_norm.rs:76-95, against the float64 closed form."""
    x = torch.tensor([i * 0.1 - 1.0 for i in range(24)], dtype=F32).view(6, 4)
    w = torch.tensor([0.5, -0.25, 1.0, 2.0])
    out = torch.empty((6, 4), device=DEV)
    ops.rmsnorm_rows(x.to(DEV), w.to(DEV), 1e-6, out)
    xd = x.double()
    want = xd / torch.sqrt((xd * xd).mean(-1, keepdim=True) + 1e-6) * w.double()
    close(out, want.float(), 1e-5)


@pytest.mark.parametrize("dtype", [F32, BF16])
def test_swiglu(ops, dtype):
    N, I = 7, 176
    gu = rnd((N, 2 * I), 7, dtype, 2.0)
    want = torch.empty((N, I), dtype=dtype)
    ref.swiglu(gu, want)
    out = torch.empty((N, I), dtype=dtype, device=DEV)
    ops.swiglu(gu.to(DEV), out)
    close(out, want, 5e-6 if dtype == F32 else 1.5e-2, 0 if dtype == F32 else 1e-2)
    # swapping gate and up must change the result (a swapped fused layout would not be seen otherwise)
    swapped = torch.cat([gu[:, I:], gu[:, :I]], 1).contiguous()
    out2 = torch.empty((N, I), dtype=dtype, device=DEV)
    ops.swiglu(swapped.to(DEV), out2)
    assert (out2.cpu().float() - want.float()).abs().max() > 0.1


# ----------------------------------------------------------------------------- matrix product

@pytest.mark.parametrize("M,N,K", [(1, 33, 40), (7, 100, 72), (64, 64, 64), (65, 130, 100), (200, 70, 300)])
def test_gemm_f32(ops, M, N, K):
    x, w = rnd((M, K), 8), rnd((N, K), 9)
    out = torch.empty((M, N), device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), out)
    want = (x.double() @ w.double().T).float()
    close(out, want, 1e-4, 1e-5, f"gemm f32 {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(1, 16, 4), (3, 176, 64), (16, 33, 2052), (17, 64, 176), (32, 1000, 260), (33, 50, 1024), (64, 100, 4096),
                                   (40, 8200, 72), (64, 9000, 68),          # wide: the tiles take 33 rows already, K in eights
                                   (65, 33, 8), (66, 2560, 40), (129, 1000, 264), (490, 2570, 1000), (70, 20000, 96)])
def test_gemm_f32_on_the_matrix_units(ops, M, N, K):
    """Every split of the 32-bit products: few rows (1, 2 or 4 groups of 16), tiles of 64 x 64 and 64 x 32, K that ends inside a
    k-tile, ragged M and N; no more off than the plain kernel is on the same operands, up to a factor for the order of sums."""
    x, w = rnd((M, K), 8), rnd((N, K), 9)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), out)
    want = x.double() @ w.double().T
    plain = torch.empty((M, N), device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), plain, force_simt=True)
    off = lambda t: float((t.cpu().double() - want).norm() / want.norm())
    assert torch.isfinite(out).all() and off(out) <= 1.25 * off(plain) + 1e-8
    # K fused steps of 2^-24 each at most, on products of size one
    close(out, want.float(), 2 ** -24 * K * 4, 1e-6, f"gemm f32 {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(1, 16384, 36), (16, 16500, 68), (17, 6144, 40), (64, 6200, 36),       # a wide W with few rows
                                   (65, 40, 36), (320, 2560, 64), (640, 96, 32), (530, 1100, 36),         # bands of unequal height,
                                   (577, 2600, 36), (1100, 33, 40), (2100, 700, 36), (257, 8200, 32)])    # counts that 8 does not divide
def test_gemm_f32_tiles_cover_the_product(ops, M, N, K):
    """Tiles of 64 x 32, 32 x 64 and 32 x 32 dealt out to the XCDs in equal runs: every one is computed, and by its rows and columns."""
    x, w = rnd((M, K), 12), rnd((N, K), 13)
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), out)
    # K fused steps of 2^-24 each at most, on products of size one
    close(out, (x.double() @ w.double().T).float(), 2 ** -24 * K * 4, 1e-6, f"gemm f32 {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K", [(250, 12250, 36), (490, 6144, 64), (320, 16380, 100), (577, 13000, 40), (640, 16384, 32), (256, 16384, 36)])
def test_gemm_f32_squares_have_the_bits_of_single_rows(ops, M, N, K):
    """Tiles of 64 x 64 at 3, 5, 8 and 10 rounds and ragged ends, and of the halves at 4 rounds: every row as the kernel for few rows has it."""
    x, w = rnd((M, K), 16).to(DEV), rnd((N, K), 17).to(DEV)
    out, one = torch.full((M, N), float("nan"), device=DEV), torch.empty((1, N), device=DEV)
    ops.gemm(x, w, out)
    assert not bool(torch.isnan(out).any())
    for m in sorted({0, 31, 32, 63, 64, M // 2, M - 2, M - 1}):
        ops.gemm(x[m:m + 1].contiguous(), w, one)
        assert torch.equal(out[m:m + 1], one), m


@pytest.mark.parametrize("M,N,K", [(17, 6144, 1024), (18, 8192, 1024), (18, 8196, 1024), (19, 6144, 1024), (17, 8192, 1020)])
def test_gemm_f32_of_few_rows_has_the_same_bits_on_both_sides_of_the_rule(ops, M, N, K):
    """Around the sizes from which the tiles take 17 rows and more: row by row the bits that the kernel for few rows gives one row alone."""
    x, w = rnd((M, K), 14).to(DEV), rnd((N, K), 15).to(DEV)
    out, one = torch.full((M, N), float("nan"), device=DEV), torch.empty((1, N), device=DEV)
    ops.gemm(x, w, out)
    for m in (0, 15, 16, M - 1):
        ops.gemm(x[m:m + 1].contiguous(), w, one)
        assert torch.equal(out[m:m + 1], one), m


@pytest.mark.parametrize("N,K", [(48, 4), (33, 68), (100, 260), (2560, 1000), (1000, 2052), (8200, 544), (9000, 612)])
def test_gemm_f32_rows_do_not_depend_on_the_batch(ops, N, K):
    """Every split of the 32-bit products adds in the same order: a row has the same bits alone, among few and among many rows."""
    M = 300
    x, w = rnd((M, K), 10).to(DEV), rnd((N, K), 11).to(DEV)
    whole = torch.empty((M, N), device=DEV)
    ops.gemm(x, w, whole)
    for m in (1, 3, 16, 17, 32, 33, 64, 65, 128, 200):
        for lo in {0, M - m}:
            out = torch.empty((m, N), device=DEV)
            ops.gemm(x[lo:lo + m].contiguous(), w, out)
            assert torch.equal(out, whole[lo:lo + m]), (m, lo)


# which kernel these take: few rows whole and in blocks of 16; tiles of 16 x 64, 32 x 64, 32 x 128, 64 x 64 and 64 x 128, whole and with K cut;
# more rows than the parts of x are kept for at a time; K that ends inside a chunk, a class and a group
F32_EDGES = [(16, 1000, 4100), (64, 130, 1000), (33, 6148, 516), (16, 6144, 2560), (17, 2564, 4096), (31, 19460, 100), (96, 19456, 260),
             (65, 2570, 1028), (128, 2560, 2048), (300, 2561, 36), (490, 2560, 516), (300, 19460, 68), (2049, 70, 132), (2300, 1100, 64)]


@pytest.mark.parametrize("M,N,K", F32_EDGES)
def test_gemm_f32_in_parts_is_as_exact_as_32_bit_steps(ops, M, N, K):
    """Operands of mixed sizes through every kernel and rule of the 32-bit products: each result within what a chain of K / 32 + 40 rounded
    steps of the sum of magnitudes allows, the whole no further from 64 bits than fused multiply-adds, and a row's bits those of the row alone."""
    x, w = rnd((M, K), 31), rnd((N, K), 32)
    x[:, ::3] *= 1e-4
    w[::5] *= 300.0
    out = torch.full((M, N), float("nan"), device=DEV)
    xd, wd = x.to(DEV), w.to(DEV)
    ops.gemm(xd, wd, out)
    plain = torch.empty((M, N), device=DEV)
    ops.gemm(xd, wd, plain, force_simt=True)
    want, size = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    diff = (out.cpu().double() - want).abs()
    assert bool((diff <= 2.0 ** -23 * (K / 32 + 40) * size).all()), float((diff / size).max())
    assert float(diff.norm()) <= float((plain.cpu().double() - want).norm()) + 1e-8 * float(want.norm())
    one = torch.empty((1, N), device=DEV)
    for m in (0, M // 2, M - 1):
        ops.gemm(xd[m:m + 1].contiguous(), wd, one)
        assert torch.equal(out[m:m + 1], one), m


@pytest.mark.parametrize("M,N,K", [(3, 100, 260), (17, 6144, 1024), (96, 2560, 2048), (300, 2561, 36), (490, 19460, 68)])
def test_gemm_f32_keeps_what_is_no_number_and_what_is_large_or_small(ops, M, N, K):
    """Infinities and NaN in x and W give what fused multiply-adds give, in their rows and columns only; the largest numbers, which round to
    an infinity in 16 bits, and rows of numbers whose parts have no 16-bit form stay what they are."""
    x, w = rnd((M, K), 33), rnd((N, K), 34)
    x[0, 1], x[1, K - 1], x[2, 0] = float("inf"), float("nan"), float("-inf")
    w[5, K // 2], w[7, :] = float("inf"), 0.0
    big = torch.finfo(F32).max
    x[M - 1], w[9] = 0.0, 0.0
    x[M - 1, K - 4], w[9, K - 4] = big, 0.5
    out, plain = torch.empty((M, N), device=DEV), torch.empty((M, N), device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), out)
    ops.gemm(x.to(DEV), w.to(DEV), plain, force_simt=True)
    out, plain = out.cpu(), plain.cpu()
    assert torch.equal(out.isnan(), plain.isnan()) and torch.equal(out.isposinf(), plain.isposinf()) and torch.equal(out.isneginf(), plain.isneginf())
    assert float(out[M - 1, 9]) == 0.5 * big and bool(torch.isnan(out[0, 7])) and not bool(torch.isfinite(out[:3]).any() and torch.isfinite(out[1]).any())
    small = rnd((M, K), 35) * 1e-36
    ops.gemm(small.to(DEV), w[:5].contiguous().to(DEV), out := torch.empty((M, 5), device=DEV))
    want = small.double() @ w[:5].double().T
    # (a chain of K fused steps of 2^-24 each; the matrix units alone, which take parts below 2^-126 for zero, are off by 2.5e-5)
    assert float((out.cpu().double() - want).norm() / want.norm()) < 2.0 ** -24 * K


@pytest.mark.parametrize("nh,nkv,hd,window", [(8, 2, 64, 0), (8, 4, 32, 100), (4, 4, 6, 0), (8, 1, 128, 64)])
def test_attention_f32_does_not_depend_on_the_batch(ops, nh, nkv, hd, window):
    """Many tokens (a wave a head) and few of the same (the keys over four waves): the same bits."""
    past, new = [300, 0, 64], [4, 500, 129]
    lens = [p + n for p, n in zip(past, new)]
    width = max((T + 63) // 64 for T in lens)
    table = shuffled_table(len(past), width, 4)
    k, v = make_cache(len(past) * width, nkv, hd, F32, 33, fill="nan")
    fill_sequences(k, v, table, lens, nkv, hd, F32, 34)
    tok_seq, tok_pos, _, _, _ = step_arrays(past, new)
    q = rnd((len(tok_seq), nh * hd), 35, scale=2.0)
    d = lambda t: t.to(DEV)
    k, v, table = d(k), dv(v), d(table)

    def run(rows):
        out = torch.empty((len(rows), nh * hd), device=DEV)
        ops.attention_f32(d(q[rows]), k, v, table, d(tok_seq[rows]), d(tok_pos[rows]), out, 0.3, window, nh, nkv, hd)
        return out
    whole = run(torch.arange(len(tok_seq)))
    assert torch.isfinite(whole).all()
    for rows in (torch.tensor([0]), torch.tensor([3, 4, 503, 504, 632]), torch.arange(200, 330)):
        assert torch.equal(run(rows), whole[d(rows)])


@pytest.mark.parametrize("hd,past,new", [(6, [300, 0], [1, 2]), (6, [0, 70], [200, 150]), (32, [1000], [1]), (128, [70], [3]),
                                         (71, [70, 0], [200, 130]), (255, [130], [2])])
def test_attention_f32_splits_and_head_sizes(ops, hd, past, new):
    """Few tokens (the keys over four waves, more waves than blocks of keys among them) and many, head sizes that 16-byte loads
    do not divide, NaN in every slot behind a sequence's end."""
    nh, nkv = 8, 2
    lens = [p + n for p, n in zip(past, new)]
    width = max((T + 63) // 64 for T in lens) + 1
    table = shuffled_table(len(past), width, 3)
    k, v = make_cache(len(past) * width, nkv, hd, F32, 30, fill="nan")
    fill_sequences(k, v, table, lens, nkv, hd, F32, 31)
    tok_seq, tok_pos, _, _, _ = step_arrays(past, new)
    q = rnd((len(tok_seq), nh * hd), 32)
    want, out = torch.empty_like(q), torch.empty_like(q, device=DEV)
    ref.attention_f32(q, torch.nan_to_num(k), torch.nan_to_num(v), table, tok_seq, tok_pos, want, 0.3, 0, nh, nkv, hd)
    d = lambda t: t.to(DEV)
    ops.attention_f32(d(q), d(k), dv(v), d(table), d(tok_seq), d(tok_pos), out, 0.3, 0, nh, nkv, hd)
    close(out, want, 1e-5, 1e-5, "attention f32")


@pytest.mark.parametrize("nh,nkv,hd", [(32, 8, 128), (8, 2, 64), (12, 4, 16), (20, 2, 96), (8, 8, 32), (17, 1, 112), (10, 2, 48), (6, 3, 80)])
@pytest.mark.parametrize("odd", [False, True])
def test_attention_f32_of_prompts_has_the_bits_of_single_tokens(ops, nh, nkv, hd, odd):
    """16 (token, head) rows a workgroup on the matrix units against a wave a row (a page table with a row a token looks like single tokens):
    tiles over the ends of sequences, heads that do not divide 16, NaN behind the sequences' ends; `odd`: keys and values among the cached
    ones that are infinite, no number, or below the normal range."""
    past, new = [300, 0, 64, 7], [90, 200, 129, 1]
    lens = [p + n for p, n in zip(past, new)]
    width = max((T + 63) // 64 for T in lens)
    table = shuffled_table(len(past), width, 4)
    k, v = make_cache(len(past) * width, nkv, hd, F32, 33, fill="nan")
    fill_sequences(k, v, table, lens, nkv, hd, F32, 34)
    if odd:
        for b, at, x in ((0, 350, float("inf")), (1, 120, float("nan")), (1, 150, -float("inf")), (2, 100, 1e-39), (2, 170, 3e38)):
            page = int(table[b, at // 64])
            v[page, at % nkv, at % hd, at % 64] = x
            k[page, (at + 1) % nkv, at % 64, at % hd] = x
    tok_seq, tok_pos, _, _, _ = step_arrays(past, new)
    q = rnd((len(tok_seq), nh * hd), 35, scale=2.0)
    d = lambda t: t.to(DEV)
    k, v, n = d(k), dv(v), len(tok_seq)
    tall = torch.cat([table, torch.zeros((n, width), dtype=I32)])
    assert ops._mostly_prompts(n, table) and not ops._mostly_prompts(n, tall) and n * nh > 8 * ops.compute_units()
    outs = []
    for t in (table, tall):
        outs.append(torch.full((n, nh * hd), 7.0, device=DEV))
        ops.attention_f32(d(q), k, v, d(t), d(tok_seq), d(tok_pos), outs[-1], 0.3, 0, nh, nkv, hd)
    a, b = outs
    assert torch.equal(torch.isnan(a), torch.isnan(b)) and bool(torch.isnan(a).any()) == odd
    assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b)), int((torch.nan_to_num(a) != torch.nan_to_num(b)).sum())


@pytest.mark.parametrize("new", [1, 600])
def test_attention_f32_keeps_what_is_no_number(ops, new):
    """A key that is no number makes every result that sees it one, also where no other key stands in its block of 64; scores of
    -inf, a block full of them among others, weigh nothing.  With few tokens (the keys over four waves) and many."""
    nh, nkv, hd, T = 4, 2, 16, 700
    pages = (T + 63) // 64
    k, v, q = rnd((pages, nkv, 64, hd), 36), rnd((pages, nkv, hd, 64), 37), rnd((new, nh * hd), 38)
    table = torch.arange(pages, dtype=I32).view(1, pages)
    tok_seq, tok_pos = torch.zeros(new, dtype=I32), torch.arange(T - new, T, dtype=I32)
    d = lambda t: t.to(DEV)

    def run(k, pos=tok_pos):
        out = torch.empty((new, nh * hd), device=DEV)
        ops.attention_f32(d(q), d(k), d(v), d(table), d(tok_seq), d(pos), out, 0.3, 0, nh, nkv, hd)
        return out.cpu()
    bad = k.clone()
    bad[5, :, 0, 3] = float("nan")                       # position 320, the first of its block
    seen = torch.full((new,), 320, dtype=I32)            # ... and the last that is seen
    assert torch.isnan(run(bad, seen)).all() and torch.isfinite(run(bad, seen - 1)).all()
    assert torch.equal(torch.isnan(run(bad)).all(1), tok_pos >= 320) and torch.equal(torch.isnan(run(bad)).any(1), tok_pos >= 320)
    q = q.view(new, nh, hd)
    q[:, :, 0] = q[:, :, 0].abs() + 0.1
    q = q.view(new, nh * hd)
    low = k.clone()
    low[2, :, :, 0] = float("-inf")                      # every score of positions 128 to 191
    got, pos = run(low), tok_pos.clamp(max=127)
    assert torch.isfinite(got).all()
    low[3:, :, :, 0] = float("-inf")
    close(run(low).to(DEV), run(k, pos), 1e-5, 1e-5, "blocks that weigh nothing")


@pytest.mark.parametrize("out_dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K", [
    (1, 48, 64), (3, 1000, 176), (16, 100, 320), (17, 40, 72), (33, 1000, 128), (48, 70, 2048), (64, 4096, 512),
    (65, 130, 104), (128, 128, 32), (200, 300, 1000), (513, 257, 4096),
    (1700, 5120, 128),                  # several tiles a workgroup, the shortest K that the streamed tiles take
    (5, 30, 20), (70, 50, 36),          # K no multiple of 8: the plain kernel takes them
    (2048, 6144, 512), (1000, 12300, 136),   # many rows, ragged edges: streamed, and through registers (K = 136)
    (1000, 12544, 128), (300, 200, 64),   # K a multiple of 64: loads straight into LDS, streamed and (K = 64) in tiles of 128 x 128
    (8, 40000, 256), (40, 33000, 72), (64, 50000, 1000),   # wide
    (1, 9000, 520), (1, 70000, 136),                       # one row: W straight from memory, K over the waves
    (8, 70000, 264), (20, 66000, 72),                      # few rows, very wide: 32-row tiles, 256 deep
    (100, 300, 1024), (256, 520, 256), (129, 4096, 384), (255, 6144, 128),   # short prompts, narrow: 64-row tiles, several of them along M
])
def test_gemm_bf16(ops, out_dtype, M, N, K):
    x, w = rnd((M, K), 10, BF16), rnd((N, K), 11, BF16)
    out = torch.empty((M, N), dtype=out_dtype, device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), out)
    want = (x.double() @ w.double().T).float()
    # float accumulation of exact bf16 products: the only error is the order of the sum and the last rounding
    atol = 1e-3 * math.sqrt(K)
    close(out, want, atol if out_dtype == F32 else atol + 0.02, 0 if out_dtype == F32 else 1e-2, f"gemm bf16 {M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,S", [(1, 48, 4096, 4), (8, 4096, 4096, 4), (8, 100, 1000, 3), (16, 64, 12288, 8),
                                     (40, 70, 2048, 2), (64, 130, 520, 5), (8, 96, 1536, 5), (50, 200, 3072, 7),
                                     (300, 520, 1024, 2), (130, 260, 640, 3), (65, 33, 4096, 4),
                                     (200, 4096, 1024, 2), (256, 1000, 2048, 4),
                                     # short prompts cut along K: tiles of 128 x 128 up to 128 rows (to 256 in four slices and more), streamed ones beyond
                                     (66, 6144, 4096, 4), (128, 200, 4096, 8), (129, 4100, 1024, 2), (256, 1000, 2560, 4),
                                     (257, 520, 4096, 8), (400, 2000, 1152, 2), (512, 4096, 1024, 2),
                                     # ... to 256 in two slices where they leave few compute units without work, and beside that line
                                     (177, 6144, 2560, 2), (256, 8192, 2688, 2), (250, 7100, 4224, 2), (176, 6144, 2560, 2), (200, 6000, 2560, 2)])
def test_gemm_bf16_partial_sums_over_slices_of_k(ops, M, N, K, S):
    """[S, M, N]: slice s holds the sum over its part of K; the slices add up to the product, also
    when K is no multiple of the slice and the last slices are short or empty."""
    x, w = rnd((M, K), 14, BF16), rnd((N, K), 15, BF16)
    out = torch.full((S, M, N), float("nan"), dtype=F32, device=DEV)
    ops.gemm(x.to(DEV), w.to(DEV), out)
    want = (x.double() @ w.double().T).float()
    close(out.sum(0), want, 1e-3 * math.sqrt(K), what=f"sum of {S} slices")
    step = ((K + S - 1) // S + 127) // 128 * 128
    first = (x[:, :step].double() @ w[:, :step].double().T).float()
    close(out[0], first, 1e-3 * math.sqrt(step), what="first slice")
    # the consumer adds the slices: resid + sum(delta) normed
    H = N
    resid = rnd((M, H), 16)
    gain = (1 + 0.1 * rnd((H,), 17)).to(BF16)
    r = resid.to(DEV)
    normed = torch.empty((M, H), dtype=BF16, device=DEV)
    ops.add_rmsnorm(r, out, gain.to(DEV), 1e-6, normed)
    want_resid = resid + out.sum(0).cpu()
    close(r, want_resid, 1e-4, 1e-5, "residual + slices")
    want_n = torch.empty((M, H), dtype=BF16)
    ref.add_rmsnorm(want_resid.clone(), None, gain, 1e-6, want_n)
    close(normed, want_n, 2e-2, 1e-2, "norm of residual + slices")
    rows = torch.tensor([M - 1, 0], dtype=I32)
    got2 = torch.empty((2, H), dtype=F32, device=DEV)
    ops.add_rmsnorm(resid.to(DEV), out, gain.to(DEV), 1e-6, got2, rows.to(DEV))
    want2 = torch.empty((2, H), dtype=F32)
    ref.add_rmsnorm(resid.clone(), out.cpu(), gain, 1e-6, want2, rows)
    close(got2, want2, 1e-4, 1e-4, "gathered rows of residual + slices")


@pytest.mark.parametrize("M,I,K", [(1, 48, 64), (1, 2560, 4096), (1, 1008, 1096), (8, 2560, 4096), (7, 112, 1000), (33, 80, 136), (64, 1024, 512),
                                   (300, 400, 264), (2048, 3072, 256), (1000, 6272, 136), (8, 32784, 72),
                                   (1000, 6272, 128), (300, 400, 192),
                                   # 65 to 256 rows: all of x in one tile of 128, 192 or 256 rows and 96 or 128 rows of W, or streamed
                                   (65, 48, 64), (100, 1040, 448), (128, 12288, 512), (129, 400, 192), (192, 2000, 320),
                                   (193, 80, 1024), (256, 4864, 640), (200, 400, 72), (1700, 2560, 192)])
def test_gemm_with_the_gated_activation_inside(ops, M, I, K):
    """silu(x . Wg^T) * (x . Wu^T) from one product over the rows of Wg and Wu in turns of 16,
    against the two products and the activation in 64-bit; every tile shape of the kernel."""
    x, wg, wu = rnd((M, K), 18, BF16), rnd((I, K), 19, BF16), rnd((I, K), 20, BF16)
    paired = ops.pair_rows(wg.to(DEV), wu.to(DEV))
    assert paired.shape == (2 * I, K)
    assert torch.equal(paired[16:32].cpu(), wu[:16]) and torch.equal(paired[32:48].cpu(), wg[16:32])
    out = torch.full((M, I), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_swiglu(x.to(DEV), paired, out)
    g, u = x.double() @ wg.double().T, x.double() @ wu.double().T
    want = (g / (1 + torch.exp(-g)) * u).float()
    # products of standard deviation sqrt(K); one bf16 rounding of the result
    close(out, want, 2e-3 * K + 0.02, 1e-2, f"gated product {M}x{I}x{K}")
    with pytest.raises(Exception, match="turns of 16"):
        ops.pair_rows(wg[:24].to(DEV), wu[:24].to(DEV))
    with pytest.raises(Exception, match="paired rows"):
        ops.gemm_swiglu(x.to(DEV), paired[:48], torch.empty((M, 24), dtype=BF16, device=DEV))


@pytest.mark.parametrize("out_dtype", [BF16, F32])
@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (1, 4096, 4096), (8, 6144, 4096), (3, 48, 96), (5, 1008, 1120), (8, 16400, 160),
                                   (16, 64, 12288), (7, 80, 2080),
                                   (8, 32784, 96), (5, 40000, 4096), (13, 32784, 96)])   # very wide from 5 rows on: two groups of rows a wave, an odd number of groups
def test_gemm_over_weights_in_fragment_order(ops, out_dtype, M, N, K):
    """The products for few rows over pack_weight(W): every k-step and every row tile lands where the
    plain product has it, also where K is no multiple of the waves' turns and N of the workgroup's rows."""
    x, w = rnd((M, K), 26, BF16), rnd((N, K), 27, BF16)
    wp = ops.pack_weight(w.to(DEV))
    assert wp.shape == (N // 16, K // 32, 64, 8)
    assert torch.equal(ops.unpack_weight(wp).cpu(), w)
    # lane = 16 * (k % 32 // 8) + n % 16, element k % 8
    assert wp[N // 16 - 1, K // 32 - 1, 16 * 2 + 5, 3] == w[N - 16 + 5, K - 32 + 2 * 8 + 3]
    out = torch.full((M, N), float("nan"), dtype=out_dtype, device=DEV)
    ops.gemm_packed(x.to(DEV), wp, out)
    want = (x.double() @ w.double().T).float()
    atol = 1e-3 * math.sqrt(K)
    close(out, want, atol if out_dtype == F32 else atol + 0.02, 0 if out_dtype == F32 else 1e-2, f"packed {M}x{N}x{K}")
    if out_dtype == F32:
        # partial sums over slices of K: each slice its own part, the slices add up, also when the last ones are short or empty
        for S in (2, 3, 7):
            parts = torch.full((S, M, N), float("nan"), dtype=F32, device=DEV)
            ops.gemm_packed(x.to(DEV), wp, parts)
            close(parts.sum(0), want, atol, what=f"packed {M}x{N}x{K} in {S} slices")
            step = -(-(K // 32) // S) * 32
            first = (x[:, :step].double() @ w[:, :step].double().T).float()
            close(parts[0], first, atol, what=f"first of {S} slices")
    assert ops.pack_weight(w[:N - 3].to(DEV)) is None and ops.pack_weight(w[:, :K - 8].to(DEV)) is None
    with pytest.raises(Exception, match="at most 16"):
        ops.gemm_packed(torch.zeros((17, K), dtype=BF16, device=DEV), wp, torch.empty((17, N), dtype=out_dtype, device=DEV))


@pytest.mark.parametrize("M,I,K", [(1, 16, 32), (1, 2560, 4096), (8, 2560, 4096), (7, 112, 992), (4, 16400, 64),
                                   (9, 2560, 4096), (13, 48, 992), (16, 12288, 512)])       # up to 16 rows: the engine's limit for this product
def test_gated_product_over_weights_in_fragment_order(ops, M, I, K):
    x, wg, wu = rnd((M, K), 28, BF16), rnd((I, K), 29, BF16), rnd((I, K), 30, BF16)
    wp = ops.pack_weight(ops.pair_rows(wg.to(DEV), wu.to(DEV)))
    out = torch.full((M, I), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_packed(x.to(DEV), wp, out, paired=True)
    g, u = x.double() @ wg.double().T, x.double() @ wu.double().T
    want = (g / (1 + torch.exp(-g)) * u).float()
    close(out, want, 2e-3 * K + 0.02, 1e-2, f"packed gated product {M}x{I}x{K}")


@pytest.mark.parametrize("gain_dtype,gain_offset", [(BF16, 0.0), (F32, 1.0)])
@pytest.mark.parametrize("M,H,K,N2", [(1, 64, 96, 48), (8, 4096, 4096, 6144), (5, 224, 1120, 80), (8, 4096, 12288, 24576),
                                      (3, 10240, 64, 32), (16, 96, 32, 16400)])
def test_norm_carried_between_two_products_over_packed_weights(ops, gain_dtype, gain_offset, M, H, K, N2):
    """The two halves of an RMSNorm between two products for few rows.  First half, as the epilogue of the product
    before it: resid += x . W^T, xs = gain * resid, ss = sums of resid^2 over groups of 16 columns.  Second half, as
    the epilogue of the product after it: sums of row m times rsqrt(sum(ss[m]) / H + eps), plain, gated, and in
    slices of K.  Together they equal the product over the normed rows."""
    eps = 1e-5
    x, w = rnd((M, K), 41, BF16), rnd((H, K), 42, BF16, 0.05)
    resid0 = rnd((M, H), 43)
    resid0[0] *= 30.0                    # rows of unequal size: a factor applied to the wrong row would show
    gain = (1 + 0.2 * rnd((H,), 44) - gain_offset).to(gain_dtype)
    wp = ops.pack_weight(w.to(DEV))
    resid = resid0.to(DEV)
    xs = torch.full((M, H), float("nan"), dtype=BF16, device=DEV)
    ss = torch.full((M, H // 16), float("nan"), dtype=F32, device=DEV)
    ops.gemm_packed(x.to(DEV), wp, None, resid_norm=(resid, gain.to(DEV), gain_offset, xs, ss))
    r = resid0.double() + x.double() @ w.double().T
    close(resid, r.float(), 1e-3 * math.sqrt(K) * 0.05 + 1e-5, 1e-6, "residual rows")
    r32 = resid.cpu()                    # what the kernel kept: the rest is computed from it
    g_all = gain_offset + gain.double()
    close(xs, (g_all * r32.double()).float(), 1e-6, 2 ** -8, "rows with the gain")
    close(ss, (r32.double() ** 2).view(M, H // 16, 16).sum(2).float(), 1e-6, 1e-5, "row statistic in groups")
    inv = torch.rsqrt((r32.double() ** 2).sum(1) / H + eps)[:, None]
    xs64 = xs.cpu().double()
    scale = (ss, H, eps)
    # plain product after the norm, bf16 and float, and in slices
    w2 = rnd((N2, H), 45, BF16, 0.05)
    wp2 = ops.pack_weight(w2.to(DEV))
    want = ((xs64 @ w2.double().T) * inv).float()
    atol = 2e-3 * float(want.abs().max()) + 1e-6
    out = torch.full((M, N2), float("nan"), dtype=F32, device=DEV)
    ops.gemm_packed(xs, wp2, out, row_scale=scale)
    close(out, want, atol, 1e-5, "product after the norm")
    parts = torch.full((3, M, N2), float("nan"), dtype=F32, device=DEV)
    ops.gemm_packed(xs, wp2, parts, row_scale=scale)
    close(parts.sum(0), want, atol, 1e-5, "product after the norm in slices")
    outb = torch.full((M, N2), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_packed(xs, wp2, outb, row_scale=scale)
    close(outb, want, atol, 2 ** -7, "product after the norm, bf16")
    # it equals the product over the normed rows up to the rounding of those rows
    normed = (g_all * r32.double() * inv).to(BF16)
    direct = (normed.double() @ w2.double().T).float()
    assert float((want - direct).abs().max()) <= 0.02 * float(direct.abs().max()) + 1e-6
    # gated product after the norm
    if N2 % 32 == 0:
        I = N2 // 2
        wg, wu = w2[:I], w2[I:]
        wpg = ops.pack_weight(ops.pair_rows(wg.to(DEV), wu.to(DEV)))
        outg = torch.full((M, I), float("nan"), dtype=BF16, device=DEV)
        ops.gemm_packed(xs, wpg, outg, paired=True, row_scale=scale)
        gg, uu = (xs64 @ wg.double().T) * inv, (xs64 @ wu.double().T) * inv
        wantg = (gg / (1 + torch.exp(-gg)) * uu).float()
        close(outg, wantg, 2e-3 * float(wantg.abs().max()) + 1e-6, 2 ** -7, "gated product after the norm")
    with pytest.raises(Exception, match="not gated"):
        ops.gemm_packed(x.to(DEV), wp, xs, resid_norm=(resid, gain.to(DEV), gain_offset, xs, ss))


def _sampled(M, N, n, seed):
    g = torch.Generator().manual_seed(seed)
    rows = torch.cat([torch.tensor([0, M - 1, 0, M - 1]), torch.randint(0, M, (n,), generator=g)])
    cols = torch.cat([torch.tensor([0, 0, N - 1, N - 1]), torch.randint(0, N, (n,), generator=g)])
    return rows, cols


def test_products_of_a_prompt_at_the_sizes_of_an_8b_layer(ops):
    """The large-tile products at full size: 2,048 rows through gate+up with the activation inside
    (24,576 paired rows, K = 4096), and through down_proj (N = 4096, K = 12288) in the two slices
    of K that the engine asks for; some hundred sampled outputs, the corners among them, against
    64-bit dot products."""
    M, H, I = 2048, 4096, 12288
    x = rnd((M, H), 70, BF16)
    wg, wu = rnd((I, H), 71, BF16, 0.02), rnd((I, H), 72, BF16, 0.02)
    out = torch.full((M, I), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_swiglu(x.to(DEV), ops.pair_rows(wg.to(DEV), wu.to(DEV)), out)
    rows, cols = _sampled(M, I, 400, 73)
    g = (x[rows].double() * wg[cols].double()).sum(1)
    u = (x[rows].double() * wu[cols].double()).sum(1)
    want = (g / (1 + torch.exp(-g)) * u).float()
    assert torch.isfinite(out).all()
    close(out[rows.to(DEV), cols.to(DEV)], want, 0.02, 1e-2, "gate+up at 8B sizes")
    del wg, wu
    assert ops.gemm_slices(M, H, I, BF16) == 2
    m = rnd((M, I), 74, BF16)
    wd = rnd((H, I), 75, BF16, 0.02)
    parts = torch.full((2, M, H), float("nan"), dtype=F32, device=DEV)
    ops.gemm(m.to(DEV), wd.to(DEV), parts)
    rows, cols = _sampled(M, H, 400, 76)
    want = (m[rows].double() * wd[cols].double()).sum(1).float()
    assert torch.isfinite(parts).all()
    close(parts.sum(0)[rows.to(DEV), cols.to(DEV)], want, 2e-3, 1e-4, "down_proj at 8B sizes, two slices")
    first = (m[rows, :I // 2].double() * wd[cols, :I // 2].double()).sum(1).float()
    close(parts[0][rows.to(DEV), cols.to(DEV)], first, 2e-3, 1e-4, "its first slice")
    # and the plain large product, bf16 out (q/k/v of a prompt: N = 6144)
    wq = rnd((6144, H), 77, BF16, 0.02)
    q = torch.full((M, 6144), float("nan"), dtype=BF16, device=DEV)
    ops.gemm(x.to(DEV), wq.to(DEV), q)
    rows, cols = _sampled(M, 6144, 400, 78)
    want = (x[rows].double() * wq[cols].double()).sum(1).float()
    close(q[rows.to(DEV), cols.to(DEV)], want, 0.02, 1e-2, "q/k/v at 8B sizes")


@pytest.mark.parametrize("M", [65, 80, 81, 128, 129, 145, 192, 208, 209, 256])
@pytest.mark.parametrize("N,K,packed", [(16, 128, True), (1008, 384, True), (8192, 256, True), (16384, 256, True), (333, 256, False)])
def test_products_of_65_to_256_rows_at_the_lines_of_their_tiles(ops, M, N, K, packed):
    """Both sides of the line between the 64 x 128 tiles and the streamed ones, ragged in both directions, W in fragment order and in
    plain rows: every value against 64 bits."""
    x, w = rnd((M, K), 86, BF16).to(DEV), rnd((N, K), 87, BF16).to(DEV)
    want = (x.double() @ w.double().T).float()
    for dt in (F32, BF16):
        out = torch.full((M, N), float("nan"), dtype=dt, device=DEV)
        ops.gemm(x, ops.pack_weight(w) if packed else w, out)
        # exact products, 32-bit sums of K terms of size one; bf16: half a unit in the last of 8 bits on top
        close(out, want, 1e-4 * math.sqrt(K), 0 if dt == F32 else 2 ** -8, f"{M}x{N}x{K}")


@pytest.mark.parametrize("M,N,K,S", [
    (129, 16, 128, 1), (300, 1040, 160 * 2, 1),              # fewer columns than a tile; the ring's shortest K
    (2305, 24592, 256, 1), (5000, 4112, 512, 1),             # several tiles a workgroup, ragged in both directions
    (700, 6144, 1024, 4), (1537, 2576, 1920, 3), (3000, 2064, 640, 2),   # slices, the last one shorter
    (1030, 777, 256, 1), (640, 1001, 512, 2)])               # plain rows, no multiple of 16: stored value by value
def test_streamed_tiles_run_on_into_the_next_tile(ops, M, N, K, S):
    """Products of many rows: a workgroup's loads run ahead into its next tile and into the next slice, the last tiles hang over
    M and N.  The sums are those of 64-bit dot products at places sampled over the output, and nothing is left unwritten."""
    x, w = rnd((M, K), 80, BF16), rnd((N, K), 81, BF16)
    wd = ops.pack_weight(w.to(DEV))
    wd = w.to(DEV) if wd is None else wd
    rows, cols = _sampled(M, N, 400, 82)
    step = ((K + S - 1) // S + 127) // 128 * 128
    for dt in ((F32,) if S > 1 else (F32, BF16)):
        out = torch.full((S, M, N) if S > 1 else (M, N), float("nan"), dtype=dt, device=DEV)
        ops.gemm(x.to(DEV), wd, out)
        assert torch.isfinite(out).all()
        for s in range(S):
            ks = slice(s * step, min(K, (s + 1) * step)) if S > 1 else slice(0, K)
            want = (x[rows, ks].double() * w[cols, ks].double()).sum(1).float()
            got = (out[s] if S > 1 else out)[rows.to(DEV), cols.to(DEV)]
            # exact products, 32-bit sums of K terms of size one; bf16: half a unit in the last of 8 bits on top
            close(got, want, 1e-3 * math.sqrt(K), 0 if dt == F32 else 2 ** -8, f"{M}x{N}x{K}, slice {s} of {S}")


PLAIN_TILES = (0, 1, 2, 8)          # the streamed tiles that also read W in plain rows


@pytest.mark.parametrize("kind", ["float", "bf16", "gated", "slices"])
@pytest.mark.parametrize("tile", range(10))
def test_every_streamed_tile(ops, tile, kind):
    """Each tile by its number, whatever the rules would take, with every output that it is compiled for: W in fragment order and
    (where compiled) in plain rows of a width that is no multiple of 16; ragged M and N, one tile and several tiles a workgroup, the
    shortest K that its ring allows, and slices whose last one is shorter.  Every value against 64 bits."""
    for M, N, K, S in ((70, 48, 256, 1), (1100, 2064, 256, 1), (5000, 4112, 256, 1), (300, 1040, 640, 2), (1300, 2576, 1024, 3)):
        if (kind == "slices") != (S > 1):
            continue
        if kind == "gated":
            N = (N + 31) // 32 * 32
        x, w = rnd((M, K), 88, BF16).to(DEV), rnd((N, K), 89, BF16).to(DEV)
        step = ((K + S - 1) // S + 127) // 128 * 128
        for packed in (True, False):
            if not packed and tile not in PLAIN_TILES:
                continue
            n = N if packed or kind == "gated" else N - 7
            wn = w[:n].contiguous()
            want = torch.stack([x[:, k:k + step].double() @ wn[:, k:k + step].double().T for k in range(0, K, step)])
            wk = ops.pack_weight(wn) if packed else wn
            tol = 1e-4 * math.sqrt(K)          # exact products, 32-bit sums of K terms of size one
            if kind == "gated":
                out = torch.full((M, N // 2), float("nan"), dtype=BF16, device=DEV)
                ops.gemm_swiglu(x, wk, out, tile=tile)
                z = want[0].view(M, N // 32, 2, 16)
                g, u = z[:, :, 0].reshape(M, -1), z[:, :, 1].reshape(M, -1)
                # (both factors carry the sums' error)
                off = (out.double() - g * torch.sigmoid(g) * u).abs() - 2 ** -8 * (g * torch.sigmoid(g) * u).abs() - tol * (g.abs() + u.abs() + 1)
            else:
                dt = BF16 if kind == "bf16" else F32
                out = torch.full((S, M, n) if S > 1 else (M, n), float("nan"), dtype=dt, device=DEV)
                ops.gemm(x, wk, out, tile=tile)
                off = (out.double().view(want.shape) - want).abs() - (2 ** -8 if dt == BF16 else 0) * want.abs() - tol
            assert torch.isfinite(out).all() and float(off.max()) <= 0, (M, N, K, S, packed, float(off.max()))


def test_there_are_ten_streamed_tiles_and_they_refuse_what_they_do_not_take(ops):
    from synaptix_amd.kernels.ops import KernelError
    x, w, out = (torch.zeros(s, dtype=BF16, device=DEV) for s in ((70, 256), (48, 256), (70, 48)))
    packed = ops.pack_weight(w)
    for tile, weight in [(10, packed), (11, packed)] + [(t, w) for t in range(10) if t not in PLAIN_TILES]:
        with pytest.raises(KernelError):
            ops.gemm(x, weight, out, tile=tile)
    with pytest.raises(KernelError):      # a ring of eight k-tiles needs a K of 256
        ops.gemm(x[:, :128].contiguous(), w[:, :128].contiguous(), out, tile=8)
    with pytest.raises(KernelError):
        ops.gemm(x.float(), w.float(), out.float(), tile=0)


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("N,K", [(800, 192), (24576, 256), (28672, 256), (32800, 256)])
@pytest.mark.parametrize("M", [128, 129, 192, 193, 256, 257])
def test_gated_products_of_129_to_256_rows(ops, M, N, K, packed):
    """At the lines between the streamed tiles and those that hold all rows of x, which go round once or not at all (N = 32,800), W in
    fragment order and in plain rows: every value against 64 bits."""
    x, w = rnd((M, K), 92, BF16).to(DEV), rnd((N, K), 93, BF16).to(DEV)
    if packed and K % 128:
        pytest.skip("in fragment order K is a multiple of 128")
    out = torch.full((M, N // 2), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_swiglu(x, ops.pack_weight(w) if packed else w, out)
    z = (x.double() @ w.double().T).view(M, N // 32, 2, 16)
    g, u = z[:, :, 0].reshape(M, -1), z[:, :, 1].reshape(M, -1)
    want = g * torch.sigmoid(g) * u
    # the sums are off by at most 1e-4 sqrt(K) (products exact, 32-bit sums of K terms of size one), and both factors carry that; one rounding
    off = (out.double() - want).abs() - 2 ** -8 * want.abs() - 1e-4 * math.sqrt(K) * (g.abs() + u.abs() + 1)
    assert torch.isfinite(out).all() and float(off.max()) <= 0, float(off.max())


@pytest.mark.parametrize("kind", ["gated", "slices"])
@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("K", [128, 192, 256, 512, 1152])
def test_products_where_the_streamed_tiles_begin(ops, K, packed, kind):
    """On both sides of the row counts and widths from which the streamed tiles are taken, and of a tile of rows (up to which W's loads
    are marked non-temporal), every value against 64 bits; nothing is left unwritten."""
    if packed and K % 128:
        pytest.skip("in fragment order K is a multiple of 128")
    for M, S in itertools.product((16, 17, 49, 64, 65, 129), (1,)) if kind == "gated" else itertools.product((56, 57, 64, 65, 128, 129), (1, 2, 4)):
        N = 800
        if S > 1 and K % (S * 128):
            continue
        x, w = rnd((M, K), 94, BF16).to(DEV), rnd((N, K), 95, BF16).to(DEV)
        weight = ops.pack_weight(w) if packed else w
        if kind == "gated":
            out = torch.full((M, N // 2), float("nan"), dtype=BF16, device=DEV)
            ops.gemm_swiglu(x, weight, out)
            z = (x.double() @ w.double().T).view(M, N // 32, 2, 16)
            g, u = z[:, :, 0].reshape(M, -1), z[:, :, 1].reshape(M, -1)
            want, room = g * torch.sigmoid(g) * u, 1e-4 * math.sqrt(K) * (g.abs() + u.abs() + 1)      # as above
            off = (out.double() - want).abs() - 2 ** -8 * want.abs() - room
        else:
            out = torch.full((S, M, N), float("nan"), dtype=F32, device=DEV)
            ops.gemm(x, weight, out if S > 1 else out[0])
            off = (out.double().sum(0) - x.double() @ w.double().T).abs() - 1e-4 * math.sqrt(K)
        assert torch.isfinite(out).all() and float(off.max()) <= 0, (M, S, float(off.max()))


@pytest.mark.parametrize("N,K", [(3072, 8192), (5120, 8192), (4096, 4096)])
@pytest.mark.parametrize("M", [57, 64, 65, 97, 128, 129, 177, 256])
def test_products_in_the_slices_of_their_tiles(ops, M, N, K):
    """57 to 256 rows in the slices that the rules pick, through the tiles that load straight into LDS and through the streamed ones."""
    x, w = rnd((M, K), 96, BF16).to(DEV), rnd((N, K), 97, BF16).to(DEV)
    S = ops.gemm_slices(M, N, K, BF16)
    assert S > 1
    want = x.double() @ w.double().T
    for weight in (w, ops.pack_weight(w)):
        out = torch.full((S, M, N), float("nan"), dtype=F32, device=DEV)
        ops.gemm(x, weight, out)
        off = (out.double().sum(0) - want).abs() - 1e-4 * math.sqrt(K)
        assert torch.isfinite(out).all() and float(off.max()) <= 0, float(off.max())


@pytest.mark.parametrize("M", [17, 32, 33, 64, 65, 128, 129, 192, 193, 256])
@pytest.mark.parametrize("N,K", [(18528, 2112), (18528, 2048), (4096, 2048), (768, 4096)])
def test_gated_and_uncut_products_over_plain_rows(ops, M, N, K):
    """17 to 256 rows over W in plain rows, through the tiles that load straight into LDS and through the streamed ones."""
    x, w = rnd((M, K), 98, BF16).to(DEV), rnd((N, K), 99, BF16).to(DEV)
    z = x.double() @ w.double().T
    out, gated = torch.full((M, N), float("nan"), dtype=F32, device=DEV), torch.full((M, N // 2), float("nan"), dtype=BF16, device=DEV)
    ops.gemm(x, w, out)
    assert torch.isfinite(out).all() and float((out.double() - z).abs().max()) <= 1e-4 * math.sqrt(K)
    ops.gemm_swiglu(x, w, gated)
    z = z.view(M, N // 32, 2, 16)
    g, u = z[:, :, 0].reshape(M, -1), z[:, :, 1].reshape(M, -1)
    want, room = g * torch.sigmoid(g) * u, 1e-4 * math.sqrt(K) * (g.abs() + u.abs() + 1)
    off = (gated.double() - want).abs() - 2 ** -8 * want.abs() - room
    assert torch.isfinite(gated).all() and float(off.max()) <= 0, float(off.max())
    if K % 128 == 0:          # the bits do not depend on how W lies
        packed = ops.pack_weight(w)
        again, gated2 = torch.empty_like(out), torch.empty_like(gated)
        ops.gemm(x, packed, again)
        ops.gemm_swiglu(x, packed, gated2)
        assert torch.equal(again, out) and torch.equal(gated2, gated)


@pytest.mark.parametrize("act", ["silu", "gelu_tanh", ("swiglu_limit", 7.0)])
@pytest.mark.parametrize("M,I,K", [(300, 1200, 256), (2100, 4112, 512)])
def test_gated_activations_of_many_rows(ops, act, M, I, K):
    """Every gated activation as the epilogue of the tiles for many rows, at inputs from nothing to far beyond where the
    sigmoid is one or zero, against 64 bits: one rounding to bf16 (2^-8 of the value) and the 32-bit sums' own error."""
    x, wg, wu = rnd((M, K), 83, BF16), rnd((I, K), 84, BF16, 0.5), rnd((I, K), 85, BF16, 0.5)
    out = torch.full((M, I), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_swiglu(x.to(DEV), ops.pack_weight(ops.pair_rows(wg.to(DEV), wu.to(DEV))), out, act)
    assert torch.isfinite(out).all()
    rows, cols = _sampled(M, I, 600, 86)
    g, u = ((x[rows].double() * m[cols].double()).sum(1) for m in (wg, wu))
    if act == "silu":
        want = g * torch.sigmoid(g) * u
    elif act == "gelu_tanh":
        want = 0.5 * g * (1 + torch.tanh(math.sqrt(2 / math.pi) * (g + 0.044715 * g ** 3))) * u
    else:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    # the sums are off by at most about K^(1/2) 2^-24 times their terms' size; both factors carry that error
    close(out[rows.to(DEV), cols.to(DEV)], want.float(), 1e-4 * math.sqrt(K), 2 ** -8 + 1e-4, f"{act} {M}x{I}x{K}")


@pytest.mark.parametrize("out_dtype", [F32, BF16])
@pytest.mark.parametrize("act", ["silu", "gelu_tanh", ("swiglu_limit", 7.0)])
def test_gated_epilogue_of_streamed_tiles_is_no_less_exact(ops, act, out_dtype):
    """The epilogue that the streamed tiles make of the hardware's base-2 functions, against 64 bits and beside the
    library functions of the plain kernel, on the same sums: rows of x hold a 1 and a power of two, so the sums
    are exact, gates from -120 to 120 (beyond e^88, where the library's exponential overflows) and from -3 to 3, and infinities."""
    K, J, P = 256, 1024, 512
    g = torch.Generator().manual_seed(7)
    x = torch.zeros(P, K)
    x[torch.arange(P), torch.arange(P) % K] = 1.0
    x[torch.arange(P), (torch.arange(P) * 7 + 3) % K] = 2.0 ** -9
    w = torch.empty(1, J, K)
    w[0, 0::2] = torch.where(torch.rand(J // 2, 1, generator=g) < 0.5, 240 * torch.rand(J // 2, K, generator=g) - 120,
                             6 * torch.rand(J // 2, K, generator=g) - 3)
    w[0, 1::2] = torch.randn(J // 2, K, generator=g)
    x, w = x.to(BF16), ((64 * w).round() / 64).to(BF16)
    z = x.double() @ w[0].double().T
    gt, up = z[:, 0::2], z[:, 1::2]
    assert torch.equal(z.float().double(), z)
    if act == "silu":
        want = gt * torch.sigmoid(gt) * up
    elif act == "gelu_tanh":
        t = 2 * math.sqrt(2 / math.pi) * (gt + 0.044715 * gt ** 3)
        want = gt * torch.sigmoid(t) * up
    else:
        gl, ul = gt.clamp(max=7.0), up.clamp(-7.0, 7.0)
        want = gl * torch.sigmoid(1.702 * gl) * (ul + 1)
    d = lambda t: t.to(DEV)
    ids = torch.arange(P, dtype=I32, device=DEV)
    seg = torch.tensor([0, P], dtype=I32, device=DEV)
    outs = []
    for plain in (False, True):
        out = torch.full((P, J // 2), float("nan"), dtype=out_dtype, device=DEV)
        ops.experts_product(d(x), d(w) if plain else ops.pack_expert_weights(d(w)), out, seg, ids, ids, gated=act, force_simt=plain)
        outs.append(out.cpu().double())
    # (results below the smallest normal number, and where the plain kernel's overflow gave nothing, tell nothing about rounding)
    tell = (want.abs() > 1e-30) & (outs[1] != 0)
    off = [((o - want).abs() / want.abs())[tell] for o in outs]
    assert float(tell.float().mean()) > 0.7
    if out_dtype == F32:
        assert float(off[0].max()) <= float(off[1].max()) and float(off[0].norm()) <= float(off[1].norm()), [float(o.max()) * 2 ** 24 for o in off]
    else:
        # half a unit in the last of 8 bits, and what a few ulp of 32 bits (|t| of them in 1.702 t, which both round) can add where that is a tie
        assert float(off[0].max()) <= 2 ** -8 * (1 + 2 ** -8) and float(off[0].norm()) <= float(off[1].norm()) * (1 + 1e-5)
    assert ((outs[0] - want).abs() <= (outs[1] - want).abs() + (1e-29 if out_dtype == F32 else 1e-29 + 2 ** -8 * want.abs()))[~tell].all()
    # infinite sums: what the plain kernel makes of them
    w[0, 0, :], w[0, 2, :] = float("inf"), -float("inf")
    a, b = torch.empty(P, J // 2, device=DEV), torch.empty(P, J // 2, device=DEV)
    one = torch.ones(P, K, dtype=BF16, device=DEV)
    ops.experts_product(one, ops.pack_expert_weights(d(w)), a, seg, ids, ids, gated=act)
    ops.experts_product(one, d(w), b, seg, ids, ids, gated=act, force_simt=True)
    assert torch.equal(torch.nan_to_num(a[:, :2]), torch.nan_to_num(b[:, :2])) and torch.equal(a[:, :2].isnan(), b[:, :2].isnan())


@pytest.mark.parametrize("counts,J,K", [([0, 1, 63, 64, 129, 300, 0, 43], 544, 320), ([48], 32, 256), ([600, 0, 5], 256, 512),
                                        ([130] * 70, 288, 256), ([257, 225, 31, 256], 544, 320), ([50] * 300, 288, 256)])
@pytest.mark.parametrize("act,gated,out_dtype", [(None, None, F32), ("gelu", None, BF16), ("gelu", None, F32), ("relu_squared", None, BF16),
                                                 (None, "silu", BF16), (None, ("swiglu_limit", 7.0), F32), (None, "gelu_tanh", BF16)])
def test_streamed_experts(ops, counts, J, K, act, gated, out_dtype):
    """Rows of many experts through the streamed tiles: experts without rows, with one, at the edges of a tile and over several
    tiles, a last round in halves of tiles; gathered rows, scattered results with weights, every epilogue; places of out that no row names stay as they were."""
    E, P = len(counts), sum(counts)
    g = torch.Generator().manual_seed(J + K)
    x, w = rnd((P + 9, K), 90, BF16), rnd((E, J, K), 91, BF16, 0.3)
    seg = torch.tensor([0] + counts).cumsum(0).to(I32)
    a_rows = torch.randint(0, P + 9, (P,), generator=g).to(I32)
    o_rows = torch.randperm(P + 5, generator=g)[:P].to(I32)
    weight = torch.rand(P, generator=g) + 0.5
    Jo = J // 2 if gated else J
    out = torch.full((P + 5, Jo), 7.0, dtype=out_dtype, device=DEV)
    d = lambda t: t.to(DEV)
    packed = ops.pack_expert_weights(d(w))
    assert packed is not None
    ops.experts_product(d(x), packed, out, d(seg), d(a_rows), d(o_rows), row_weight=d(weight), act=act, gated=gated)
    want = torch.full((P + 5, Jo), 7.0, dtype=torch.float64)
    for e in range(E):
        rows = slice(int(seg[e]), int(seg[e + 1]))
        z = x[a_rows[rows].long()].double() @ w[e].double().T
        if gated:
            gt, up = z[:, 0::2], z[:, 1::2]
            if gated == "silu":
                z = gt * torch.sigmoid(gt) * up
            elif gated == "gelu_tanh":
                z = torch.nn.functional.gelu(gt, approximate="tanh") * up
            else:
                gt, up = gt.clamp(max=7.0), up.clamp(-7.0, 7.0)
                z = gt * torch.sigmoid(1.702 * gt) * (up + 1)
        elif act == "gelu":
            z = torch.nn.functional.gelu(z)
        elif act == "relu_squared":
            z = torch.relu(z) ** 2
        want[o_rows[rows].long()] = z * weight[rows, None].double()
    # 32-bit sums of K products; a square and a gate carry their inputs' error as a share of the result; bf16 rounds by 2^-9
    close(out, want.float(), 2e-4 * math.sqrt(K), 1e-4 if out_dtype == F32 else 2 ** -8 + 1e-4, f"{counts} {J} x {K} {act} {gated}")


@pytest.mark.parametrize("counts", [[60, 70, 64], [300, 250]])       # the lower tile; plain loads of W
@pytest.mark.parametrize("out_dtype", [BF16, F32])
@pytest.mark.parametrize("gated", ["silu", ("swiglu_limit", 7.0), "gelu_tanh", None])
def test_streamed_experts_of_every_gate(ops, counts, gated, out_dtype):
    test_streamed_experts(ops, counts, 288, 320, None, gated, out_dtype)


def test_slices_fill_the_compute_units(ops):
    """The host-side rule for the products over packed weights: one slice where the workgroups fill their
    rounds, more where they would leave the last round half empty."""
    assert ops.packed_slices(4096, 4096) == 1 and ops.packed_slices(151936, 4096) == 1
    assert ops.packed_slices(5120, 25600) == 3 and ops.packed_slices(6144, 4096) == 2
    assert ops.packed_slices(2560, 4096) == 3
    assert ops.packed_slices(2560, 1024) == 1          # no slice shorter than 1,024
    for N in range(16, 12000, 16):
        s = ops.packed_slices(N, 8192)
        assert 1 <= s <= 8


@pytest.mark.parametrize("M,N,K,S", [
    (9, 48, 128, 1), (16, 4096, 4096, 1), (33, 208, 256, 1), (64, 6144, 4096, 1), (64, 144, 384, 3),
    (100, 4112, 384, 1), (128, 208, 4096, 8), (130, 6144, 1024, 1), (200, 4096, 1024, 2), (256, 1008, 2560, 4),
    (257, 528, 4096, 8), (300, 96, 128, 1), (512, 4096, 1024, 2), (700, 272, 640, 1),
    (1700, 5120, 128, 1),               # several tiles a workgroup, the shortest K of the streamed tiles
    (2053, 528, 256, 1), (1000, 12304, 128, 1), (2048, 6144, 512, 1),   # the large tiles, ragged edges
    (8, 70000 // 16 * 16, 256, 1), (20, 66000 // 16 * 16, 128, 1),      # few rows, very wide
    (40, 80, 96, 1), (300, 48, 160, 1),                                   # K no multiple of 128: in blocks of 16 rows
])
def test_tiled_gemm_reads_weights_in_fragment_order(ops, M, N, K, S):
    """The tiles for 9 rows and more over pack_weight(W): the same sums in the same order as over plain rows
    (bit for bit where both run the same tile), for every tile shape, with ragged edges in M and N, and as
    partial sums over slices of K."""
    x, w = rnd((M, K), 16, BF16), rnd((N, K), 17, BF16)
    wd = w.to(DEV)
    wp = ops.pack_weight(wd)
    assert wp is not None
    want = (x.double() @ w.double().T).float()
    atol = 1e-3 * math.sqrt(K)
    for out_dtype in ((F32,) if S > 1 else (BF16, F32)):
        shape = (S, M, N) if S > 1 else (M, N)
        got = torch.full(shape, float("nan"), dtype=out_dtype, device=DEV)
        ops.gemm(x.to(DEV), wp, got)
        total = got.float().sum(0) if S > 1 else got
        close(total, want, atol if out_dtype == F32 else atol + 0.02, 0 if out_dtype == F32 else 1e-2,
              f"gemm over fragment order {M}x{N}x{K}")
        if K % 128 == 0 and not (N >= 65536 and K % 256):   # (very wide and K no multiple of 256: plain rows take another tile)
            plain = torch.full(shape, float("nan"), dtype=out_dtype, device=DEV)
            ops.gemm(x.to(DEV), wd, plain)
            assert torch.equal(plain, got), "the same tiles over both layouts must give the same bits"


@pytest.mark.parametrize("M,I,K", [(9, 48, 128), (16, 2560, 4096), (33, 80, 128), (64, 1024, 512), (100, 176, 384),
                                   (128, 12288, 4096), (192, 1040, 256), (256, 2560, 1024), (300, 112, 128),
                                   (1000, 6160, 256), (2048, 1024, 512), (20, 40000, 128), (40, 48, 96)])
def test_tiled_gated_gemm_reads_weights_in_fragment_order(ops, M, I, K):
    x = rnd((M, K), 18, BF16)
    wg, wu = rnd((I, K), 19, BF16, 0.5), rnd((I, K), 20, BF16, 0.5)
    paired = ops.pair_rows(wg.to(DEV), wu.to(DEV))
    wp = ops.pack_weight(paired)
    g = x.double() @ wg.double().T
    want = (g / (1 + torch.exp(-g)) * (x.double() @ wu.double().T)).float()
    got = torch.full((M, I), float("nan"), dtype=BF16, device=DEV)
    ops.gemm_swiglu(x.to(DEV), wp, got)
    close(got, want, 0.03 + 2e-3 * math.sqrt(K), 2e-2, f"gated gemm over fragment order {M}x{I}x{K}")
    if K % 128 == 0 and 2 * I < 65536:
        plain = torch.empty((M, I), dtype=BF16, device=DEV)
        ops.gemm_swiglu(x.to(DEV), paired, plain)
        assert torch.equal(plain, got)


def test_embedding_from_a_table_in_fragment_order(ops):
    V, H = 1008, 4128
    table = rnd((V, H), 21, BF16)
    ids = torch.tensor([0, 15, 16, 17, V - 1, 500, 31], dtype=I32)
    out = torch.full((ids.numel(), H), float("nan"), dtype=F32, device=DEV)
    ops.embed(ops.pack_weight(table.to(DEV)), ids.to(DEV), out)
    assert torch.equal(out.cpu(), table[ids.long()].to(F32))


def test_gemm_bf16_paths_agree(ops):
    """The MFMA kernels and the plain kernel compute the same sums."""
    for M in (4, 40, 300):
        x, w = rnd((M, 256), 12, BF16).to(DEV), rnd((96, 256), 13, BF16).to(DEV)
        a = torch.empty((M, 96), dtype=F32, device=DEV)
        b = torch.empty((M, 96), dtype=F32, device=DEV)
        ops.gemm(x, w, a)
        ops.gemm(x, w, b, force_simt=True)
        close(a, b, 2e-4, what=f"mfma vs plain, M={M}")


# ----------------------------------------------------------------------------- cache write + attention

def dv(v):
    """V pages as plain (dim, token) rows on the CPU -> on the device in the kernels' own order."""
    from synaptix_amd.kernels import ops as real_ops
    return real_ops.v_pages_to_kernel_order(v).to(DEV)


def hv(v):
    """V pages from the device back to plain (dim, token) rows on the CPU."""
    from synaptix_amd.kernels import ops as real_ops
    return real_ops.v_pages_from_kernel_order(v.cpu())


def make_cache(n_pages, nkv, hd, dtype, seed, fill="garbage"):
    """Pages filled with large values: whatever a kernel reads beyond a sequence's end shows."""
    k = rnd((n_pages, nkv, 64, hd), seed, dtype, 50.0)
    v = rnd((n_pages, nkv, hd, 64), seed + 1, dtype, 50.0)
    if fill == "nan":
        k[:], v[:] = float("nan"), float("nan")
    return k, v


def step_arrays(past, new):
    tok_seq, tok_pos, starts = [], [], [0]
    for i, (p, n) in enumerate(zip(past, new)):
        tok_seq += [i] * n
        tok_pos += list(range(p, p + n))
        starts.append(starts[-1] + n)
    t = lambda a: torch.tensor(a, dtype=I32)
    return t(tok_seq), t(tok_pos), t(starts), t(past), t([p + n for p, n in zip(past, new)])


def shuffled_table(n_seqs, width, seed):
    """Each sequence's pages lie scattered over the pool."""
    g = torch.Generator().manual_seed(seed)
    perm = torch.randperm(n_seqs * width, generator=g).to(I32)
    return perm.view(n_seqs, width).contiguous()


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("nh,nkv,hd,rot,norm", [(4, 2, 16, 16, True), (6, 3, 48, 32, True), (8, 1, 128, 128, False),
                                                (3, 3, 80, 0, True)])
def test_qk_norm_rope_kv_write(ops, dtype, nh, nkv, hd, rot, norm):
    past, new = [3, 70, 0], [5, 1, 66]
    tok_seq, tok_pos, _, _, _ = step_arrays(past, new)
    N = len(tok_seq)
    table = shuffled_table(3, 3, 1)
    qkv = rnd((N, (nh + 2 * nkv) * hd), 20, dtype)
    qg = (1 + 0.1 * rnd((hd,), 21)).to(dtype) if norm else None
    kg = (1 + 0.1 * rnd((hd,), 22)).to(dtype) if norm else None
    cos = sin = None
    if rot:
        ang = torch.arange(200, dtype=F32)[:, None] * (10000.0 ** (-torch.arange(rot // 2, dtype=F32) * 2 / rot))[None]
        cos, sin = torch.cos(ang), torch.sin(ang)
    k0, v0 = make_cache(9, nkv, hd, dtype, 23)
    kw, vw, qw = k0.clone(), v0.clone(), torch.empty((N, nh * hd), dtype=dtype)
    ref.qk_norm_rope_kv_write(qkv, qw, kw, vw, table, tok_seq, tok_pos, qg, kg, 1e-5, cos, sin, nh, nkv, hd)
    d = lambda t: None if t is None else t.to(DEV)
    kd, vd, qd = k0.to(DEV), dv(v0), torch.empty((N, nh * hd), dtype=dtype, device=DEV)
    ops.qk_norm_rope_kv_write(d(qkv), qd, kd, vd, d(table), d(tok_seq), d(tok_pos), d(qg), d(kg), 1e-5, d(cos), d(sin),
                              nh, nkv, hd)
    tol = dict(atol=1e-5, rtol=1e-5) if dtype == F32 else dict(atol=3e-2, rtol=1e-2)
    close(qd, qw, what="q", **tol)
    close(kd, kw, what="k pages", **tol)
    assert torch.equal(hv(vd), vw), "v is a copy"
    # untouched places of the pages stay as they were
    untouched = (kw == k0)
    assert torch.equal(kd.cpu()[untouched], k0[untouched])
    # the same from float partial sums [S, N, width] (a product cut along K): they are added first
    if dtype == BF16:
        parts = rnd((3, N, (nh + 2 * nkv) * hd), 24)
        parts[2] = qkv.float() - parts[0] - parts[1]
        kd3, vd3, qd3 = k0.to(DEV), dv(v0), torch.empty((N, nh * hd), dtype=dtype, device=DEV)
        ops.qk_norm_rope_kv_write(d(parts), qd3, kd3, vd3, d(table), d(tok_seq), d(tok_pos), d(qg), d(kg), 1e-5, d(cos),
                                  d(sin), nh, nkv, hd)
        close(qd3, qw, what="q from partial sums", **tol)
        close(kd3, kw, what="k pages from partial sums", **tol)
        close(hv(vd3), vw, 2e-2, 1e-2, what="v pages from partial sums")
    # a reader of another layer's cache writes nothing
    kd2, vd2 = k0.to(DEV), dv(v0)
    ops.qk_norm_rope_kv_write(d(qkv), qd, kd2, vd2, d(table), d(tok_seq), d(tok_pos), d(qg), d(kg), 1e-5, d(cos), d(sin),
                              nh, nkv, hd, write_kv=False)
    assert torch.equal(kd2.cpu(), k0) and torch.equal(hv(vd2), v0)
    close(qd, qw, what="q without cache write", **tol)


@pytest.mark.parametrize("parts", [0, 2, 3, 4, 5])
def test_prompt_intake_has_the_same_bits_with_one_and_four_tokens_a_lane(ops, parts):
    """2,801 tokens at once (four tokens a lane, but for two parts) and in pieces of 401, 100 and 37 (one a lane, or up to 64 tokens in more
    than four parts a wave a head, which adds a head's squares in another order): the same q, keys and values."""
    nh, nkv, hd, N = 40, 8, 128, 2801
    g = torch.Generator(device=DEV).manual_seed(3)
    rows = torch.randn(((parts,) if parts else ()) + (N, (nh + 2 * nkv) * hd), generator=g, device=DEV)
    rows = rows if parts else rows.to(BF16)
    gain = (1 + 0.1 * rnd((hd,), 22)).to(BF16).to(DEV)
    cos, sin = torch.randn(3000, hd // 2, generator=g, device=DEV), torch.randn(3000, hd // 2, generator=g, device=DEV)
    pages = (N + 63) // 64
    table = torch.randperm(pages, generator=torch.Generator().manual_seed(1)).to(I32)[None].to(DEV)
    pos, seq = torch.arange(N, dtype=I32, device=DEV), torch.zeros(N, dtype=I32, device=DEV)

    def run(piece):
        q = torch.full((N, nh * hd), float("nan"), dtype=BF16, device=DEV)
        k, v = torch.zeros((pages, nkv, 64, hd), dtype=BF16, device=DEV), torch.zeros((pages, nkv, hd, 64), dtype=BF16, device=DEV)
        for a in range(0, N, piece):
            ops.qk_norm_rope_kv_write(rows[..., a:a + piece, :].contiguous(), q[a:a + piece], k, v, table, seq[a:a + piece], pos[a:a + piece], gain, gain,
                                      1e-5, cos, sin, nh, nkv, hd)
        return q, k, v
    whole = run(N)
    assert not bool(torch.isnan(whole[0]).any())
    for piece in (401, 100, 37):
        got = run(piece)
        assert torch.equal(got[2], whole[2]), piece
        for a, b in zip(got[:2], whole[:2]):
            if parts > 4 and piece <= 64:
                # another order of 128 squares moves a head's factor by 2^-20 at most, so a value by that of the two products it is the
                # difference of (below 16 each), and to the next number of 16 bits (2^-7 of it at most)
                close(a, b, 2.0 ** -15, 2.0 ** -7, "q and k in more than four parts")
            else:
                assert torch.equal(a, b), piece


@pytest.mark.parametrize("nh,nkv,hd", [(1, 1, 16), (5, 3, 64), (8, 2, 128), (2, 3, 256), (40, 8, 128)])
@pytest.mark.parametrize("step", ["one", "eight", "ragged", "singles", "gaps", "long"])
def test_values_of_a_prompt_step_in_pieces_of_eight(ops, step, nh, nkv, hd):
    """Sequences that begin and end anywhere among the eight tokens of a wave and among the eight positions of a piece, single tokens
    between them, positions that do not follow each other: the values are copied, in place, and nothing else is written; keys and
    queries as by the twin."""
    past, new = {"one": ([13], [1]), "eight": ([56], [8]), "ragged": ([8, 0, 61, 5, 17], [9, 8, 30, 3, 26]), "singles": ([7, 8, 0, 30], [1, 1, 1, 1]),
                 "gaps": ([0, 3], [40, 30]), "long": ([1, 0], [70, 135])}[step]
    tok_seq, tok_pos, _, _, _ = step_arrays(past, new)
    if step == "gaps":      # every third place from the 12th on is left out, and the last tokens run backwards
        tok_pos = torch.tensor([p if i < 12 else p + i // 3 for i, p in enumerate(tok_pos.tolist())], dtype=I32)
        tok_pos[-9:] = tok_pos[-9:].flip(0)
    N, table = len(tok_seq), shuffled_table(5, 3, 3)
    qkv = rnd((N, (nh + 2 * nkv) * hd), 25, BF16)
    qg, kg = ((1 + 0.1 * rnd((hd,), 26 + i)).to(BF16) for i in range(2))
    ang = torch.arange(200, dtype=F32)[:, None] * (10000.0 ** (-torch.arange(hd // 2, dtype=F32) * 2 / hd))[None]
    cos, sin = torch.cos(ang), torch.sin(ang)
    k0, v0 = make_cache(15, nkv, hd, BF16, 28)
    kw, vw, qw = k0.clone(), v0.clone(), torch.empty((N, nh * hd), dtype=BF16)
    ref.qk_norm_rope_kv_write(qkv, qw, kw, vw, table, tok_seq, tok_pos, qg, kg, 1e-5, cos, sin, nh, nkv, hd)
    d = lambda t: t.to(DEV)
    # (as whole rows, and as partial sums of which all but one are zero: 65 tokens and more take the same kernel)
    for rows in (qkv, torch.stack([torch.zeros_like(qkv.float()), qkv.float()])):
        kd, vd, qd = d(k0), dv(v0), torch.empty((N, nh * hd), dtype=BF16, device=DEV)
        ops.qk_norm_rope_kv_write(d(rows), qd, kd, vd, d(table), d(tok_seq), d(tok_pos), d(qg), d(kg), 1e-5, d(cos), d(sin), nh, nkv, hd)
        assert torch.equal(hv(vd), vw), "v is a copy"
        close(qd, qw, 3e-2, 1e-2, what="q")
        close(kd, kw, 3e-2, 1e-2, what="k pages")
        assert torch.equal(kd.cpu()[kw == k0], k0[kw == k0])


def fill_sequences(k, v, table, lens, nkv, hd, dtype, seed):
    """Write O(1) keys and values for positions below each length; the rest stays garbage."""
    for b, T in enumerate(lens):
        kk = rnd((T, nkv, hd), seed + 10 * b, dtype)
        vv = rnd((T, nkv, hd), seed + 10 * b + 1, dtype)
        for t in range(T):
            page = int(table[b, t // 64])
            k[page, :, t % 64, :] = kk[t]
            v[page, :, :, t % 64] = vv[t]


ATTN_SHAPES = [
    # nh, nkv, hd, past, new, window
    (4, 2, 16, [0, 0, 0], [5, 17, 70], 0),
    (8, 1, 32, [0, 100, 63], [130, 1, 2], 0),
    (6, 3, 48, [10, 0], [40, 200], 0),
    (8, 2, 64, [600, 0], [1, 8], 0),            # the reference's decode shape (2,8,2,1,600,64) beside a short one
    (32, 8, 128, [0], [300], 0),
    (4, 4, 128, [0, 40], [33, 1], 0),
    (4, 2, 96, [0, 5], [150, 100], 37),          # a window that ends inside pages
    (5, 5, 16, [200], [1], 64),
    (8, 2, 64, [100, 64, 127], [70, 64, 2], 0),   # chunks of a prompt that start inside a page, at its edge, before its end
    (32, 8, 128, [100, 1000], [150, 130], 0),     # the same at the head size and group of the large models
    (6, 2, 48, [33], [300], 50),                  # a chunk over several pages with a window
    (8, 4, 64, [5, 0, 190], [260, 129, 3], 70),   # head size 64 with a window, sequences that end inside pages
    (16, 2, 128, [0, 77], [513, 200], 0),         # eight heads a group, several tiles of 128 rows
    (32, 8, 128, [5, 190], [260, 131], 70),       # the head size of the large models with a window whose edge lies inside pages
]


@pytest.mark.parametrize("dtype", [F32, BF16])
@pytest.mark.parametrize("nh,nkv,hd,past,new,window", ATTN_SHAPES)
def test_attention_prefill(ops, dtype, nh, nkv, hd, past, new, window):
    B = len(past)
    lens = [p + n for p, n in zip(past, new)]
    width = max((T + 63) // 64 for T in lens) + 1
    table = shuffled_table(B, width, 3)
    # what lies in the pages behind a sequence's end is NaN for the head sizes of the kernel with 32 query rows a
    # wave (and finite garbage elsewhere): a value that leaked from there, times a weight of zero, would show
    k, v = make_cache(B * width, nkv, hd, dtype, 30, fill="nan" if (hd in (64, 128) and dtype == BF16) else "garbage")
    fill_sequences(k, v, table, lens, nkv, hd, dtype, 31)
    tok_seq, tok_pos, starts, past_t, len_t = step_arrays(past, new)
    N = len(tok_seq)
    q = rnd((N, nh * hd), 32, dtype)
    scale = 1 / math.sqrt(hd)
    want = torch.empty((N, nh * hd), dtype=F32)
    ref.attention_f32(q.float(), torch.nan_to_num(k.float()), torch.nan_to_num(v.float()), table, tok_seq, tok_pos, want,
                      scale, window, nh, nkv, hd)
    d = lambda t: t.to(DEV)
    out = torch.empty((N, nh * hd), dtype=dtype, device=DEV)
    if dtype == F32:
        ops.attention_f32(d(q), d(k), dv(v), d(table), d(tok_seq), d(tok_pos), out, scale, window, nh, nkv, hd)
        close(out, want, 1e-4, what="attention f32")
    else:
        ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(starts), d(past_t), out, scale, window, nh, nkv, hd)
        close(out, want, 2e-2, 1e-2, what="attention prefill bf16")
        # both kernels where the head size allows both: waves of 16 and of 32 query rows
        for variant in (1, 2):
            out.fill_(float("nan"))
            if variant == 2 and hd not in (64, 128):
                with pytest.raises(Exception, match="waves of 32 rows"):
                    ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(starts), d(past_t), out, scale, window,
                                               nh, nkv, hd, variant=variant)
                continue
            ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(starts), d(past_t), out, scale, window, nh, nkv,
                                       hd, variant=variant)
            close(out, want, 2e-2, 1e-2, what=f"attention prefill bf16, variant {variant}")
            # sequences with a single new token left out (a step of prompts and single tokens hands them to the
            # kernel for single tokens): their rows stay as they were, the others are computed as before
            if 1 in new and any(n > 1 for n in new):
                out.fill_(7.0)
                ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(starts), d(past_t), out, scale, window, nh, nkv,
                                           hd, variant=variant, skip_below=2)
                single = torch.tensor([n == 1 for n in new])[tok_seq.long()]
                assert bool((out.cpu()[single] == 7.0).all()), "a single token's row was written"
                close(out.cpu()[~single], want[~single], 2e-2, 1e-2, what=f"prompts beside skipped single tokens, variant {variant}")


@pytest.mark.parametrize("nh,nkv,hd,past,new,window,softcap,sloped", [
    (4, 2, 16, [0, 0], [40, 130], 0, 0.0, True),          # a penalty in the distance alone
    (8, 2, 64, [100, 0], [70, 129], 0, 2.0, False),       # a soft cap alone (head size 64: the kernel with 16 rows a wave takes it)
    (32, 8, 128, [30], [300], 0, 1.0, True),              # both, at the head size and group of the large models
    (6, 3, 48, [10, 0], [40, 200], 50, 3.0, True),        # with a window
])
def test_attention_with_terms_on_the_scores(ops, nh, nkv, hd, past, new, window, softcap, sloped):
    """score = cap * tanh(score / cap) - slope[head] * (query position - key position) before mask and softmax, in
    every attention kernel: 32-bit, prompt (bf16), single tokens in splits (bf16), against the plain statement."""
    B = len(past)
    lens = [p + n for p, n in zip(past, new)]
    width = max((T + 63) // 64 for T in lens) + 1
    table = shuffled_table(B, width, 5)
    slopes = torch.tensor([0.5 ** (1 + h % 5) for h in range(nh)], dtype=F32) if sloped else None
    tok_seq, tok_pos, starts, past_t, len_t = step_arrays(past, new)
    N = len(tok_seq)
    scale = 1 / math.sqrt(hd)
    d = lambda t: None if t is None else t.to(DEV)
    for dtype in (F32, BF16):
        k, v = make_cache(B * width, nkv, hd, dtype, 50)
        fill_sequences(k, v, table, lens, nkv, hd, dtype, 51)
        q = rnd((N, nh * hd), 52, dtype, 2.0)              # scores large enough that the cap bends them
        want = torch.empty((N, nh * hd), dtype=F32)
        ref.attention_f32(q.float(), torch.nan_to_num(k.float()), torch.nan_to_num(v.float()), table, tok_seq, tok_pos, want,
                          scale, window, nh, nkv, hd, slopes, softcap)
        plain = torch.empty_like(want)
        ref.attention_f32(q.float(), torch.nan_to_num(k.float()), torch.nan_to_num(v.float()), table, tok_seq, tok_pos, plain,
                          scale, window, nh, nkv, hd)
        assert float((want - plain).abs().max()) > 0.1     # the terms matter at these sizes
        out = torch.empty((N, nh * hd), dtype=dtype, device=DEV)
        if dtype == F32:
            ops.attention_f32(d(q), d(k), dv(v), d(table), d(tok_seq), d(tok_pos), out, scale, window, nh, nkv, hd,
                              slopes=d(slopes), softcap=softcap)
            close(out, want, 2e-4, what="attention f32 with terms")
            continue
        ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(starts), d(past_t), out, scale, window, nh, nkv, hd,
                                   slopes=d(slopes), softcap=softcap)
        close(out, want, 2e-2, 1e-2, what="attention prefill bf16 with terms")
        if hd in (64, 128):
            with pytest.raises(Exception, match="no terms on the scores"):
                ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(starts), d(past_t), out, scale, window, nh, nkv,
                                           hd, variant=2, slopes=d(slopes), softcap=softcap)
        # single tokens: the last token of each sequence as a decode step over the same cache
        last = torch.tensor([int(starts[b + 1]) - 1 for b in range(B)])
        outd = torch.empty((B, nh * hd), dtype=BF16, device=DEV)
        for splits in (1, 3):
            work = torch.empty(B * nh * splits * (hd + 2), dtype=F32, device=DEV)
            ops.attention_decode_bf16(d(q[last].contiguous()), d(k), dv(v), d(table), d(torch.tensor(lens, dtype=I32)), outd,
                                      work, splits, scale, window, nh, nkv, hd, slopes=d(slopes), softcap=softcap)
            close(outd, want[last], 2e-2, 1e-2, what=f"attention decode bf16 with terms, {splits} splits")


def merged_in_kernel(run, two_kernels, want, lens, splits, window, nh, nkv, work):
    """The same call with the merge of the splits inside the one launch, by the workgroup that finishes last:
    first with every sequence in `splits` splits, then with the host's work list, which gives long sequences
    more of them; twice each with the same counters, which the kernel has to leave at zero.  Before every run
    the partial results' memory is filled with NaN by another kernel: a workgroup that merged what an earlier
    launch left in its cache, and not what the other workgroups of this launch have written, would show it."""
    if splits == 1:
        return
    chunks = -(-(nh // nkv) // 16)
    counters = torch.zeros(len(lens) * nkv * chunks, dtype=I32, device=DEV)
    items = torch.tensor(rt.decode_items(lens, splits, window or None), dtype=I32, device=DEV)
    for what, kw in (("merged in the kernel", dict(counters=counters)),
                     ("with a work list", dict(counters=counters, items=items)),
                     ("with a work list, merged by the second kernel", dict(items=items))):
        outs = []
        for _ in range(2):
            got = torch.full_like(two_kernels, float("nan"))
            work.fill_(float("nan"))
            run(got, **kw)
            close(got, want, 2e-2, 1e-2, what=f"decode attention {what}")
            outs.append(got.cpu())
            assert int(counters.abs().sum()) == 0, f"{what}: counters are not back at zero"
        assert torch.equal(outs[0], outs[1]), f"{what}: two runs differ"
    # the same splits merged by either way: the same sums in another order
    got = torch.empty_like(two_kernels)
    run(got, counters=counters)
    close(got, two_kernels.float().cpu(), 1e-2, 1e-2, what="merge in the kernel against the merge kernel")


@pytest.mark.parametrize("nh,nkv,hd,lens,window,splits", [
    (8, 2, 64, [600, 3], 0, 4),                 # crates/synaptix-kernels-cuda/tests/cuda_flash_decode.rs:101 GQA, Tkv=600
    (4, 4, 128, [40], 0, 8),                    # more splits than pages (empty splits), ibid. 130-183
    (40, 2, 32, [129, 64, 65, 1], 0, 3),        # 20 heads a group: two chunks of 16
    (8, 1, 16, [1000, 77], 0, 16),
    (4, 2, 96, [500, 30], 100, 5),
    (32, 8, 128, [2100] * 3, 0, 11),
    (6, 2, 48, [35], 0, 1),                     # head sizes that are no multiple of 32, three heads a group
    (6, 2, 48, [200, 35, 64], 0, 3),
    (5, 1, 80, [100, 300], 0, 2),
    (4, 4, 112, [70], 0, 1),
    (8, 2, 256, [130, 700], 0, 4),
    (32, 8, 128, [7000, 40], 0, 32),            # long contexts: 32 and 64 splits, most of them empty for the short sequence
    (8, 2, 64, [6500, 130, 7000], 0, 64),
    (4, 1, 32, [4100], 0, 24),
    (32, 8, 128, [3000, 500, 2600, 100, 1500], 0, 16),   # 640 workgroups: more than two a compute unit, merged by the second kernel
])
def test_attention_decode_bf16(ops, nh, nkv, hd, lens, window, splits):
    B = len(lens)
    width = max((T + 63) // 64 for T in lens) + 2
    table = shuffled_table(B, width, 4)
    k, v = make_cache(B * width, nkv, hd, BF16, 40, fill="nan" if hd == 64 else "garbage")
    fill_sequences(k, v, table, lens, nkv, hd, BF16, 41)
    tok_seq = torch.arange(B, dtype=I32)
    tok_pos = torch.tensor([T - 1 for T in lens], dtype=I32)
    q = rnd((B, nh * hd), 42, BF16)
    scale = 1 / math.sqrt(hd)
    want = torch.empty((B, nh * hd), dtype=F32)
    kf, vf = torch.nan_to_num(k.float()), torch.nan_to_num(v.float())
    ref.attention_f32(q.float(), kf, vf, table, tok_seq, tok_pos, want, scale, window, nh, nkv, hd)
    d = lambda t: t.to(DEV)
    out = torch.empty((B, nh * hd), dtype=BF16, device=DEV)
    work = torch.empty(B * nh * splits * (hd + 2), dtype=F32, device=DEV)
    ops.attention_decode_bf16(d(q), d(k), dv(v), d(table), d(torch.tensor(lens, dtype=I32)), out, work, splits, scale,
                              window, nh, nkv, hd)
    close(out, want, 2e-2, 1e-2, what="attention decode bf16")
    merged_in_kernel(lambda out2, **kw: ops.attention_decode_bf16(
        d(q), d(k), dv(v), d(table), d(torch.tensor(lens, dtype=I32)), out2, work, splits, scale, window, nh, nkv, hd, **kw),
        out, want, lens, splits, window, nh, nkv, work)


@pytest.mark.parametrize("nh,nkv,hd,rows,hi,window", [
    (32, 8, 128, 33, 3000, 0),                  # one workgroup more than a compute unit
    (32, 8, 128, 64, 300, 0),
    (4, 4, 16, 65, 700, 0),
    (8, 8, 64, 48, 900, 200),                   # a window
    (64, 16, 128, 17, 4000, 0),                 # two sequences a place
])
def test_attention_decode_over_bins(ops, nh, nkv, hd, rows, hi, window):
    """More sequences x kv heads than compute units, one much longer than the rest and some of a single token: the list that
    gives every compute unit the same share of the keys, long sequences cut and merged inside the launch."""
    gen = torch.Generator().manual_seed(rows)
    lens = torch.randint(1, hi, (rows,), generator=gen).tolist()
    lens[0], lens[1], lens[-1] = 3 * hi, hi, 1
    width = (max(lens) + 63) // 64 + 1
    pages = [(n + 63) // 64 for n in lens]
    table = torch.zeros((rows, width), dtype=I32)
    ids, at = torch.randperm(sum(pages), generator=gen).to(I32), 0
    for b, p in enumerate(pages):
        table[b, :p] = ids[at:at + p]
        at += p
    k, v = make_cache(sum(pages), nkv, hd, BF16, 80)
    fill_sequences(k, v, table, lens, nkv, hd, BF16, 82)
    q = rnd((rows, nh * hd), 81, BF16)
    want = torch.empty((rows, nh * hd), dtype=F32)
    lens_t, scale = torch.tensor(lens, dtype=I32), 1 / math.sqrt(hd)
    ref.attention_f32(q.float(), k.float(), v.float(), table, torch.arange(rows, dtype=I32), lens_t - 1,
                      want, scale, window, nh, nkv, hd)
    places, d = ops.decode_bins(rows, nkv), lambda t: t.to(DEV)
    assert places == 256 // nkv
    items = rt.decode_bins(lens, ops.DECODE_BIN_SPLITS, places, window or None)
    T = ops.DECODE_BIN_SPLITS * rows
    assert window or max(items[4 * i + 1] >> 16 for i in range(T)) > 1
    counters = torch.zeros(rows * nkv, dtype=I32, device=DEV)
    work = torch.full((rows * nh * ops.DECODE_BIN_SPLITS * (hd + 2),), float("nan"), dtype=F32, device=DEV)
    for kw in (dict(counters=counters), {}):                # merged in the launch, and by the second kernel
        out = torch.full((rows, nh * hd), float("nan"), dtype=BF16, device=DEV)
        ops.attention_decode_bf16(d(q), d(k), dv(v), d(table), d(lens_t), out, work, ops.DECODE_BIN_SPLITS, scale, window, nh, nkv,
                                  hd, items=torch.tensor(items, dtype=I32, device=DEV), **kw)
        close(out, want, 2e-2, 1e-2, what="decode attention over bins")
    assert int(counters.abs().sum()) == 0


@pytest.mark.parametrize("nh,nkv,hd,rows,hi,window,parts", [(32, 8, 128, 33, 2000, 0, 4), (8, 8, 64, 48, 900, 200, 0), (16, 4, 32, 65, 500, 0, 2)])
def test_fused_decode_over_bins(ops, nh, nkv, hd, rows, hi, window, parts):
    """The same through the kernel that a decode step runs, which makes q, k and v of the new tokens itself and writes them to the cache."""
    gen = torch.Generator().manual_seed(rows)
    lens = torch.randint(1, hi, (rows,), generator=gen).tolist()
    lens[0], lens[1], lens[-1] = 3 * hi, hi, 1
    width = (max(lens) + 63) // 64 + 1
    pages = [(n + 63) // 64 for n in lens]
    table = torch.zeros((rows, width), dtype=I32)
    ids, at = torch.randperm(sum(pages), generator=gen).to(I32), 0
    for b, p in enumerate(pages):
        table[b, :p] = ids[at:at + p]
        at += p
    k, v = make_cache(sum(pages), nkv, hd, BF16, 83)
    fill_sequences(k, v, table, lens, nkv, hd, BF16, 84)
    qkv = rnd((rows, (nh + 2 * nkv) * hd), 85, F32)
    qkv = (qkv[None] * (torch.arange(1, parts + 1, dtype=F32)[:, None, None] / sum(range(parts + 1)))).contiguous() if parts else qkv.to(BF16)
    qg, kg = ((1 + 0.2 * rnd((hd,), 86 + i)).to(BF16) for i in range(2))
    ang = torch.arange(max(lens) + 1, dtype=F32)[:, None] * (0.3 / (1 + torch.arange(hd // 2, dtype=F32)))[None, :]
    cos, sin = torch.cos(ang), torch.sin(ang)
    seq_len, scale = torch.tensor(lens, dtype=I32), 1 / math.sqrt(hd)
    k_ref, v_ref, q_ref = k.clone(), v.clone(), torch.empty((rows, nh * hd), dtype=BF16)
    ref.qk_norm_rope_kv_write(qkv, q_ref, k_ref, v_ref, table, torch.arange(rows, dtype=I32), seq_len - 1, qg, kg, 1e-5, cos, sin, nh, nkv, hd)
    want = torch.empty((rows, nh * hd), dtype=F32)
    ref.attention_f32(q_ref.float(), k_ref.float(), v_ref.float(), table, torch.arange(rows, dtype=I32), seq_len - 1, want, scale, window, nh, nkv, hd)
    S = ops.DECODE_BIN_SPLITS
    items = rt.decode_bins(lens, S, ops.decode_bins(rows, nkv, nh // nkv), window or None)
    assert window or max(items[4 * i + 1] >> 16 for i in range(S * rows)) > 1
    d = lambda t: t.to(DEV)
    counters = torch.zeros(rows * nkv, dtype=I32, device=DEV)
    work = torch.full((rows * nh * S * (hd + 2),), float("nan"), dtype=F32, device=DEV)
    for kw in (dict(counters=counters), {}):
        kd, vd, out = d(k), dv(v), torch.full((rows, nh * hd), float("nan"), dtype=BF16, device=DEV)
        ops.attention_decode_fused_bf16(d(qkv), kd, vd, d(table), d(seq_len), out, work, S, scale, window, nh, nkv, hd, d(qg), d(kg), 1e-5,
                                        d(cos), d(sin), items=torch.tensor(items, dtype=I32, device=DEV), **kw)
        close(out, want, 2e-2, 1e-2, what="fused decode attention over bins")
        close(kd, k_ref.float(), 2e-2, 1e-2, what="k pages after the step")
        close(hv(vd), v_ref.float(), 2e-2, 1e-2, what="v pages after the step")
    assert int(counters.abs().sum()) == 0


@pytest.mark.parametrize("lens,splits", [([2061] * 8, 4), ([2061], 16), ([3908, 457, 1200, 2500], 8)])
def test_merge_inside_the_launch_reads_what_this_launch_wrote(ops, lens, splits):
    """The workgroup that merges the splits reads partial results that workgroups on other XCDs, each with a
    second-level cache of its own, wrote within the same launch.  200 launches at a decode step's shapes, the
    memory of the partial results filled with NaN by another kernel before each and the keys of other launches
    read in between: every output equals the first, none is NaN."""
    nh, nkv, hd = 32, 8, 128
    B = len(lens)
    width = max((T + 63) // 64 for T in lens) + 1
    table = shuffled_table(B, width, 6)
    k, v = make_cache(B * width, nkv, hd, BF16, 70)
    fill_sequences(k, v, table, lens, nkv, hd, BF16, 71)
    q = rnd((B, nh * hd), 72, BF16)
    d = lambda t: t.to(DEV)
    qd, kd, vd, td, ld = d(q), d(k), dv(v), d(table), d(torch.tensor(lens, dtype=I32))
    work = torch.empty(B * nh * splits * (hd + 2), dtype=F32, device=DEV)
    counters = torch.zeros(B * nkv, dtype=I32, device=DEV)
    items = torch.tensor(rt.decode_items(lens, splits), dtype=I32, device=DEV)
    other = torch.randn(64 << 20, device=DEV)          # 256 MB that a kernel in between reads
    first = None
    for i in range(200):
        out = torch.full((B, nh * hd), float("nan"), dtype=BF16, device=DEV)
        work.fill_(float("nan"))
        if i % 3 == 0:
            other.sum()
        ops.attention_decode_bf16(qd, kd, vd, td, ld, out, work, splits, 1 / math.sqrt(hd), 0, nh, nkv, hd,
                                  counters=counters, items=items if i % 2 else None)
        if first is None:
            first = {}
        key = i % 2
        if key not in first:
            assert torch.isfinite(out.float()).all()
            first[key] = out.clone()
        else:
            assert torch.equal(out, first[key]), f"launch {i} differs from the first of its kind"
    assert int(counters.abs().sum()) == 0


@pytest.mark.parametrize("nh,nkv,hd,rot,norm,lens,window,splits,parts,own", [
    (4, 2, 16, 16, True, [1, 5, 64, 65, 200], 0, 1, 0, True),        # a first token, page edges
    (8, 2, 128, 128, True, [700, 33, 129], 0, 4, 8, True),           # float partial sums, splits
    (6, 2, 48, 32, True, [300, 64], 0, 3, 3, True),                  # partial rotation, head size 48
    (4, 1, 64, 64, False, [500, 2], 100, 2, 0, True),                # no q/k norm, a window
    (40, 2, 32, 0, True, [90, 300], 0, 2, 2, True),                  # no rotation, 20 heads a group (two chunks)
    (8, 4, 128, 128, True, [257, 1000], 0, 8, 4, False),             # reads a cache that another layer wrote
    (32, 8, 128, 128, True, [7000, 33], 0, 32, 4, True),             # long contexts: 32 and 64 splits
    (4, 1, 64, 64, True, [6500, 100, 6401], 0, 64, 0, True),
])
def test_attention_decode_with_qkv_intake(ops, nh, nkv, hd, rot, norm, lens, window, splits, parts, own):
    """Decode attention that makes q, k and v from the fused projection itself equals the q/k kernel
    followed by plain decode attention: the same outputs and the same cache contents afterwards."""
    B, heads = len(lens), nh + 2 * nkv
    width = max((T + 63) // 64 for T in lens) + 2
    table = shuffled_table(B, width, 5)
    k, v = make_cache(B * width, nkv, hd, BF16, 60)
    fill_sequences(k, v, table, lens, nkv, hd, BF16, 61)
    qkv_full = rnd((B, heads * hd), 62, F32)
    if parts:
        cut = torch.rand((parts, 1, 1), generator=torch.Generator().manual_seed(63)) + 0.1
        qkv = (qkv_full[None] * (cut / cut.sum())).contiguous()       # float partial sums that add up to it
    else:
        qkv = qkv_full.to(BF16)
    qg = (1 + 0.2 * rnd((hd,), 64)).to(BF16) if norm else None
    kg = (1 + 0.2 * rnd((hd,), 65)).to(BF16) if norm else None
    cos = sin = None
    if rot:
        ang = torch.arange(max(lens) + 1, dtype=F32)[:, None] * (0.3 / (1 + torch.arange(rot // 2, dtype=F32)))[None, :]
        cos, sin = torch.cos(ang), torch.sin(ang)
    seq_len = torch.tensor(lens, dtype=I32)
    tok_seq, tok_pos = torch.arange(B, dtype=I32), seq_len - 1
    scale = 1 / math.sqrt(hd)
    # the two-kernel way, on the CPU reference
    k_ref, v_ref = k.clone(), v.clone()
    q_ref = torch.empty((B, nh * hd), dtype=BF16)
    ref.qk_norm_rope_kv_write(qkv, q_ref, k_ref, v_ref, table, tok_seq, tok_pos, qg, kg, 1e-5, cos, sin, nh, nkv, hd,
                              write_kv=own)
    want = torch.empty((B, nh * hd), dtype=F32)
    ref.attention_f32(q_ref.float(), k_ref.float(), v_ref.float(), table, tok_seq, tok_pos, want, scale, window, nh, nkv, hd)
    d = lambda t: None if t is None else t.to(DEV)
    kd, vd = d(k), dv(v)
    out = torch.empty((B, nh * hd), dtype=BF16, device=DEV)
    work = torch.empty(B * nh * splits * (hd + 2), dtype=F32, device=DEV)
    ops.attention_decode_fused_bf16(d(qkv), kd, vd, d(table), d(seq_len), out, work, splits, scale, window, nh, nkv, hd,
                                    d(qg), d(kg), 1e-5, d(cos), d(sin), write_kv=own)
    close(out, want, 2e-2, 1e-2, what="decode attention with q/k/v intake")
    merged_in_kernel(lambda out2, **kw: ops.attention_decode_fused_bf16(
        d(qkv), kd, vd, d(table), d(seq_len), out2, work, splits, scale, window, nh, nkv, hd, d(qg), d(kg), 1e-5, d(cos),
        d(sin), write_kv=own, **kw), out, want, lens, splits, window, nh, nkv, work)
    # the cache afterwards: the new rows written (or nothing touched)
    close(kd, k_ref.float(), 2e-2, 1e-2, what="k pages after the step")
    close(hv(vd), v_ref.float(), 2e-2, 1e-2, what="v pages after the step")
    if not own:
        assert torch.equal(kd.cpu(), k) and torch.equal(hv(vd), v)


def test_attention_far_key_stands_out(ops):
    """One key among hundreds is made to dominate: the output must be that key's value, in every
    kernel.  A kernel that loses a page, a split or the cache's start would not show it with
    random data."""
    nh, nkv, hd, T = 4, 2, 64, 700
    scale = 1 / math.sqrt(hd)
    for far in (0, 63, 64, 350, T - 1):
        table = shuffled_table(1, 12, far)
        k, v = make_cache(12, nkv, hd, BF16, 50)
        fill_sequences(k, v, table, [T], nkv, hd, BF16, 51)
        q = rnd((1, nh * hd), 52, BF16)
        page = int(table[0, far // 64])
        for h in range(nkv):   # the far key is 20 x the query of the group's first head
            k[page, h, far % 64, :] = (q.view(nh, hd)[h * 2] * 20).to(BF16)
        want = v[page, :, :, far % 64].float()            # [nkv, hd]
        d = lambda t: t.to(DEV)
        lens = torch.tensor([T], dtype=I32)
        out = torch.empty((1, nh * hd), dtype=BF16, device=DEV)
        work = torch.empty(nh * 6 * (hd + 2), dtype=F32, device=DEV)
        ops.attention_decode_bf16(d(q), d(k), dv(v), d(table), d(lens), out, work, 6, scale, 0, nh, nkv, hd)
        got = out.cpu().float().view(nh, hd)
        for h in range(nkv):
            close(got[h * 2], want[h], 3e-2, 2e-2, f"decode, far key {far}")
        outp = torch.empty((1, nh * hd), dtype=BF16, device=DEV)
        ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(torch.tensor([0, 1], dtype=I32)),
                                   d(torch.tensor([T - 1], dtype=I32)), outp, scale, 0, nh, nkv, hd)
        gotp = outp.cpu().float().view(nh, hd)
        for h in range(nkv):
            close(gotp[h * 2], want[h], 3e-2, 2e-2, f"prefill, far key {far}")
        o32 = torch.empty((1, nh * hd), dtype=F32, device=DEV)
        ops.attention_f32(d(q.float()), d(k.float()), d(v.float()), d(table), d(torch.zeros(1, dtype=I32)),
                          d(torch.tensor([T - 1], dtype=I32)), o32, scale, 0, nh, nkv, hd)
        got32 = o32.cpu().view(nh, hd)
        for h in range(nkv):
            close(got32[h * 2], want[h], 1e-3, 1e-3, f"f32, far key {far}")


def test_attention_window_edge(ops):
    """The key just outside the window dominates if it is seen: it must not be."""
    nh, nkv, hd, T, W = 2, 1, 32, 300, 100
    scale = 1 / math.sqrt(hd)
    table = shuffled_table(1, 6, 9)
    k, v = make_cache(6, nkv, hd, BF16, 60)
    fill_sequences(k, v, table, [T], nkv, hd, BF16, 61)
    q = rnd((1, nh * hd), 62, BF16)
    edge = T - 1 - W          # the last key outside: visible keys are j > T-1-W
    page = int(table[0, edge // 64])
    k[page, 0, edge % 64, :] = (q.view(nh, hd)[0] * 20).to(BF16)
    tok_seq, tok_pos = torch.zeros(1, dtype=I32), torch.tensor([T - 1], dtype=I32)
    want = torch.empty((1, nh * hd), dtype=F32)
    ref.attention_f32(q.float(), k.float(), v.float(), table, tok_seq, tok_pos, want, scale, W, nh, nkv, hd)
    seen = torch.empty((1, nh * hd), dtype=F32)
    ref.attention_f32(q.float(), k.float(), v.float(), table, tok_seq, tok_pos, seen, scale, W + 1, nh, nkv, hd)
    assert (want - seen).abs().max() > 1.0, "the test's key does not dominate"
    d = lambda t: t.to(DEV)
    out = torch.empty((1, nh * hd), dtype=BF16, device=DEV)
    work = torch.empty(nh * 3 * (hd + 2), dtype=F32, device=DEV)
    ops.attention_decode_bf16(d(q), d(k), dv(v), d(table), d(torch.tensor([T], dtype=I32)), out, work, 3, scale, W, nh,
                              nkv, hd)
    close(out, want, 2e-2, 1e-2, "decode at the window's edge")
    ops.attention_prefill_bf16(d(q), d(k), dv(v), d(table), d(torch.tensor([0, 1], dtype=I32)),
                               d(torch.tensor([T - 1], dtype=I32)), out, scale, W, nh, nkv, hd)
    close(out, want, 2e-2, 1e-2, "prefill at the window's edge")
    o32 = torch.empty((1, nh * hd), dtype=F32, device=DEV)
    ops.attention_f32(d(q.float()), d(k.float()), d(v.float()), d(table), d(tok_seq), d(tok_pos), o32, scale, W, nh, nkv,
                      hd)
    close(o32, want, 1e-4, what="f32 at the window's edge")


# ----------------------------------------------------------------------------- sampling

@pytest.mark.parametrize("V", [1000, 999, 40004])
def test_sample_rows_greedy_and_ties(ops, V):
    x = rnd((5, V), 70)
    x[1, 17] = x[1, 900] = 9.0           # the last of equal maxima wins
    x[2, :] = 0.0                        # all equal: the last index
    out = torch.empty(5, dtype=I32, device=DEV)
    ops.sample_rows(x.to(DEV), None, None, out)
    want = [int(x[0].argmax()), 900, V - 1, int(x[3].argmax()), int(x[4].argmax())]
    assert out.cpu().tolist() == want


def test_sample_rows_temperature(ops):
    V, R = 333, 64
    x = rnd((R, V), 71, scale=3.0)
    temps = torch.tensor([0.7, 1.0, 0.0, 1.5] * (R // 4))
    g = torch.Generator().manual_seed(5)
    u = torch.rand(R, generator=g)
    want = torch.empty(R, dtype=I32)
    ref.sample_rows(x, temps, u, want)
    out = torch.empty(R, dtype=I32, device=DEV)
    ops.sample_rows(x.to(DEV), temps.to(DEV), u.to(DEV), out)
    got = out.cpu()
    # a draw falls on the other side of a boundary only if u is within rounding of the CDF there
    differ = int((got != want).sum())
    assert differ <= 1, f"{differ} of {R} draws differ"
    # u = 1 can never be below the last cumulative sum of rounded probabilities: the last index
    ops.sample_rows(x.to(DEV), torch.ones(R).to(DEV), torch.full((R,), 1.5).to(DEV), out)
    assert out.cpu().tolist() == [V - 1] * R


@pytest.mark.parametrize("V,left", [(1, 1), (31, 5), (1023, 1023), (1025, 40), (16384, 16384), (16385, 16385), (33000, 33000), (151936, 50), (151937, 3)])
def test_sample_rows_draws_where_the_sum_passes_u(ops, V, left):
    """Chunks of every length, with most entries dropped and with none, and u at both ends: the drawn entry is where the 64-bit
    running sum passes u, up to the roundings of V additions in 32 bits (2^-24 each), and never a dropped one."""
    g = torch.Generator().manual_seed(V)
    x = torch.full((6, V), -math.inf)
    for r in range(6):
        keep = torch.randperm(V, generator=g)[:left]
        x[r, keep] = 3 * torch.randn(left, generator=g)
    u = torch.tensor([0.0, 1.0, 0.5, 0.999, 1e-6, 0.31])
    t = torch.tensor([1.0, 1.0, 0.7, 1.0, 1.5, 1.0])
    out = torch.empty(6, dtype=I32, device=DEV)
    ops.sample_rows(x.to(DEV), t.to(DEV), u.to(DEV), out)
    p = torch.softmax(x.double() / t.double()[:, None], -1)
    cum, off = p.cumsum(-1), 2 ** -24 * (V // 1024 + 1 + 1024)
    for r, i in enumerate(out.tolist()):
        before = float(cum[r, i] - p[r, i])
        assert p[r, i] > 0 and before <= float(u[r]) + off and float(u[r]) <= float(cum[r, i]) + off, (r, i)


@pytest.mark.parametrize("V,left", [(2000, 700), (16384, 16000), (16385, 500), (33000, 900), (151936, 50)])
def test_sample_rows_draws_no_dropped_entry(ops, V, left):
    """u within a few steps of 2^-24 of every place where the running sum may pass it, and beyond its end: the chunks' sums
    are rounded apart from each other, and what they leave between them belongs to no dropped entry."""
    g = torch.Generator().manual_seed(V)
    x = torch.full((V,), -math.inf)
    keep = torch.randperm(V, generator=g)[:left].sort().values
    x[keep] = 2 * torch.randn(left, generator=g)
    cum = torch.softmax(x.double(), 0)[keep].cumsum(0).float()
    steps = torch.arange(-4, 5, dtype=F32) * 2 ** -24
    u = torch.cat([(cum[:: max(1, left // 60), None] + steps).flatten(), torch.tensor([0.0, 1 - 2 ** -24, 1.0, 1.5])])
    rows = x.expand(u.numel(), V).contiguous().to(DEV)
    out = torch.empty(u.numel(), dtype=I32, device=DEV)
    ops.sample_rows(rows, torch.ones(u.numel(), device=DEV), u.to(DEV), out)
    got = out.cpu().long()
    assert torch.isfinite(x[got]).all() and got[-1] == keep[-1]
    nan = torch.full((2, 1000), float("nan"), device=DEV)
    nan[1] = -math.inf
    ops.sample_rows(nan, torch.ones(2, device=DEV), torch.full((2,), 0.5, device=DEV), out[:2])
    assert out[:2].tolist() == [999, 999]


def test_sample_rows_frequencies(ops):
    """Frequencies of many draws lie within 0.01 of the probabilities
    (as crates/synaptix-infer/tests/ref_infer.rs:114-166, with fewer draws)."""
    V, R = 50, 20000
    logits = rnd((1, V), 72, scale=1.5)
    x = logits.expand(R, V).contiguous()
    g = torch.Generator().manual_seed(6)
    u = torch.rand(R, generator=g)
    out = torch.empty(R, dtype=I32, device=DEV)
    ops.sample_rows(x.to(DEV), torch.full((R,), 0.8).to(DEV), u.to(DEV), out)
    freq = torch.bincount(out.cpu().long(), minlength=V).float() / R
    p = torch.softmax(logits[0] / 0.8, 0)
    assert (freq - p).abs().max() < 0.012


def test_products_of_random_shapes(ops):
    """Shapes drawn at random over every kind of product (plain, as partial sums for a reader that adds them, gated)
    through the entry points that the parts use (parts.linear): each lands in whichever kernel the sizes select, in
    fragment order where the sizes allow it and in plain rows where they do not, and equals the 64-bit product."""
    import random
    from synaptix_amd.parts.linear import Matrix, linear, linear_for_sum
    r = random.Random(11)
    done = 0
    while done < 48:
        M = r.choice([1, 2, 5, 8, 9, 13, 16, 17, 32, 33, 64, 65, 100, 128, 129, 255, 257, 300, 513, 700])
        K = r.choice([8, 24, 32, 40, 64, 96, 128, 136, 192, 256, 264, 512, 1000, 1024, 2080, 4096])
        N = r.choice([8, 16, 24, 32, 48, 80, 96, 128, 160, 200, 384, 400, 1000, 1008, 2048, 4096, 6144, 32784])
        kind = r.choice(["plain", "sum", "gated"])
        if kind == "gated":
            N = max(32, N // 32 * 32)
        if M * N * K > 6e9:
            continue
        done += 1
        x, w = rnd((M, K), 300 + done, BF16), rnd((N, K), 400 + done, BF16, 0.05)
        full = x.double() @ w.double().T
        atol = 4e-4 * math.sqrt(K) + 1e-3
        if kind == "gated":
            m = Matrix(ops.pair_rows(w[:N // 2].contiguous().to(DEV), w[N // 2:].contiguous().to(DEV)))
            out = torch.full((M, N // 2), float("nan"), dtype=BF16, device=DEV)
            ops.gemm_swiglu(x.to(DEV), m.data, out)
            g, u = full[:, :N // 2], full[:, N // 2:]
            close(out, (g / (1 + torch.exp(-g)) * u).float(), atol + 0.02, 1e-2, f"gated {M}x{N}x{K}")
        else:
            m = Matrix(w.to(DEV))
            got = linear(x.to(DEV), m, F32) if kind == "plain" else linear_for_sum(x.to(DEV), m)
            close(got.sum(0) if got.dim() == 3 else got, full.float(), atol, what=f"{kind} {M}x{N}x{K}")


def test_attention_of_random_shapes(ops):
    """The attention tests above at shapes drawn at random: head sizes 16 to 256, groups of 1 to 20 heads, sequences that
    begin, end or are cut at page edges, windows down to one key, any number of splits."""
    import random
    r = random.Random(12)
    for _ in range(10):
        hd = r.choice([16, 32, 48, 64, 80, 96, 112, 128, 160, 256])
        nkv = r.choice([1, 2, 3, 4, 8])
        nh = nkv * r.choice([1, 2, 3, 4, 7, 8, 17, 20])
        if nh * hd > 8192:
            continue
        B = r.randint(1, 4)
        past = [r.choice([0, 0, 1, 63, 64, 65, 100, 200, 500]) for _ in range(B)]
        new = [r.choice([1, 2, 31, 32, 33, 64, 100, 128, 129, 200, 300]) for _ in range(B)]
        window = r.choice([0, 0, 0, 1, 37, 64, 70, 200])
        lens = [r.choice([1, 2, 63, 64, 65, 130, 300, 700, 2100, 5000]) for _ in range(B)]
        splits = r.choice([1, 2, 3, 4, 8, 16, 32])
        rot = r.choice([0, hd, hd, hd // 2 if (hd // 2) % 2 == 0 else hd])
        test_attention_prefill(ops, BF16, nh, nkv, hd, past, new, window)
        test_attention_decode_bf16(ops, nh, nkv, hd, lens, window, splits)
        test_attention_decode_with_qkv_intake(ops, nh, nkv, hd, rot, r.random() < 0.7, lens, window, splits,
                                              r.choice([0, 0, 2, 4, 8]), r.random() < 0.8)


@pytest.mark.parametrize("nf", [2, 4, 6])
@pytest.mark.parametrize("M", [9, 16, 17, 33, 48, 49, 64, 65, 96, 97, 128])
def test_products_of_few_rows_straight_to_registers(ops, nf, M):
    """gemm_rows_kernel by the number of its rows of W, wherever that many rows of x fit: N that is no multiple of a workgroup's rows, K whose
    pairs of steps do not divide by four waves nor by the slices (some empty), every output, against 64 bits at every place.  The
    bounds: 32-bit sums of K products of bf16 numbers, 2^-8 of a result that is rounded."""
    if M > {2: 128, 4: 96, 6: 48}[nf]:
        pytest.skip("not compiled: more sums than registers")
    for N, K, slices in ((32, 128, 1), (224, 640, 1), (208, 384, 2), (1008, 2176, 3), (96, 1024, 8), (16, 256, 5)):
        x, w = rnd((M, K), M + K, BF16), rnd((N, K), N + K, BF16, 0.05)
        full, wp = x.double() @ w.double().T, ops.pack_weight(w.to(DEV))
        bound = 2 ** -24 * 8 * math.sqrt(K) + 2 ** -22 * (x.double().abs() @ w.double().abs().T)
        for dt in (F32, BF16) if slices == 1 else (F32,):
            out = torch.full((slices, M, N) if slices > 1 else (M, N), float("nan"), dtype=dt, device=DEV)
            ops.gemm(x.to(DEV), wp, out, rows=nf)
            got = (out.double().sum(0) if slices > 1 else out.double()).cpu()
            assert bool(((got - full).abs() <= bound + (2 ** -8 * full.abs() if dt == BF16 else 0)).all()), (N, K, slices, dt)
        if slices == 1:
            out = torch.full((M, N), float("nan"), device=DEV)
            ops.gemm(x.to(DEV), wp, out, point="relu_squared", rows=nf)
            assert bool(((out.cpu().double() - full.clamp(min=0) ** 2).abs() <= 2 * full.abs() * bound + bound ** 2 + 2 ** -22 * full ** 2).all())
        if N % 32 == 0 and slices == 1:
            paired = ops.pack_weight(ops.pair_rows(w[:N // 2].contiguous(), w[N // 2:].contiguous()).to(DEV))
            out = torch.full((M, N // 2), float("nan"), dtype=BF16, device=DEV)
            ops.gemm_swiglu(x.to(DEV), paired, out, rows=nf)
            g, u = full[:, :N // 2], full[:, N // 2:]
            want = g * torch.sigmoid(g) * u
            assert bool(((out.cpu().double() - want).abs() <= 2 ** -7 * want.abs() + 4 * bound.amax() * (1 + u.abs() + g.abs())).all()), (N, K)


def test_the_rule_for_products_of_few_rows_gives_sizes_that_run(ops):
    """Whatever the sizes, what the rule picks goes round once, fits the registers and leaves every slice work of its own."""
    for M in range(1, 140, 3):
        for N in (16, 48, 1024, 2560, 4096, 6144, 9728, 24576, 51200):
            for K in (128, 1024, 2560, 4096, 9728, 25600):
                for gated in (False, True):
                    s = 1 if gated else max(1, ops.rows_slices(M, N, K))
                    nf = ops.rows_tile(M, N, K, s, gated)
                    assert nf == 0 or (M <= {2: 128, 4: 96, 6: 48}[nf] and -(-N // (16 * nf)) * s <= ops.compute_units() and (s == 1 or K >= 512 * s))
                    assert nf or s == 1


def _filter(ops, x, options, ids=None, in_place=False):
    """ops.filter_rows over rows x [R, V] with options = list of dicts (k, p, mp, T, rep, pres, freq) and ids = list of lists."""
    R, V = x.shape
    col = lambda key, default, dt: torch.tensor([o.get(key, default) for o in options], dtype=dt).to(DEV)
    flat, starts = [], [0]
    for r in range(R):
        flat += list(ids[r]) if ids else []
        starts.append(len(flat))
    xd = x.to(DEV).contiguous()
    out = xd if in_place else torch.full_like(xd, float("nan"))
    counts = torch.zeros(R * V, dtype=I32, device=DEV) if flat else None
    ops.filter_rows(xd, out, col("T", 1.0, F32), col("k", 0, I32), col("p", 1.0, F32), col("mp", 0.0, F32),
                    col("rep", 1.0, F32), col("pres", 0.0, F32), col("freq", 0.0, F32),
                    torch.tensor(flat, dtype=I32).to(DEV) if flat else None,
                    torch.tensor(starts, dtype=I32).to(DEV) if flat else None, counts)
    torch.cuda.synchronize()
    if counts is not None:
        assert int(counts.abs().sum()) == 0, "the penalties' counters are not left zero"
    return out.cpu()


def _plain_filter(x, o, ids):
    """The plain processors in the reference's order (tests/plain_qwen3.py)."""
    import plain_qwen3 as P
    want = x.clone()
    if o.get("rep", 1.0) != 1.0:
        want = P.repetition_penalty(want, ids, o["rep"], 0)
    if o.get("pres", 0.0) != 0.0 or o.get("freq", 0.0) != 0.0:
        want = P.presence_frequency(want, ids, o.get("pres", 0.0), o.get("freq", 0.0), 0)
    T = o.get("T", 1.0)
    if T > 0 and T != 1.0:
        want = want / torch.tensor(T, dtype=F32)
    if o.get("k", 0):
        want = P.top_k(want, o["k"])
    if o.get("p", 1.0) < 1.0:
        want = P.top_p(want, o["p"]) if o["p"] <= 0.9 else _top_p_in_64_bit(want, o["p"])
    if o.get("mp", 0.0) > 0.0:
        want = P.min_p(want, o["mp"])
    return want


def _top_p_in_64_bit(x, p):
    """The rule of the plain top_p (a candidate stays while the sum of those before it is at most p * the sum of
    all; sorted by probability, equal ones in index order) with sums in 64-bit.  The reference adds up in 32-bit,
    one candidate after the other (crates/synaptix-infer/src/sampling/top_p.rs:31-40): deep in the tail of a large
    vocabulary a candidate is less than half a unit in the last place of that sum, the sum stands still and the
    cut is never reached; the kernel's sums are exact, so for p near 1 it is held against the rule, not against
    that rounding."""
    probs = torch.exp(x.double() - x.max().double())
    order = torch.argsort(probs, descending=True, stable=True)
    sp = probs[order]
    before = torch.cumsum(sp, 0) - sp
    out = x.clone()
    out[order[(before > p * probs.sum()) & torch.isfinite(x[order])]] = float("-inf")
    return out


@pytest.mark.parametrize("V", [97, 1000, 40000])
def test_filter_rows_against_the_plain_processors(ops, V):
    """Every processor alone and all together, rows with different options in one launch, against the plain
    processors: the same entries dropped, the kept ones equal up to the rounding of the penalty's power."""
    options = [dict(k=1), dict(k=17), dict(k=V - 1), dict(k=V), dict(p=0.9), dict(p=0.3), dict(p=0.999), dict(mp=0.05),
               dict(T=0.7), dict(T=0.0, k=5), dict(rep=1.3), dict(pres=0.4, freq=0.2), dict(rep=0.8, pres=-0.1),
               dict(T=0.8, k=40, p=0.85, mp=0.02, rep=1.2, pres=0.3, freq=0.1), dict(T=1.5, k=300, p=0.5), dict()]
    R = len(options)
    x = rnd((R, V), 90, scale=3.0)
    g = torch.Generator().manual_seed(V)
    ids = [torch.randint(-2, V + 3, (60,), generator=g).tolist() for _ in range(R)]       # some ids lie outside the vocabulary
    for r in range(R):
        ids[r] += ids[r][:20]                                                              # and some come several times
    got = _filter(ops, x, options, ids)
    for r, o in enumerate(options):
        want = _plain_filter(x[r], o, [t for t in ids[r] if t >= 0])
        differ = torch.isinf(got[r]) != torch.isinf(want)
        if o.get("p", 1.0) > 0.9 and bool(differ.any()):
            # deep in the tail neighbours in the sorted order lie 1e-8 of the mass apart, less than the rounding of
            # a 32-bit exponential: an entry may fall on the other side only if it stands that close to the cut
            probs = torch.exp(x[r].double() - x[r].max().double())
            above = torch.stack([probs[probs > probs[j]].sum() for j in differ.nonzero().flatten()]) / probs.sum()
            assert int(differ.sum()) <= 2 and bool(((above - o["p"]).abs() < 1e-6).all()), (r, o, above)
            want = torch.where(differ, got[r], want)
        assert torch.equal(torch.isinf(got[r]), torch.isinf(want)), (r, o, int(differ.sum()))
        keep = ~torch.isinf(want)
        close(got[r][keep], want[keep], 1e-5, 1e-5, what=f"kept logits of row {r}")
    again = _filter(ops, x, options, ids, in_place=True)
    assert torch.equal(torch.nan_to_num(again, neginf=-1e30), torch.nan_to_num(got, neginf=-1e30)), "in place, and the same bits twice"


@pytest.mark.parametrize("V,shift", [(3, 0), (1000, 0), (1027, 0), (8192, 0), (33001, 0), (33004, 1), (151936, 0), (262144, 0)])
def test_draw_top_k_gives_what_the_filters_and_the_draw_give(ops, V, shift):
    """The one path against the two kernels it stands for, token by token: k from 1 to the largest, one value in many places, rows of
    -inf but for a few, infinities and NaN, penalties with tokens outside the row, u at both ends, rows whose memory begins
    `shift` entries into a 16-byte line."""
    top = min(ops.DRAW_TOP_K_MAX, V - 1)
    ks = sorted({1, min(2, top), min(50, top), min(257, top), top})
    options = [dict(k=k, **o) for k in ks for o in (dict(), dict(T=0.7, p=0.9), dict(mp=0.05), dict(T=0.0, p=0.5),
                                                    dict(T=1.5, p=0.8, mp=0.02, rep=1.2, pres=0.3, freq=0.1))]
    g = torch.Generator().manual_seed(V)
    kinds = []
    for i in range(len(options)):
        x = torch.randn(V, generator=g) * 2.5
        kind = i % 8
        if kind == 1:
            x = x.round()                                        # ties at every cut
        elif kind == 2:
            x = torch.full((V,), 1.5)
        elif kind == 3:
            x[torch.randperm(V, generator=g)[:V - max(1, V // 4000)]] = float("-inf")
        elif kind == 4:
            x[torch.randint(0, V, (3,), generator=g)] = float("inf")
        elif kind == 5:
            x[torch.randint(0, V, (2,), generator=g)] = float("nan")
        elif kind == 6:
            x[:] = float("-inf")
            x[V - 1] = float("nan")
        kinds.append(x)
    R = len(options)
    whole = torch.empty(R * V + 4, dtype=F32, device=DEV)
    x = whole[shift:shift + R * V].view(R, V)
    x.copy_(torch.stack(kinds))
    col = lambda key, default, dt=F32: torch.tensor([o.get(key, default) for o in options], dtype=dt).to(DEV)
    ids = [torch.randint(-2, V + 3, (1 + 40 * (r % 6),), generator=g).tolist() * (1 + r % 2) for r in range(R)]
    flat = torch.tensor(sum(ids, []), dtype=I32).to(DEV)
    starts = torch.tensor([0] + torch.tensor([len(i) for i in ids]).cumsum(0).tolist(), dtype=I32).to(DEV)
    args = [col("T", 1.0), col("k", 0, I32), col("p", 1.0), col("mp", 0.0), col("rep", 1.0), col("pres", 0.0), col("freq", 0.0)]
    draw = torch.tensor([1.0 if o.get("T", 1.0) > 0 else 0.0 for o in options]).to(DEV)
    for with_ids in (True, False):
        left = torch.empty_like(x)
        counts = torch.zeros(R * V, dtype=I32, device=DEV)
        ops.filter_rows(x, left, *args, *((flat, starts, counts) if with_ids else ()))
        for u in (torch.rand(R, generator=g), torch.zeros(R), torch.full((R,), 0.99999994), torch.ones(R)):
            want, got = torch.full((R,), -1, dtype=I32, device=DEV), torch.full((R,), -2, dtype=I32, device=DEV)
            ops.sample_rows(left, draw, u.to(DEV), want)
            ops.draw_top_k(x, got, max(ks), *args, draw, u.to(DEV), *((flat, starts) if with_ids else ()))
            assert got.tolist() == want.tolist(), (V, with_ids, [(i, options[i], i % 8) for i in range(R) if got[i] != want[i]])


def test_filter_rows_counts_in_memory_of_any_content(ops):
    """The penalties' counters need not be zero, and calls on two streams from two threads give what they give one after another."""
    import threading
    from synaptix_amd.sampling import GenerationConfig, SequenceSampler, sample_batch
    V, R = 5000, 4
    x, g = rnd((R, V), 150, scale=3.0).to(DEV), torch.Generator().manual_seed(151)
    ids = torch.randint(0, 40, (R * 300,), generator=g).to(I32).to(DEV)
    starts = torch.arange(0, R * 300 + 1, 300, dtype=I32, device=DEV)
    one, off = torch.ones(R, device=DEV), torch.zeros(R, device=DEV)
    outs = []
    for counts in (torch.zeros(R * V, dtype=I32, device=DEV), torch.randint(-9, 9, (R * V,), generator=g).to(I32).to(DEV)):
        outs.append(torch.empty_like(x))
        ops.filter_rows(x, outs[-1], one, off.to(I32), one, off, 1.1 * one, 0.2 * one, 0.1 * one, ids, starts, counts)
    assert torch.equal(*outs)

    cfg = GenerationConfig(temperature=0.8, top_k=40, repetition_penalty=1.3, frequency_penalty=0.2)
    rows = [rnd((8, 33000), 160 + i, scale=3.0).to(DEV) for i in range(2)]
    batches = lambda: [[SequenceSampler(cfg, list(range(50 * i, 50 * i + 400)), 7 * i + r) for r in range(8)] for i in range(2)]
    steps = lambda i, samplers: [sample_batch(rows[i], samplers) for _ in range(20)]
    want = [steps(i, b) for i, b in enumerate(batches())]
    got, side = [None, None], batches()
    torch.cuda.synchronize()

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = steps(i, side[i])
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads], [t.join() for t in threads]
    assert got == want


def _sampled_tokens(monkeypatch, ops, rows, configs, either):
    """The tokens of sample_batch over `rows` (a list of batches of logits, a step each) for samplers of these configurations, on the
    route that its rule picks (either: on the two kernels whatever it picks), and how often ops.draw_top_k ran."""
    from synaptix_amd.sampling import SequenceSampler, sample_batch, sampler
    calls, draw = [], ops.draw_top_k
    with monkeypatch.context() as m:
        m.setattr(ops, "draw_top_k", lambda *a: (calls.append(1), draw(*a))[1])
        if either:
            m.setattr(sampler, "_shared_top_k", lambda *a: 0)
        samplers = [SequenceSampler(c, list(range(30 * i, 30 * i + 40)) * 3, 11 * i) for i, c in enumerate(configs)]
        return [sample_batch(x, samplers) for x in rows], len(calls)


_MIXED = [dict(temperature=0.7, top_p=0.9, repetition_penalty=1.3), dict(temperature=1.4, min_p=0.05, presence_penalty=0.7),
          dict(temperature=0.0, frequency_penalty=0.4), dict(temperature=0.9, top_p=0.6, min_p=0.02, frequency_penalty=-0.3, repeat_last_n=25),
          dict(temperature=1.0), dict(temperature=0.0, top_p=0.3, repetition_penalty=1.2, presence_penalty=-0.5, repeat_last_n=7),
          dict(temperature=1.0, top_p=0.0), dict(temperature=0.8, top_p=1.5, min_p=1.0), dict(temperature=1e-30, top_p=0.9),
          dict(temperature=50.0, top_p=0.97, min_p=-1.0, repetition_penalty=0.5), dict(temperature=0.0, repetition_penalty=1e-3, presence_penalty=1e30)]


@pytest.mark.parametrize("V", [32768, 33001, 151936])
def test_sample_batch_gives_the_same_tokens_over_slices_and_by_whole_rows(ops, monkeypatch, V):
    """Rows that differ in every option (a column handed over as another would show), with tokens that are penalised again in later steps;
    no row drawn from; a row without top-k or with one too large, which takes the batch to whole rows; sixty rows."""
    from synaptix_amd.sampling import GenerationConfig
    ks = [50, 1, 7, 128, 3, 64, 20, 5, 2, 100, 9]
    mixed = [GenerationConfig(top_k=k, **o) for k, o in zip(ks, _MIXED)]
    greedy = [GenerationConfig(top_k=k, **dict(o, temperature=0.0)) for k, o in zip(ks, _MIXED)]
    for n, (configs, routed) in enumerate([(mixed, True), (greedy, True), (mixed * 6, True),
                                           (mixed[:3] + [GenerationConfig(temperature=0.9, top_p=0.8)], False),
                                           ([GenerationConfig(top_k=min(V // 128, 512), **o) for o in _MIXED], True),
                                           ([GenerationConfig(top_k=min(V // 128, 512) + 1, **o) for o in _MIXED], False),
                                           ([GenerationConfig(top_k=V // 256, **dict(o, temperature=0.0)) for o in _MIXED], V // 256 <= 512),
                                           ([GenerationConfig(top_k=V // 256 + 1, **dict(o, temperature=0.0)) for o in _MIXED], False)]):
        rows = [rnd((len(configs), V), 170 + 10 * n + i, scale=2.5).to(DEV) for i in range(4)]
        rows[1] = rows[1].round()
        got, calls = _sampled_tokens(monkeypatch, ops, rows, configs, False)
        want, none = _sampled_tokens(monkeypatch, ops, rows, configs, True)
        assert got == want and calls == (len(rows) if routed else 0) and none == 0, n


@pytest.mark.parametrize("route", ["slices", "whole rows"])
def test_sample_batch_from_two_threads_on_two_streams(ops, monkeypatch, route):
    """Calls that may be under way at once, on each route, give what the two kernels give one call after another."""
    import threading
    from synaptix_amd.sampling import GenerationConfig, sampler
    cfg = GenerationConfig(temperature=0.8, top_k=40, top_p=0.9, repetition_penalty=1.3, frequency_penalty=0.2)
    rows = [[rnd((8, 33000), 180 + i, scale=3.0).to(DEV)] * 20 for i in range(2)]
    want = [_sampled_tokens(monkeypatch, ops, r, [cfg] * 8, True)[0] for r in rows]
    if route == "whole rows":
        monkeypatch.setattr(sampler, "_shared_top_k", lambda *a: 0)
    from synaptix_amd.sampling import SequenceSampler, sample_batch
    side = [[SequenceSampler(cfg, list(range(30 * i, 30 * i + 40)) * 3, 11 * i) for i in range(8)] for _ in range(2)]
    got = [None, None]
    torch.cuda.synchronize()

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            got[i] = [sample_batch(x, side[i]) for x in rows[i]]
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    [t.start() for t in threads], [t.join() for t in threads]
    assert got == want


def test_filter_rows_with_equal_values(ops):
    """Equal values at the k-th place and at the boundary of the probability mass: of equal entries the first in
    index order stay, so that top-k keeps exactly k; rows of one value only; rows that are -inf but for a few."""
    V = 5000
    g = torch.Generator().manual_seed(3)
    coarse = torch.randint(-4, 5, (V,), generator=g).float()              # nine values, hundreds of each
    flat = torch.full((V,), 1.5)
    few = torch.full((V,), float("-inf"))
    few[[7, 4000, 123]] = torch.tensor([2.0, 1.0, 2.0])
    x = torch.stack([coarse, coarse, coarse, flat, flat, few, few, coarse])
    options = [dict(k=50), dict(k=900), dict(p=0.6), dict(k=3), dict(p=0.5), dict(k=2), dict(p=0.7), dict(k=700, p=0.8, mp=0.2)]
    got = _filter(ops, x, options)

    def first_k(row, k):
        order = torch.argsort(row, descending=True, stable=True)
        keep = torch.zeros(V, dtype=torch.bool)
        keep[order[:k]] = True
        return keep

    def first_by_mass(row, p):
        probs = torch.exp(row.double() - row.max().double())
        order = torch.argsort(probs, descending=True, stable=True)
        sp = probs[order]
        before = torch.cumsum(sp, 0) - sp
        keep = torch.zeros(V, dtype=torch.bool)
        keep[order[(before <= p * probs.sum()) & torch.isfinite(row[order])]] = True
        return keep

    kept = ~torch.isinf(got)
    assert torch.equal(kept[0], first_k(coarse, 50)) and int(kept[0].sum()) == 50
    assert torch.equal(kept[1], first_k(coarse, 900)) and int(kept[1].sum()) == 900
    assert torch.equal(kept[2], first_by_mass(coarse, 0.6))
    assert kept[3].nonzero().flatten().tolist() == [0, 1, 2]
    assert torch.equal(kept[4], first_by_mass(flat, 0.5)) and int(kept[4].sum()) == V // 2 + 1
    assert kept[5].nonzero().flatten().tolist() == [7, 123]
    assert kept[6].nonzero().flatten().tolist() == [7, 123]            # 2/(2e^2+e) of the mass before the second, 0.84 before the third
    both = first_k(coarse, 700)
    row = torch.where(both, coarse, torch.full_like(coarse, float("-inf")))
    both &= first_by_mass(row, 0.8)
    both &= torch.exp(coarse - coarse.max()) >= 0.2
    assert torch.equal(kept[7], both)
    assert torch.equal(got[kept], x[kept])                                # what stays is untouched


def test_filter_rows_at_the_vocabulary_of_the_large_models(ops):
    """151,936 logits a row, as the models' output head gives them; a sampled token after the filters lies among
    the entries that were kept."""
    import plain_qwen3 as P
    V = 151936
    x = rnd((3, V), 95, scale=2.5)
    options = [dict(T=0.7, k=50, p=0.9), dict(p=0.95, mp=0.001), dict(T=0.9, k=2000, rep=1.1)]
    ids = [list(range(100, 400)) * 2, [], [5, 5, 5, 9]]
    got = _filter(ops, x, options, ids)
    for r, o in enumerate(options):
        want = _plain_filter(x[r], o, ids[r])
        assert torch.equal(torch.isinf(got[r]), torch.isinf(want)), (r, int((torch.isinf(got[r]) != torch.isinf(want)).sum()))
    out = torch.empty(3, dtype=I32, device=DEV)
    ops.sample_rows(got.to(DEV), torch.ones(3).to(DEV), torch.tensor([0.3, 0.999, 0.0]).to(DEV), out)
    for r, t in enumerate(out.cpu().tolist()):
        assert math.isfinite(float(got[r, t]))


def test_measured_ceilings_are_plausible(ops):
    """The two probes run and report rates of the right order for this kind of machine."""
    read_gbs, mfma_tflops = ops.measure_ceilings(DEV, read_bytes=1 << 28, repeats=2)
    assert 500 < read_gbs < 8000 * 1.05, read_gbs          # below the HBM peak, far above PCIe
    assert 100 < mfma_tflops < 2500 * 1.05, mfma_tflops    # below the bf16 peak


def test_stream_scope_holds_the_stream_that_is_current_when_it_opens(ops):
    """Inside a scope kernels go to the stream that was current at its start; a scope opened under another
    stream takes that one; leaving restores what was held before."""
    def held():
        return ops._stream().value or 0      # the default stream is the null handle

    main = torch.cuda.current_stream().cuda_stream
    side = torch.cuda.Stream()
    assert held() == main
    with ops.stream_scope():
        assert held() == main
        with torch.cuda.stream(side):
            assert held() == main          # the scope's stream, not torch's current one
            with ops.stream_scope():
                assert held() == side.cuda_stream
                x, gain = rnd((3, 64), 50).to(DEV), torch.ones(64, device=DEV)
                out = torch.empty((3, 64), device=DEV)
                ops.rmsnorm_rows(x, gain, 1e-6, out)    # launched on the side stream
            assert held() == main
        side.synchronize()
        want = torch.empty((3, 64))
        ref.rmsnorm_rows(x.cpu(), gain.cpu(), 1e-6, want)
        close(out, want, 1e-5, what="launched under a nested scope")
    assert held() == main


@pytest.mark.parametrize("rows", [1, 9])
def test_tokens_reach_pinned_memory_as_they_reach_the_device(ops, rows):
    """sample_rows into pinned host memory, launched and replayed from a graph with new logits: what the device gets; plain host memory is refused."""
    x = rnd((rows, 3000), 61).to(DEV)
    want, got = torch.empty(rows, dtype=I32, device=DEV), torch.full((rows,), -1, dtype=I32, pin_memory=True)
    t, u = torch.full((rows,), 0.7, device=DEV), torch.rand(rows, generator=torch.Generator().manual_seed(2)).to(DEV)
    ops.sample_rows(x, t, u, want)
    ops.sample_rows(x, t, u, got)
    torch.cuda.synchronize()
    assert torch.equal(got, want.cpu())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.sample_rows(x, t, u, got)
    for i in range(4):
        x.copy_(rnd((rows, 3000), 70 + i))
        ops.sample_rows(x, t, u, want)
        graph.replay()
        torch.cuda.current_stream().synchronize()
        assert torch.equal(got, want.cpu()), i
    for bad in (torch.empty(rows, dtype=I32), torch.empty(rows + 1, dtype=I32, pin_memory=True), torch.empty(rows, dtype=torch.int64, pin_memory=True)):
        with pytest.raises(ops.KernelError):
            ops.sample_rows(x, t, u, bad)


@pytest.mark.parametrize("M", [512, 513, 700, 1729, 2051])
@pytest.mark.parametrize("N,K", [(1024, 1024), (4096, 4096), (2560, 4096), (2576, 1152), (48, 2048), (5120, 512)])
def test_products_of_many_rows_add_to_the_residual_rows_what_the_norm_would(M, N, K):
    """One product that adds its sums to the rows against the product and the norm that adds: the same sums, added once, so the same bits
    wherever K is not cut; rows beyond M and the rows' neighbours in memory stay as they are.  All tiles that the sizes take."""
    from synaptix_amd.kernels import ops
    from synaptix_amd.parts import RmsNorm
    from synaptix_amd.parts.linear import DeferredProduct, Matrix, deferred_product, linear
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn((M, K), generator=g, device=DEV).bfloat16()
    w = Matrix((0.02 * torch.randn((N, K), generator=g, device=DEV)).bfloat16())
    room = torch.randn((M + 2, N), generator=g, device=DEV)
    before = room.clone()
    assert ops.gemm_adds(M, N, K) and not ops.gemm_adds(ops.ADDS_MIN_ROWS - 1, N, K)
    ops.gemm_add(x, w.packed, room[1:-1])
    want = before[1:-1] + linear(x, w, torch.float32)
    same_tile = ops.gemm_slices(M, N, K, torch.bfloat16) == 1
    if same_tile:
        assert torch.equal(room[1:-1], want)
    # (else the plain product may go through other tiles: K / 32 roundings of the sums' size in another order)
    assert float((room[1:-1] - want).abs().max()) <= K / 32 * 2.0 ** -23 * float((want - before[1:-1]).abs().max()) + 2.0 ** -23 * float(want.abs().max())
    assert torch.equal(room[0], before[0]) and torch.equal(room[-1], before[-1])
    # through the norm, which takes the product that has not been run; with rows picked it runs it and leaves the residual alone
    norm = RmsNorm("n", N, 1e-6)
    norm.gain = (1 + 0.1 * torch.randn((N,), generator=g, device=DEV)).bfloat16()
    delta = deferred_product(x, w)
    picked = torch.tensor([M - 1, 0, 5], dtype=torch.int32, device=DEV)
    for rows in (picked, None):
        resid = [before[1:-1].clone() for _ in range(2)]
        got = norm.add_apply(resid[0], delta, torch.bfloat16, rows=rows)
        ref = norm.add_apply(resid[1], linear(x, w, torch.float32), torch.bfloat16, rows=rows)
        if same_tile:
            assert isinstance(delta, DeferredProduct) and delta.many and torch.equal(got, ref) and torch.equal(resid[0], resid[1])
        assert rows is None or torch.equal(resid[0], before[1:-1])
