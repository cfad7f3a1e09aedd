"""Each kernel alone against a plain float64 / torch reference of the same op, at sizes
other than the engine's tests use (head sizes in steps of 16, widths and vocabularies that
are no power of two, many heads and groups)."""
import ctypes
import importlib
import math
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import plain_model as pm

pytestmark = pytest.mark.gpu
K = importlib.import_module("daisi-llogos_amd.ops.kernels")
DEV = "cuda:0"
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}
RT = {"float32": 2e-6, "bfloat16": 1e-2}        # relative to the result's scale


def _t(a, dtype=torch.float32):
    return torch.tensor(np.asarray(a), dtype=dtype, device=DEV)


def _np(t):
    return t.detach().cpu().double().numpy()


def _close(got, want, dtype, scale=None):
    want = np.asarray(want, dtype=np.float64)
    scale = scale if scale is not None else max(1e-6, np.abs(want).max())
    err = np.abs(_np(got) - want).max() / scale
    assert err <= RT[dtype], f"relative error {err:.3e} > {RT[dtype]}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_embed(dtype):
    rng = np.random.default_rng(0)
    table = _t(rng.standard_normal((331, 200)), DT[dtype])
    ids = _t([0, 330, 7, 7, 129], torch.int32)
    out = K.embed(table, ids)
    assert out.dtype == torch.float32 and torch.equal(out, table.float()[ids.long()])


@pytest.mark.parametrize("table_dtype,dtype", [("bfloat16", "bfloat16"), ("float32", "float32"), ("bfloat16", "float32")])
@pytest.mark.parametrize("T,H,half,scale", [(1, 2048, 32, 1.0), (5, 200, 7, 1.5), (64, 4100, 64, 1.0), (300, 1028, 16, 0.5), (3, 8200, 0, 1.0), (2, 16384, 1, 1.0)])
def test_step_open_is_embedding_norm_and_rotary_table(table_dtype, dtype, T, H, half, scale):
    """The bits of the three kernels, whose layout of a row it keeps."""
    rng = np.random.default_rng(T + H)
    table, w = _t(rng.standard_normal((97, H)), DT[table_dtype]), _t(1 + 0.1 * rng.standard_normal(H))
    ids, pos = _t(rng.integers(0, 97, T), torch.int32), _t(rng.integers(0, 100000, T), torch.int32)
    freqs = _t(rng.random(half), torch.float64) if half else None
    cs = torch.full((T, half, 2), float("nan"), device=DEV) if half else None
    x = torch.full((T, H), float("nan"), device=DEV)
    assert K.step_opens(table, w)
    rows = K.rmsnorm(x, w, 1e-5, DT[dtype], opening=K.Opening(table, ids, scale, pos, SimpleNamespace(inv_freq=freqs, amplitude=1.25), cs))
    want = K.embed(table, ids, scale)
    assert torch.equal(x, want) and torch.equal(rows, K.rmsnorm(want, w, 1e-5, DT[dtype]))
    assert not half or torch.equal(cs, K.rope_table(pos, freqs, 1.25))


@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1024, 1029, 20000])
@pytest.mark.parametrize("shift", [0, 1])
def test_words_from_pinned_memory(n, shift):
    """By fours where both sides are aligned to 16 bytes, one by one elsewhere and at the end; nothing behind the last word is touched."""
    host = torch.randint(-2 ** 31, 2 ** 31 - 1, (n + shift,), dtype=torch.int32).pin_memory()
    dst = torch.full((n + 9,), 7, dtype=torch.int32, device=DEV)
    code = K._lib().llogos_copy_words(ctypes.c_void_p(dst.data_ptr()), ctypes.c_void_p(host.data_ptr() + 4 * shift), n, K._stream())
    torch.cuda.synchronize()
    assert code == 0 and torch.equal(dst[:n].cpu(), host[shift:]) and (dst[n:] == 7).all()
    assert K._lib().llogos_copy_words(ctypes.c_void_p(dst.data_ptr()), ctypes.c_void_p(host.data_ptr()), 0, K._stream()) == -1


@pytest.mark.parametrize("H", [30, 16388])
def test_step_open_leaves_other_widths_to_the_kernels_apart(H):
    assert not K.step_opens(_t(np.ones((3, H))), _t(np.ones(H)))
    with pytest.raises(K.KernelError):
        K.rmsnorm(torch.empty(1, H, device=DEV), _t(np.ones(H)), 1e-5, torch.float32, opening=K.Opening(_t(np.ones((3, H))), _t([1], torch.int32)))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H", [80, 1000, 4100])
def test_rmsnorm(dtype, H):
    rng = np.random.default_rng(1)
    x = rng.standard_normal((7, H)) * 3
    d = rng.standard_normal((7, H))
    w = 1 + 0.1 * rng.standard_normal(H)
    xd, dd, wd = _t(x), _t(d, DT[dtype]), _t(w)
    want = pm.rms_norm(x, w, 1e-5)
    _close(K.rmsnorm(xd, wd, 1e-5, DT[dtype]), want, dtype)
    # with a pending delta: the sum is written back in float32 and the norm is of the sum
    xs = x + _np(dd)
    out = K.rmsnorm(xd, wd, 1e-5, DT[dtype], delta=dd)
    assert np.abs(_np(xd) - xs).max() < 1e-6
    _close(out, pm.rms_norm(xs, w, 1e-5), dtype)
    # selected rows, no write back
    x2 = _t(x)
    rows = _t([6, 0, 3], torch.int32)
    out = K.rmsnorm(x2, wd, 1e-5, DT[dtype], delta=dd, rows=rows, write_back=False)
    assert torch.equal(x2, _t(x))
    _close(out, pm.rms_norm(xs[[6, 0, 3]], w, 1e-5), dtype)
    z = K.rmsnorm(torch.zeros(2, H, device=DEV), wd, 1e-6, DT[dtype])
    assert torch.count_nonzero(z) == 0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("M,N,K_", [(1, 331, 80), (5, 96, 1000), (70, 130, 67), (200, 257, 129)])
def test_gemm(dtype, M, N, K_):
    rng = np.random.default_rng(2)
    a = _t(rng.standard_normal((M, K_)), DT[dtype])
    w = _t(rng.standard_normal((N, K_)) * 0.1, DT[dtype])
    b = _t(rng.standard_normal(N))
    want = pm.linear(_np(a), _np(w), _np(b))
    _close(K.gemm(a, w, b, DT[dtype]), want, dtype)
    _close(K.gemm(a, w, None, torch.float32), pm.linear(_np(a), _np(w)), "float32" if dtype == "float32" else dtype)
    # a view with a row stride (the first columns of a wider buffer) and the first rows of w
    wide = _t(rng.standard_normal((M, K_ + 13)), DT[dtype])
    _close(K.gemm(wide[:, :K_], w[:N // 2], None, DT[dtype]), pm.linear(_np(wide)[:, :K_], _np(w)[:N // 2]), dtype)
    # reference vector (tests/Daisi.Llogos.Tests/Cpu/MathOpsTests.cs:10-28)
    o = K.gemm(_t([[1, 2, 3], [4, 5, 6]], DT[dtype]), _t([[7, 9, 11], [8, 10, 12]], DT[dtype]), None, torch.float32)
    assert _np(o).tolist() == [[58, 64], [139, 154]]


@pytest.mark.parametrize("M,N,K_", [(1, 4096, 4096), (8, 331, 1000), (16, 100, 72), (17, 4096, 14336), (64, 257, 2048),
                                    (33, 6144, 4096), (5, 20000, 4096), (16, 70001, 1000), (7, 1000, 5120),
                                    (9, 333, 8192), (3, 200, 6000)])
def test_gemm_few_rows_on_the_matrix_cores(M, N, K_):
    rng = np.random.default_rng(7)
    a = _t(rng.standard_normal((M, K_)), torch.bfloat16)
    w = _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    b = _t(rng.standard_normal(N))
    want = pm.linear(_np(a), _np(w))
    scale = np.abs(want).max()
    for kernel, rbs in ((K.gemm_skinny_bf16, (1, 2, 4)), (K.gemm_skinny_lds_bf16, (1, 2))):
        for splits in (1, 2, 5, 8):
            for rb in rbs:
                out = kernel(a, w, None, torch.float32, splits, rb)
                assert out is not None and out.dtype == torch.float32 and out.shape[1:] == (M, N)
                assert np.abs(_np(out).sum(0) - want).max() <= 2e-6 * scale * math.sqrt(K_)
    if M <= 16 and K_ <= 8192:                                          # activations held in registers
        for strips in (1, 3, 8):
            out = K.gemm_skinny_stationary_bf16(a, w, b, torch.float32, strips)
            assert out is not None and np.abs(_np(out)[0] - (want + _np(b))).max() <= 2e-6 * scale * math.sqrt(K_)
    # silu(gate) * up made inside the product, from a bfloat16 row or from float32 partial sums
    if K_ % 16 == 0:
        I = K_ // 2
        act = pm.silu(_np(a)[:, :I]) * _np(a)[:, I:]
        act = _np(_t(act, torch.bfloat16))                              # the kernel rounds it to bfloat16
        want_sw = pm.linear(act, _np(w)[:, :I])
        w_half = w[:, :I].contiguous()
        for src in (a, torch.stack([a.float() * 0.25, a.float() * 0.75])):
            out = K.gemm_skinny_lds_bf16(src, w_half, None, torch.float32, 2, 1, swiglu=True)
            assert np.abs(_np(out).sum(0) - want_sw).max() <= 2e-2 * max(1.0, np.abs(want_sw).max())
    plain = K.gemm(a, w, b, torch.bfloat16)
    assert np.abs(_np(plain) - (want + _np(b))).max() <= 1e-2 * scale
    prod = K.gemm_product(a, w, torch.bfloat16)
    assert np.abs(_np(K.sum_parts(prod, b, torch.float32)) - (want + _np(b))).max() <= (1e-2 if prod.dtype == torch.bfloat16 else 1e-5) * scale
    # a row's result does not depend on how many other rows the batch has, bit for bit among
    # batches of up to 16, of 17 to 32 and of 33 to 64 rows (the plan is made for those classes),
    # and up to rounding between them
    if M > 1:
        fewest = 1 if M <= 16 else (17 if M <= 32 else 33)
        few = K.sum_parts(K.gemm_product(a[:fewest], w, torch.bfloat16), None, torch.float32)
        many = K.sum_parts(prod, None, torch.float32)
        assert torch.equal(few, many[:fewest])
        alone = K.sum_parts(K.gemm_product(a[:1], w, torch.bfloat16), None, torch.float32)
        assert np.abs(_np(alone) - _np(many[:1])).max() <= 1e-2 * scale
    assert K.gemm_skinny_bf16(a[:, :K_ - 4], w[:, :K_ - 4].contiguous(), None, torch.float32) is None   # k % 8


@pytest.mark.parametrize("M,N,K_", [(65, 257, 2048), (96, 4096, 14336), (97, 100, 1000), (128, 5120, 17408), (111, 333, 72)])
def test_gemm_of_65_to_128_rows_on_the_matrix_cores(M, N, K_):
    """The LDS few-row product at 65 to 128 rows: every number of blocks along k and both widths
    of a wave's strip of w; a row's result is the same bit for bit for every batch of this class."""
    rng = np.random.default_rng(8)
    a = _t(rng.standard_normal((M, K_)), torch.bfloat16)
    w = _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    b = _t(rng.standard_normal(N))
    want = pm.linear(_np(a), _np(w))
    scale = np.abs(want).max()
    for splits in (1, 3, 8):
        for rb in (1, 2):
            out = K.gemm_skinny_lds_bf16(a, w, None, torch.float32, splits, rb)
            assert out is not None and out.dtype == torch.float32 and out.shape[1:] == (M, N)
            assert np.abs(_np(out).sum(0) - want).max() <= 2e-6 * scale * math.sqrt(K_)
    out = K.gemm_skinny_lds_bf16(a, w, b, torch.bfloat16, 1, 1)
    assert np.abs(_np(out)[0] - (want + _np(b))).max() <= 1e-2 * scale
    assert K.gemm_skinny_lds_bf16(torch.cat([a, a]), w, None, torch.float32, 1, 1) is None            # more than 128 rows
    assert K.gemm_skinny_lds_bf16(a.float().repeat(1, 2), w, None, torch.float32, 1, 1, swiglu=True) is None  # fused producer: 64 rows
    prod = K.gemm_product(a, w, torch.bfloat16, f32_ok=True)
    assert (prod.dim() == 3) == (K.long_inner(w) and K.lds_splits(M, N, K_) > 1)
    many = K.sum_parts(prod, None, torch.float32)
    assert np.abs(_np(many) - want).max() <= (1e-5 if prod.dtype == torch.float32 else 1e-2) * scale
    if K.long_inner(w):
        few = K.sum_parts(K.gemm_product(a[:65], w, torch.bfloat16, f32_ok=True), None, torch.float32)
        assert torch.equal(few, many[:65])


@pytest.mark.parametrize("M,N,K_", [(17, 3000, 1024), (33, 16 * 9 * 5 + 7, 2048), (64, 4096, 4096), (100, 777, 512), (128, 2048, 640)])
def test_gemm_with_operands_straight_into_lds(M, N, K_):
    """The third form of the few-row product: every height of its blocks and several numbers
    of blocks along k; its results equal the LDS few-row product's bit for bit for the same
    parts of k, whatever the height."""
    rng = np.random.default_rng(9)
    a = _t(rng.standard_normal((M, K_)), torch.bfloat16)
    w = _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    b = _t(rng.standard_normal(N))
    want = pm.linear(_np(a), _np(w))
    scale = np.abs(want).max()
    for splits in (1, 2, 5):
        same = K.gemm_skinny_lds_bf16(a, w, None, torch.float32, splits, 1)
        for strips in (2, 3, 4, 7, 9):
            out = K.gemm_strips_bf16(a, w, None, torch.float32, splits, strips)
            assert out is not None and out.shape == same.shape
            assert np.abs(_np(out).sum(0) - want).max() <= 2e-6 * scale * math.sqrt(K_)
            assert torch.equal(out, same), (splits, strips)
    out = K.gemm_strips_bf16(a, w, b, torch.bfloat16, 1, 7)
    assert np.abs(_np(out)[0] - (want + _np(b))).max() <= 1e-2 * scale
    wide = _t(rng.standard_normal((M, K_ + 24)), torch.bfloat16)              # a view with a row stride
    out = K.gemm_strips_bf16(wide[:, :K_], w, None, torch.float32, 1, 8)
    assert np.abs(_np(out)[0] - pm.linear(_np(wide)[:, :K_], _np(w))).max() <= 2e-6 * scale * math.sqrt(K_)
    assert K.gemm_strips_bf16(a[:, :K_ - 8], w[:, :K_ - 8].contiguous(), None, torch.float32, 1, 7) is None   # k % 64
    assert K.gemm_strips_bf16(a, w, None, torch.float32, 1, 10) is None                                       # too high


def test_tall_products_through_the_dispatch_take_the_third_form():
    """A matrix as tall as the Qwen3-14B gate/up projection, few columns: the plan for 17 to 64
    rows is the third form, and a row's result is the same for every batch of such a class."""
    rng = np.random.default_rng(10)
    N, K_ = 34816, 1024
    w = torch.randn((N, K_), device=DEV, dtype=torch.bfloat16, generator=torch.Generator(device=DEV).manual_seed(3)) * 0.05
    a = _t(rng.standard_normal((64, K_)), torch.bfloat16)
    assert K.skinny_plan(33, N, K_)[0] == "strips" and K.skinny_plan(64, N, K_) == K.skinny_plan(33, N, K_)
    many = K.sum_parts(K.gemm_product(a, w, torch.bfloat16, f32_ok=True), None, torch.float32)
    few = K.sum_parts(K.gemm_product(a[:33], w, torch.bfloat16, f32_ok=True), None, torch.float32)
    assert torch.equal(few, many[:33])
    want = _np(a.float() @ w.float().t())
    assert np.abs(_np(many) - want).max() <= 2e-5 * max(1.0, np.abs(want).max())
    plain = K.gemm(a, w, None, torch.float32)
    assert np.abs(_np(plain) - want).max() <= 2e-5 * max(1.0, np.abs(want).max())


def test_products_of_random_shapes_through_the_dispatch():
    """Whatever kernel and split of k the plan picks for a shape, the product is right: row
    counts up to 64 and beyond, widths and depths that are multiples of 8 and of nothing else."""
    rng = np.random.default_rng(21)
    for case in range(40):
        M = int(rng.choice([1, 2, 5, 8, 13, 16, 17, 31, 33, 64, 70, 100, 128, 130]))
        K_ = 8 * int(rng.integers(1, 1100))                                # up to 8,792
        N = int(rng.integers(1, 40000)) if case % 4 else int(rng.integers(16384, 72000))
        if case % 5 == 3:
            N = int(rng.integers(1, K_ // 2 + 2))                           # few rows of w for its length
        a = _t(rng.standard_normal((M, K_)), torch.bfloat16)
        w = torch.randn((N, K_), device=DEV, dtype=torch.bfloat16, generator=torch.Generator(device=DEV).manual_seed(case)) * 0.05
        b = _t(rng.standard_normal(N))
        want = _np(a.float() @ w.float().t())                              # float32 on the device stands in for float64 here
        scale = max(1.0, np.abs(want).max())
        prod = K.gemm_product(a, w, torch.bfloat16, f32_ok=bool(case % 2))
        got = _np(K.sum_parts(prod, b, torch.float32))
        tol = (1e-2 if prod.dtype == torch.bfloat16 else 2e-5) * scale
        assert np.abs(got - (want + _np(b))).max() <= tol, (case, M, N, K_, K.skinny_plan(M, N, K_))
        got = _np(K.gemm(a, w, b, torch.float32))
        assert np.abs(got - (want + _np(b))).max() <= 2e-5 * scale, (case, M, N, K_)


def test_prompt_products_of_random_shapes_on_packed_weights():
    """Prompts through the dispatch with a packed copy at hand: whatever the plan picks (the tiled product in one
    part or in parts of k for matrices much longer than high, the library's elsewhere), every number of stages of
    64 and every way they fall into parts, heights below one block of rows, token counts that fill no tile."""
    rng = np.random.default_rng(33)
    seen = set()
    for case in range(36):
        M = int(rng.choice([129, 130, 190, 256, 257, 300, 511, 512, 513, 700, 1024]))
        K_ = 64 * int(rng.integers(1, 40)) if case % 3 else 64 * int(rng.choice([9, 10, 11, 13, 17, 18, 19, 35]))
        N = int(rng.integers(1, max(2, K_ // 2))) if case % 2 else int(rng.integers(1, 3000))
        a = _t(rng.standard_normal((M, K_)), torch.bfloat16)
        w = torch.randn((N, K_), device=DEV, dtype=torch.bfloat16, generator=torch.Generator(device=DEV).manual_seed(case)) * 0.05
        pw = K.pack_weights(w)
        want = _np(a.float() @ w.float().t())
        scale = max(1.0, np.abs(want).max())
        plan = K.tiles_plan(M, N, K_)
        seen.add(plan)
        prod = K.gemm_product(a, w, torch.bfloat16, f32_ok=True, packed=pw)
        assert (prod.dim() == 3 and prod.shape[0] == plan[0]) if plan is not None and plan[0] > 1 else prod.shape[-2:] == (M, N)
        got = _np(K.sum_parts(prod, None, torch.float32))
        assert np.abs(got - want).max() <= (1e-2 if prod.dtype == torch.bfloat16 else 2e-5) * scale, (case, M, N, K_, plan)
        for parts in (2, 4):                                               # every split the kernel takes, whether the plan asks for it or not
            if K_ // 64 // parts >= 2:
                got = K.gemm_tiles_bf16(a, pw, None, torch.float32, parts=parts, token_tiles=int(rng.choice([0, 2, 4])))
                assert got.shape == (parts, M, N)
                assert np.abs(_np(got.sum(0)) - want).max() <= 2e-5 * scale, (case, M, N, K_, parts)
    assert {p[0] for p in seen if p is not None} >= {1, 2, 4} and None in seen        # what the cases were drawn to cover


@pytest.mark.parametrize("N,K_", [(70, 16), (2048, 8192), (17000, 1000), (33000, 2049), (66000, 530), (5, 4099), (300, 7)])
def test_float32_product_of_few_rows_is_the_tiled_product_bit_for_bit(N, K_, monkeypatch):
    """Few rows in float32 go to kernels of their own; they add in the order of the tiled kernel, so a row's
    result is the same bits whichever of them a step's row count selects, alone or beside others, and right."""
    rng = np.random.default_rng(N)
    a = _t(rng.standard_normal((40, K_)))
    w = _t(rng.standard_normal((N, K_)) * 0.05)
    b = _t(rng.standard_normal(N))
    monkeypatch.setattr(K, "F32_FORM", 6)                                  # the tiled kernel, whatever 40 rows would choose
    tiled = K.gemm_generic(a, w, b, torch.float32)
    monkeypatch.setattr(K, "F32_FORM", 0)
    want = pm.linear(_np(a), _np(w), _np(b))
    assert np.abs(_np(tiled) - want).max() <= 2e-6 * max(1.0, np.abs(want).max()) * math.sqrt(K_)
    for M in (1, 2, 3, 4, 7, 8, 9, 16, 31, 32, 40):
        few = K.gemm_generic(a[:M], w, b, torch.float32)
        assert torch.equal(few, tiled[:M]), (M, N, K_, (few - tiled[:M]).abs().max().item())
    # several tiles of rows: the same bits again
    big = torch.cat([a, _t(rng.standard_normal((160, K_)))])
    out = K.gemm_generic(big, w, b, torch.float32)
    assert torch.equal(out[:40], tiled)
    assert torch.equal(out[195:200], K.gemm_generic(big[195:200].contiguous(), w, b, torch.float32))
    wide = _t(rng.standard_normal((5, K_ + 3)))                            # rows that do not start at a multiple of 16 bytes
    few = K.gemm_generic(wide[:, :K_], w, None, torch.float32)
    many = K.gemm_generic(torch.cat([wide, wide * 0 + 1.0] * 4)[:, :K_], w, None, torch.float32)
    assert torch.equal(few, many[:5])


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("N,K_", [(1, 1), (5, 1024), (130, 1040), (3585, 2052), (6145, 1028), (8193, 1028), (40, 16), (7, 1025), (2049, 515), (16387, 33)])
def test_float32_products_of_the_fewest_rows(M, N, K_, monkeypatch):
    """The lanes' kernel, at the sizes where it takes one, two, four or eight rows of w a wave and where the few-row kernel
    serves, with k around its lanes' and waves' shares: the few-row kernel's bits."""
    rng = np.random.default_rng(N)
    a, w, b = _t(rng.standard_normal((M, K_))), _t(rng.standard_normal((N, K_)) * 0.05), _t(rng.standard_normal(N))
    got = K.gemm_generic(a, w, b, torch.float32)
    for form in (8, 1):
        monkeypatch.setattr(K, "F32_FORM", form)
        out = torch.full((M, N + 1), 7.0, device=DEV)
        assert torch.equal(K.gemm_generic(a, w, b, torch.float32, out=out[:, :N]), got), form
        assert (out[:, N:] == 7.0).all()


def test_the_generic_entry_takes_float32_throughout():
    """The library's entry for any types hands float32 operands on to the float32 product: the same bits, with and without a
    bias, into rows of a wider result."""
    rng = np.random.default_rng(2)
    for M, N, K_ in ((1, 70, 40), (33, 65, 255)):
        a, w, b = _t(rng.standard_normal((M, K_))), _t(rng.standard_normal((N, K_))), _t(rng.standard_normal(N))
        for bias in (b, None):
            out = torch.full((M, N + 3), 7.0, device=DEV)
            code = K._lib().llogos_gemm_generic(K._p(out), K.F32, K._p(a), K.F32, K._p(w), K.F32, K._p(bias), M, N, K_, K_, N + 3, K._stream())
            assert code == 0
            assert torch.equal(out[:, :N], K.gemm_generic(a, w, bias, torch.float32)) and (out[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K_", [(17, 1, 32), (48, 64, 256), (49, 65, 288), (79, 130, 64), (81, 63, 544), (161, 200, 2048), (321, 33, 224)])
def test_float32_ring_gives_the_bits_of_the_tiles(M, N, K_, monkeypatch):
    """The ring's tiles at remainders of their rows and columns, one stage of k, groups of 256 k that are whole and that are not, rows of a
    and of the result that are wider than their values, a bias, values that are no number in one row and one matrix row."""
    rng = np.random.default_rng(M + K_)
    wide, w, b = _t(rng.standard_normal((M, K_ + 8))), _t(rng.standard_normal((N, K_)) * 0.1), _t(rng.standard_normal(N))
    for special in (False, True):
        if special:
            wide[M // 2, 5], wide[M - 1, K_ - 1], w[N // 2, K_ // 2] = float("inf"), float("nan"), float("-inf")
        for a, out in ((wide[:, :K_], torch.zeros((M, N + 3), device=DEV)[:, :N]), (wide[:, :K_].contiguous(), torch.zeros((M, N), device=DEV))):
            for bias in (None, b):
                monkeypatch.setattr(K, "F32_FORM", 6)
                want = K.gemm_generic(a, w, bias, torch.float32, out=torch.zeros_like(out))
                for form in range(9, 13):
                    monkeypatch.setattr(K, "F32_FORM", form)
                    got = K.gemm_generic(a, w, bias, torch.float32, out=out)
                    assert torch.equal(got.view(torch.int32) if got.is_contiguous() else got.contiguous().view(torch.int32),
                                       want.contiguous().view(torch.int32)) or (special and torch.allclose(got, want, rtol=0, atol=0, equal_nan=True)), form
                monkeypatch.setattr(K, "F32_FORM", 0)
                assert special or torch.equal(K.gemm_generic(a, w, bias, torch.float32, out=out), want)


@pytest.mark.parametrize("M,N,K_", [(1, 16, 16), (17, 33, 40), (33, 70, 272), (64, 129, 4112), (65, 31, 255), (130, 66, 2049), (200, 250, 513)])
def test_float32_product_gives_the_same_bits_in_every_form(M, N, K_, monkeypatch):
    """The forms of the float32 product (few rows in three heights of blocks, tiles in three sizes, pairs of rows) at remainders of
    tiles, of blocks of 16 and of 256 k and of 16 bytes: one result, and right (a sum is at most 16 + 16 + K / 256
    additions deep)."""
    rng = np.random.default_rng(M)
    a, w, b = _t(rng.standard_normal((M, K_))), _t(rng.standard_normal((N, K_)) * 0.05), _t(rng.standard_normal(N))
    chosen = K.gemm_generic(a, w, b, torch.float32)
    bound = 2.0 ** -24 * (34 + K_ / 256) * (_np(a.abs()) @ _np(w.abs()).T + np.abs(_np(b)))
    assert (np.abs(_np(chosen) - pm.linear(_np(a), _np(w), _np(b))) <= bound).all()
    for form in range(1, 9):
        monkeypatch.setattr(K, "F32_FORM", form)
        out = torch.full((M, N + 3), 7.0, device=DEV)
        assert torch.equal(K.gemm_generic(a, w, b, torch.float32, out=out[:, :N]), chosen), form
        assert (out[:, N:] == 7.0).all()


def test_rope_table_is_double_precision():
    pos = _t([0, 1, 4095, 100000], torch.int32)
    f = pm.rope_frequencies(64, 5e5)
    cs = _np(K.rope_table(pos, _t(f, torch.float64)))
    ang = np.array([0, 1, 4095, 100000])[:, None] * f[None, :]
    assert np.abs(cs[..., 0] - np.cos(ang)).max() < 1e-7 and np.abs(cs[..., 1] - np.sin(ang)).max() < 1e-7


def _page_index(hd):
    """(keys, values): index tensors [64, hd] of where (token, dimension) lies in one kv head's part
    of a page, by the cache's own rule (cache/pages.py)."""
    pages = importlib.import_module("daisi-llogos_amd.cache.pages")
    ki, vi = pages.page_offsets(hd)
    return torch.tensor(ki, device=DEV), torch.tensor(vi, device=DEV)


def _pages(n_seqs, max_len, rng):
    """A shuffled page table: sequences' pages lie anywhere in the pool."""
    per = (max_len + 63) // 64
    ids = rng.permutation(n_seqs * per + 3)[:n_seqs * per].reshape(n_seqs, per)
    return ids.astype(np.int32), n_seqs * per + 3


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("nh,nkv,hd,rot,pairing,norm", [
    (4, 2, 16, 16, 0, False), (6, 1, 32, 32, 0, True), (5, 5, 48, 24, 0, True), (8, 2, 80, 80, 1, False),
    (3, 3, 128, 64, 1, True), (2, 1, 256, 256, 0, False), (8, 2, 128, 128, 0, True), (5, 5, 128, 128, 0, False),
    (8, 2, 128, 128, 1, False), (5, 1, 128, 4, 1, True), (4, 1, 128, 30, 1, False)])
@pytest.mark.parametrize("lens,new", [([70, 3], [5, 3]), ([70, 30], [40, 27]), ([70, 69], [69, 60])])
def test_qk_rope_cache(dtype, nh, nkv, hd, rot, pairing, norm, lens, new):
    """Two sequences; this step brings the last `new` tokens of each: a few tokens, and runs
    that cross a page's end and start in the middle of one."""
    rng = np.random.default_rng(3)
    T = sum(new)
    tok_seq = np.repeat(np.arange(2), new).astype(np.int32)
    tok_pos = np.concatenate([np.arange(l - n, l) for l, n in zip(lens, new)]).astype(np.int32)
    table, n_pages = _pages(2, 70, rng)
    width = (nh + 2 * nkv) * hd
    qkv = _t(rng.standard_normal((T, width)), DT[dtype])
    bias = _t(rng.standard_normal(width)) if norm else None              # bias and norm together: bias first
    orig = _np(qkv) + (_np(bias) if bias is not None else 0)
    qw = 1 + 0.1 * rng.standard_normal(hd)
    kw = 1 + 0.1 * rng.standard_normal(hd)
    f = pm.rope_frequencies(rot, 1e4)
    cs = K.rope_table(_t(tok_pos, torch.int32), _t(f, torch.float64))
    kp = torch.zeros((n_pages, nkv, 64 * hd), dtype=DT[dtype], device=DEV)
    vp = torch.zeros((n_pages, nkv, 64 * hd), dtype=DT[dtype], device=DEV)
    args = (nh, nkv, hd, rot, pairing, _t(qw) if norm else None, _t(kw) if norm else None, 1e-5,
            cs, kp, vp, _t(table, torch.int32), _t(tok_seq, torch.int32), _t(tok_pos, torch.int32))
    q_out = K.qk_rope_cache(qkv, bias, DT[dtype], *args)
    # the same projection as three float32 partial sums gives the same result
    third = qkv.float() / 4
    q_parts = K.qk_rope_cache(torch.stack([third, 2 * third, third]), bias, DT[dtype], *args)
    assert torch.equal(q_parts, q_out)
    q, k, v = orig[:, :nh * hd], orig[:, nh * hd:(nh + nkv) * hd], orig[:, (nh + nkv) * hd:]
    if norm:
        q = pm.per_head_rms_norm(q, qw, nh, hd, 1e-5)
        k = pm.per_head_rms_norm(k, kw, nkv, hd, 1e-5)
    rope = pm.rope_split_half if pairing == 0 else pm.rope_interleaved
    q, k = rope(q, tok_pos, nh, hd, f), rope(k, tok_pos, nkv, hd, f)
    _close(q_out, q, dtype)
    kc, vc = _np(kp), _np(vp)
    ki, vi = (_np(i).astype(np.int64) for i in _page_index(hd))
    for t in range(T):
        page = table[tok_seq[t], tok_pos[t] // 64]
        got_k = kc[page][:, ki[tok_pos[t] % 64]].reshape(-1)
        got_v = vc[page][:, vi[tok_pos[t] % 64]].reshape(-1)
        assert np.abs(got_k - k[t]).max() <= RT[dtype] * max(1, np.abs(k).max())
        assert np.abs(got_v - v[t]).max() <= RT[dtype] * max(1, np.abs(v).max())
    assert np.count_nonzero(kc) == T * nkv * hd and np.count_nonzero(vc) == T * nkv * hd   # nothing else was written


def _attention_case(dtype, nh, nkv, hd, lens, new, window=0, sinks=0, seed=4, scale_q=1.0):
    """Fills a paged cache with random keys and values for sequences of `lens` positions, of
    which the last `new` are this step's queries; returns the kernel's and the plain result."""
    rng = np.random.default_rng(seed)
    B, T = len(lens), sum(new)
    table, n_pages = _pages(B, max(lens), rng)
    kp = torch.zeros((n_pages, nkv, 64 * hd), dtype=DT[dtype], device=DEV)
    vp = torch.zeros((n_pages, nkv, 64 * hd), dtype=DT[dtype], device=DEV)
    ki, vi = _page_index(hd)
    ks = [rng.standard_normal((l, nkv * hd)) for l in lens]
    vs = [rng.standard_normal((l, nkv * hd)) for l in lens]
    for b in range(B):
        kb, vb = _t(ks[b], DT[dtype]), _t(vs[b], DT[dtype])
        ks[b], vs[b] = _np(kb), _np(vb)
        for p0 in range(0, lens[b], 64):                                # page by page
            n = min(64, lens[b] - p0)
            kp[table[b, p0 // 64]][:, ki[:n]] = kb[p0:p0 + n].view(n, nkv, hd).permute(1, 0, 2)
            vp[table[b, p0 // 64]][:, vi[:n]] = vb[p0:p0 + n].view(n, nkv, hd).permute(1, 0, 2)
    stride = nh * hd + 24                                               # queries sit in a wider row
    qbuf = _t(rng.standard_normal((T, stride)) * scale_q, DT[dtype])
    tok_seq = np.repeat(np.arange(B), new).astype(np.int32)
    tok_pos = np.concatenate([np.arange(l - n, l) for l, n in zip(lens, new)]).astype(np.int32)
    return dict(q=qbuf, stride=stride, kp=kp, vp=vp, ki=ki, vi=vi, table=_t(table, torch.int32), ks=ks, vs=vs,
                tok_seq=tok_seq, tok_pos=tok_pos, new=new, lens=lens)


def _plain_attention(c, nh, nkv, hd, window=0, sinks=0, scale=None):
    outs = []
    q = _np(c["q"])[:, :nh * hd]
    o = 0
    for b, (l, n) in enumerate(zip(c["lens"], c["new"])):
        full_q = np.zeros((l, nh * hd))
        full_q[l - n:] = q[o:o + n]
        outs.append(pm.attention(full_q, c["ks"][b], c["vs"][b], nh, nkv, hd, scale=scale, window=window,
                                 sinks=sinks, rows=range(l - n, l))[l - n:])
        o += n
    return np.concatenate(outs)


ATTN_SHAPES = [(4, 2, 16), (6, 1, 32), (5, 5, 48), (8, 2, 64), (6, 3, 80), (4, 1, 96), (7, 7, 112),
               (32, 8, 128), (3, 1, 256)]


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("nh,nkv,hd", ATTN_SHAPES)
def test_attention_whole_prompts_and_single_tokens(dtype, nh, nkv, hd):
    for lens, new in (([70, 3, 130], [70, 3, 130]),                     # whole prompts
                      ([300, 1, 65, 64], [1, 1, 1, 1]),                 # one token each
                      ([200, 90], [72, 5])):                            # continued prompts
        c = _attention_case(dtype, nh, nkv, hd, lens, new)
        ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32),
                                   is_decode=max(new) == 1, max_context=max(lens), batch=len(lens),
                                   n_tokens=sum(new), cu_seqlens=np.concatenate([[0], np.cumsum(new)]).tolist(),
                                   cu_dev=_t(np.concatenate([[0], np.cumsum(new)]), torch.int32),
                                   starts=[l - n for l, n in zip(lens, new)], shared={}))()
        out = K.attention(ctx, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd))
        _close(out, _plain_attention(c, nh, nkv, hd), dtype)


@pytest.mark.parametrize("window,sinks", [(0, 0), (100, 70)])
@pytest.mark.parametrize("nh,nkv,hd", [(6, 2, 64), (20, 1, 64), (3, 3, 128), (10, 2, 128)])
def test_float32_attention_of_a_token_alone_and_in_a_prompt(nh, nkv, hd, window, sinks):
    """On the matrix cores' 32-bit instruction: a token's result is the same bits alone and in a prompt (groups that fill
    no tile of 16 rows and more than one), what lies behind a sequence's end and in pages given back is never read, and a
    value that is no number reaches only the tokens that see it."""
    lens, new = [300, 65, 5], [300, 30, 1]
    c = _attention_case("float32", nh, nkv, hd, lens, new)
    table = c["table"].clone()
    for b, n in enumerate(lens):                                        # NaN behind the end of a sequence's last page
        page = int(table[b, (n - 1) // 64])
        c["kp"][page][:, c["ki"][n - 64 * ((n - 1) // 64):]] = float("nan")
        c["vp"][page][:, c["vi"][n - 64 * ((n - 1) // 64):]] = float("nan")
        table[b, (n - 1) // 64 + 1:] = 10 ** 6                           # a page of no pool
    cu = np.concatenate([[0], np.cumsum(new)])
    pos = _t(c["tok_pos"], torch.int32)
    ctx = type("Ctx", (), dict(tok_pos=pos, is_decode=False, batch=3, n_tokens=sum(new), cu_seqlens=cu.tolist(), cu_dev=_t(cu, torch.int32)))()
    call = lambda x, q, t: K.attention_f32(x, q, c["stride"], c["kp"], c["vp"], t, nh, nkv, hd, 1 / math.sqrt(hd), window, sinks)
    out = call(ctx, c["q"], table)
    _close(out, _plain_attention(c, nh, nkv, hd, window, sinks), "float32")
    for t in (0, 15, 63, 64, 170, 299, 300, 329, 330):
        one = type("Ctx", (), dict(tok_pos=pos[t:t + 1], is_decode=True, batch=1, n_tokens=1))()
        row = table[int(c["tok_seq"][t])][None].clone()
        if window:
            row[:, max(0, -(-sinks // 64)):max(0, (int(pos[t]) - window + 1) // 64)] = 10 ** 6
        assert torch.equal(call(one, c["q"][t:t + 1], row)[0], out[t]), t
    c["vp"][int(table[0, 2])][:, c["vi"][150 - 128]] = float("inf")     # token 150 of the first sequence
    after = call(ctx, c["q"], table)
    sees = np.array([s == 0 and p >= 150 and (not window or p - 150 < window) for s, p in zip(c["tok_seq"], c["tok_pos"])])
    clean = torch.isfinite(after).all(1).cpu().numpy()
    assert np.array_equal(clean, ~sees)
    assert torch.equal(after[_t(~sees, torch.bool)], out[_t(~sees, torch.bool)])


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("longest", [3, 64, 65, 200, 500, 1100])
def test_float32_attention_with_waves_for_the_pages_there_are(hd, longest):
    """One to sixteen waves a tile by the most pages a sequence has, and more sequences than a wave has lanes, some without a
    token: the bits of the form that knows nothing of the pages."""
    nh, nkv, rng = 3, 1, np.random.default_rng(longest)
    new = [int(n) for n in rng.integers(0, 4, 130)]
    lens = [n + int(rng.integers(0, 30)) if n else 0 for n in new]
    lens[70], new[70] = longest, 2
    c = _attention_case("float32", nh, nkv, hd, [max(l, 1) for l in lens], new)
    cu = np.concatenate([[0], np.cumsum(new)])
    pos = np.concatenate([np.arange(l - n, l) for l, n in zip(lens, new)])
    ctx = lambda **kw: type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(pos, torch.int32), batch=130, n_tokens=sum(new), is_decode=False,
                                            cu_seqlens=cu.tolist(), cu_dev=_t(cu, torch.int32), **kw))()
    call = lambda x: K.attention_f32(x, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd))
    out = call(ctx(max_context=max(lens)))
    assert torch.equal(out, call(ctx()))
    want = K.attention_generic(c["q"], c["stride"], c["kp"], c["vp"], c["table"], _t(c["tok_seq"], torch.int32), _t(pos, torch.int32), nh, nkv, hd,
                               1 / math.sqrt(hd))
    _close(out, _np(want), "float32")


@pytest.mark.parametrize("hd", [64, 128])
def test_float32_attention_of_a_prompt_of_many_tiles(hd):
    """600 tokens of 32 heads are 1,200 blocks of four waves: the bits of tokens that come alone, with sixteen waves a tile
    or eight."""
    nh, L = 32, 600
    c = _attention_case("float32", nh, nh, hd, [L], [L])
    pos = _t(c["tok_pos"], torch.int32)
    call = lambda x, q: K.attention_f32(x, q, c["stride"], c["kp"], c["vp"], c["table"], nh, nh, hd, 1 / math.sqrt(hd))
    out = call(type("Ctx", (), dict(tok_pos=pos, is_decode=False, batch=1, n_tokens=L, cu_seqlens=[0, L], cu_dev=_t([0, L], torch.int32), max_context=L))(), c["q"])
    for t in (0, 63, 64, 127, 255, 256, 511, 598, 599):
        one = type("Ctx", (), dict(tok_pos=pos[t:t + 1], is_decode=True, batch=1, n_tokens=1, max_context=L))()
        assert torch.equal(call(one, c["q"][t:t + 1])[0], out[t]), t


@pytest.mark.parametrize("window,sinks", [(0, 0), (100, 70)])
@pytest.mark.parametrize("nh,nkv,hd", [(8, 2, 64), (3, 1, 128), (1, 1, 64), (20, 1, 128)])
@pytest.mark.parametrize("width", [5, 16, 17, 70])
def test_float32_attention_with_pages_in_several_blocks(nh, nkv, hd, width, window, sinks):
    """Single tokens whose pages go to several blocks, added by the block with the last ticket or by a second kernel: the bits of one block a tile, at
    the edges of pages and of a block's four, for groups that fill no tile and more than one, with pages given back; the counters end at zero."""
    longest = min(64 * width, 1100 if width > 16 else 1024)
    lens = sorted({1, 64, 65, 256, 257, 320, longest - 1, longest})
    lens = [n for n in lens if n <= longest]
    assert K.f32_pages_form(len(lens) * -(-nh // nkv // 16) * nkv, width, longest) == ("tickets" if width <= 16 else "merge")
    c = _attention_case("float32", nh, nkv, hd, lens, [1] * len(lens))
    table = torch.full((len(lens), width), 10 ** 6, dtype=torch.int32, device=DEV)
    for b, n in enumerate(lens):
        table[b, :-(-n // 64)] = c["table"][b, :-(-n // 64)]
        if window:
            table[b, max(0, -(-sinks // 64)):max(0, (n - window) // 64)] = 10 ** 6
    shares = type("Runtime", (), dict(attention_shares=[], branch_attention_shares=[]))()
    ctx = lambda **kw: type("Ctx", (), dict(tok_pos=_t(np.array(lens) - 1, torch.int32), is_decode=True, batch=len(lens), n_tokens=len(lens), **kw))()
    call = lambda x: K.attention_f32(x, c["q"], c["stride"], c["kp"], c["vp"], table, nh, nkv, hd, 1 / math.sqrt(hd), window, sinks)
    want = call(ctx())                                                   # (neither a longest context nor counters: one block a tile)
    x = ctx(runtime=shares, max_context=longest)
    for _ in range(3):
        assert torch.equal(call(x), want)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        got = call(x)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(got, want)
    assert (len(shares.attention_shares) == 1) == (width <= 16) and all(int(t.abs().sum()) == 0 for _, t in shares.attention_shares)


@pytest.mark.parametrize("types", [("float32", "float32", "float32"), ("float32", "bfloat16", "float32"), ("float32", "bfloat16", "bfloat16"),
                                   ("bfloat16", "bfloat16", "bfloat16"), ("bfloat16", "bfloat16", "float32")])
@pytest.mark.parametrize("T,N,K_,odd", [(1, 1, 1, 0), (17, 5, 3, 0), (65, 64, 256, 0), (64, 66, 260, 0), (70, 129, 36, 1), (130, 62, 33, 1), (3, 200, 512, 4)])
def test_products_of_heads(T, N, K_, odd, types):
    """One product a head: k below, at and beyond the kernel's blocks of 32, heights and row counts around its tiles of 64, rows
    and heads that begin anywhere (odd strides: value by value), with and without the gate; what lies between the heads'
    results stays.  A sum is K products deep; bfloat16 results round once more."""
    rng, Hn = np.random.default_rng(K_), 3
    ta, tw, to = (DT[t] for t in types)
    wide = _t(rng.standard_normal((T, Hn, K_ + odd)), ta)
    a, w = wide[:, :, :K_], _t(rng.standard_normal((Hn, N, K_)), tw)
    logits = _t(rng.standard_normal((T, Hn + 2)))
    plain = np.einsum("thk,hnk->thn", _np(a), _np(w))
    deep = np.einsum("thk,hnk->thn", np.abs(_np(a)), np.abs(_np(w))) * (K_ + 8) * 2.0 ** -24
    for gate in (None, logits):
        buf = torch.full((T, Hn, N + odd), 7.0, dtype=to, device=DEV)
        K.head_products(a, w, buf[:, :, :N], gate=gate)
        factor = 1.0 if gate is None else 1 / (1 + np.exp(-_np(gate)[:, :Hn, None]))
        want = plain * factor
        bound = deep * factor + np.abs(want) * (2.0 ** -8 if types[2] == "bfloat16" else 2.0 ** -20) + 1e-30
        assert (np.abs(_np(buf[:, :, :N]) - want) <= bound).all()
        assert (buf[:, :, N:] == 7.0).all()


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("low", [(20,), tuple(range(64, 128)), tuple(range(0, 64)), (0, 70, 130, 190)])
def test_float32_attention_of_keys_whose_weights_underflow(hd, low):
    """Keys that a row sees with a weight that underflows to 0, alone in a page, a whole page of them before or behind the
    others: their values, infinite or not a number, count for nothing, and the result is the bits of values of 0."""
    nh, nkv, L = 4, 2, 200
    c = _attention_case("float32", nh, nkv, hd, [L], [L])
    c["q"][:, :nh * hd] = 1.0 + 0.1 * c["q"][:, :nh * hd].clamp(-1, 1)
    c["kp"] *= 0.01
    cu = np.array([0, L])
    ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32), batch=1, n_tokens=L, is_decode=False,
                               cu_seqlens=[0, L], cu_dev=_t(cu, torch.int32), max_context=L))()
    call = lambda: K.attention(ctx, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd))
    rows = torch.tensor([t > max(low) if low[0] == 0 else True for t in range(L)], device=DEV)      # rows that see another key
    outs = []
    for value in (0.0, float("inf"), float("nan")):
        for t in low:
            page = int(c["table"][0, t // 64])
            c["kp"][page][:, c["ki"][t % 64]] = -40.0                    # a score below -300 beside ones near 0
            c["vp"][page][:, c["vi"][t % 64]] = value
        outs.append(call())
    assert torch.isfinite(outs[0]).all()
    assert torch.equal(outs[1][rows], outs[0][rows]) and torch.equal(outs[2][rows], outs[0][rows])


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("window,sinks", [(0, 0), (70, 5)])
def test_float32_attention_of_tokens_in_any_order(hd, window, sinks):
    """Tokens of a sequence in any order of positions, single tokens of sequences in any order, steps of which nothing is known
    but every token's sequence and position (tokens of the sequences mixed), pages whose rows are wider than a head."""
    nh, nkv, rng = 6, 2, np.random.default_rng(hd)
    lens, new = [200, 90, 3], [200, 33, 3]
    c = _attention_case("float32", nh, nkv, hd, lens, new)
    want = _plain_attention(c, nh, nkv, hd, window, sinks)
    cu, T = np.concatenate([[0], np.cumsum(new)]), sum(new)
    call = lambda rows, **kw: K.attention(
        type("Ctx", (), dict(tok_seq=_t(c["tok_seq"][rows], torch.int32), tok_pos=_t(c["tok_pos"][rows], torch.int32), batch=3, n_tokens=len(rows), **kw))(),
        c["q"][_t(rows, torch.int64)], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd), window, sinks)
    shuffled = np.concatenate([rng.permutation(np.arange(a, b)) for a, b in zip(cu, cu[1:])])
    _close(call(shuffled, is_decode=False, cu_seqlens=cu.tolist(), cu_dev=_t(cu, torch.int32)), want[shuffled], "float32")
    mixed = rng.permutation(T)
    _close(call(mixed, is_decode=False, cu_seqlens=None, cu_dev=None), want[mixed], "float32")
    last = np.array([T - 1, 199, 232])
    _close(call(last, is_decode=True, cu_seqlens=[0, 1, 2, 3], cu_dev=None), want[last], "float32")
    if not window:                                                      # key pages of hd + 16 dimensions a row
        kw_, vw = (torch.zeros((p.shape[0], nkv, 64 * (hd + 16)), device=DEV) for p in (c["kp"], c["vp"]))
        ki, vi = _page_index(hd + 16)
        kw_[:, :, ki[:, :hd].reshape(-1)] = c["kp"][:, :, c["ki"].reshape(-1)]
        vw[:, :, vi[:, :hd].reshape(-1)] = c["vp"][:, :, c["vi"].reshape(-1)]
        ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32), batch=3, n_tokens=T, is_decode=False,
                                   cu_seqlens=cu.tolist(), cu_dev=_t(cu, torch.int32)))()
        got = K.attention(ctx, c["q"], c["stride"], kw_, vw, c["table"], nh, nkv, hd, 1 / math.sqrt(hd))
        _close(got.view(T, nh, -1)[:, :, :hd].reshape(T, nh * hd), want, "float32")


@pytest.mark.parametrize("window,sinks", [(0, 0), (200, 70)])
@pytest.mark.parametrize("nh,nkv,hd,batch,longest", [(8, 4, 128, 64, 700),      # one block a sequence, three pages a wave
                                                     (8, 4, 64, 70, 1500),       # batches beyond the captured sizes
                                                     (16, 2, 64, 128, 700),
                                                     (8, 4, 128, 4, 1500),       # one page a wave, six blocks merged
                                                     (4, 1, 128, 4, 3300),       # 13 blocks merged
                                                     (8, 2, 128, 16, 5000)])     # several pages a wave and several blocks
def test_single_token_attention_with_blocks_of_every_size(nh, nkv, hd, batch, longest, window, sinks):
    """The decode kernel gives a wave more pages when there are many blocks; every form must
    agree with the plain attention, whatever the lengths of the other sequences.  With a window
    the pages between the sinks and the window are not the sequence's any more (the cache gives
    them back): they hold NaN here, which would spoil the result if a wave took one of them."""
    rng = np.random.default_rng(batch)
    lens = [int(x) for x in rng.integers(1, longest // 3, batch)]
    lens[1], lens[batch // 2], lens[-1] = longest, 64, 65
    new = [1] * batch
    c = _attention_case("bfloat16", nh, nkv, hd, lens, new, seed=batch)
    for b, l in enumerate(lens):                                        # unwritten page tails must not matter
        if l % 64:
            page = int(c["table"][b, l // 64])
            c["kp"][page][:, c["ki"][l % 64:]] = float("nan")
            c["vp"][page][:, c["vi"][l % 64:]] = float("nan")
        for pi in range((l + 63) // 64 if window else 0):
            if pi * 64 >= sinks and pi * 64 + 63 <= l - 1 - window:     # no key of the page is visible from position l - 1
                page = int(c["table"][b, pi])
                c["kp"][page] = float("nan")
                c["vp"][page] = float("nan")
    ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32),
                               is_decode=True, max_context=max(lens), batch=batch, n_tokens=batch,
                               cu_seqlens=list(range(batch + 1)), cu_dev=None, starts=[l - 1 for l in lens],
                               shared={}))()
    out = K.attention_mfma_bf16(ctx, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd),
                                window, sinks)
    assert out is not None
    _close(out, _plain_attention(c, nh, nkv, hd, window, sinks), "bfloat16")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_attention_of_random_shapes(dtype):
    """Heads, groups, head sizes, lengths, windows and sinks drawn at random: prompts whole and
    continued, and single tokens, whichever kernel the dispatch takes."""
    rng = np.random.default_rng(31)
    for case in range(24):
        hd = int(rng.choice([16, 32, 48, 64, 64, 96, 128, 128, 256]))
        nkv = int(rng.choice([1, 2, 3, 8]))
        nh = nkv * int(rng.choice([1, 2, 4, 5, 16]))
        B = int(rng.integers(1, 5))
        lens = [int(rng.integers(1, 400)) for _ in range(B)]
        kind = case % 3
        new = [1] * B if kind == 0 else (lens if kind == 1 else [int(rng.integers(1, l + 1)) for l in lens])
        window = int(rng.choice([0, 0, 1, 64, 100]))
        sinks = int(rng.choice([0, 4])) if window else 0
        c = _attention_case(dtype, nh, nkv, hd, lens, new, seed=100 + case)
        for b, l in enumerate(lens):                                        # unwritten page tails must not matter
            if l % 64:
                page = int(c["table"][b, l // 64])
                c["kp"][page][:, c["ki"][l % 64:]] = float("nan")
                c["vp"][page][:, c["vi"][l % 64:]] = float("nan")
        ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32),
                                   is_decode=max(new) == 1, max_context=max(lens), batch=B, n_tokens=sum(new),
                                   cu_seqlens=np.concatenate([[0], np.cumsum(new)]).tolist(),
                                   cu_dev=_t(np.concatenate([[0], np.cumsum(new)]), torch.int32),
                                   starts=[l - n for l, n in zip(lens, new)], shared={}))()
        out = K.attention(ctx, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd), window, sinks)
        want = _plain_attention(c, nh, nkv, hd, window, sinks)
        err = np.abs(_np(out) - want).max()
        assert err <= RT[dtype] * max(1.0, np.abs(want).max()), (case, nh, nkv, hd, lens, new, window, sinks, err)


@pytest.mark.parametrize("tile_rows,halves", [(64, 1), (128, 1), (128, 2)])
@pytest.mark.parametrize("nh,nkv,hd", [(6, 2, 64), (8, 2, 128), (3, 3, 128)])
@pytest.mark.parametrize("window,sinks", [(0, 0), (100, 0), (70, 5)])
def test_prompt_attention_on_the_matrix_cores(tile_rows, halves, nh, nkv, hd, window, sinks):
    """The prompt kernels (pages read by each wave; pages shared through LDS by one set of waves
    or by two that take the pages in turn) on long and short sequences, whole and continued,
    with pages half written, and with odd and even numbers of pages a tile."""
    K.PREFILL_TILE_ROWS, K.PREFILL_HALVES = tile_rows, halves
    try:
        for lens, new in (([300, 129, 5, 64], [300, 129, 5, 64]), ([400, 90, 257], [200, 33, 129]),
                          ([1100, 700], [1100, 190])):
            c = _attention_case("bfloat16", nh, nkv, hd, lens, new, seed=11)
            ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32),
                                       is_decode=False, max_context=max(lens), batch=len(lens), n_tokens=sum(new),
                                       cu_seqlens=np.concatenate([[0], np.cumsum(new)]).tolist(),
                                       cu_dev=_t(np.concatenate([[0], np.cumsum(new)]), torch.int32),
                                       starts=[l - n for l, n in zip(lens, new)], shared={}))()
            # what lies behind the written part of a page must not matter: poison it
            for b, l in enumerate(lens):
                if l % 64:
                    page = int(c["table"][b, l // 64])
                    c["kp"][page][:, c["ki"][l % 64:]] = float("nan")
                    c["vp"][page][:, c["vi"][l % 64:]] = float("nan")
            out = K.attention_mfma_bf16(ctx, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd,
                                        1 / math.sqrt(hd), window, sinks)
            assert out is not None
            _close(out, _plain_attention(c, nh, nkv, hd, window, sinks), "bfloat16")
    finally:
        K.PREFILL_TILE_ROWS = K.PREFILL_HALVES = 0


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_attention_finds_a_far_key_among_hundreds(dtype):
    """One early key matches the query strongly; the output must be its value."""
    nh, nkv, hd, L = 4, 2, 64, 700
    c = _attention_case(dtype, nh, nkv, hd, [L], [1], scale_q=0.01)
    q = c["q"]
    far = 5
    page, off = int(c["table"][0, far // 64]), far % 64
    key = torch.zeros(hd, device=DEV); key[3] = 40.0
    c["kp"][page][:, c["ki"][off]] = key.to(c["kp"].dtype)
    q[0, :nh * hd] = (key.repeat(nh) * 2).to(q.dtype)                   # score 40 * 80 / 8 = 400 for that key
    ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32),
                               is_decode=True, max_context=L, batch=1, n_tokens=1, cu_seqlens=[0, 1], cu_dev=None,
                               starts=[L - 1], shared={}))()
    out = _np(K.attention(ctx, q, c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd)))
    want = np.concatenate([c["vs"][0][far].reshape(nkv, hd)[h // 2] for h in range(nh)])
    assert np.abs(out[0] - want).max() < 1e-5


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("hd", [32, 64, 128])
@pytest.mark.parametrize("window,sinks", [(64, 0), (70, 0), (5, 2), (128, 64), (1, 0)])
def test_attention_window_edges(dtype, window, sinks, hd):
    nh, nkv = 4, 2
    for lens, new in (([300, 66], [1, 1]), ([200, 10], [200, 10]), ([257], [100])):
        c = _attention_case(dtype, nh, nkv, hd, lens, new, seed=9)
        # keys just outside and just inside the window stand out, so an off-by-one shows
        for b, l in enumerate(lens):
            for p in (l - 1 - window, l - window):
                if p >= max(sinks, 0) and p >= 0:
                    page, off = int(c["table"][b, p // 64]), p % 64
                    c["kp"][page][:, c["ki"][off]] *= 6.0
                    c["ks"][b][p] = _np(c["kp"][page][:, c["ki"][off]]).reshape(-1)    # as stored
        ctx = type("Ctx", (), dict(tok_seq=_t(c["tok_seq"], torch.int32), tok_pos=_t(c["tok_pos"], torch.int32),
                                   is_decode=max(new) == 1, max_context=max(lens), batch=len(lens),
                                   n_tokens=sum(new), cu_seqlens=np.concatenate([[0], np.cumsum(new)]).tolist(),
                                   cu_dev=_t(np.concatenate([[0], np.cumsum(new)]), torch.int32),
                                   starts=[l - n for l, n in zip(lens, new)], shared={}))()
        out = K.attention(ctx, c["q"], c["stride"], c["kp"], c["vp"], c["table"], nh, nkv, hd, 1 / math.sqrt(hd),
                          window, sinks)
        _close(out, _plain_attention(c, nh, nkv, hd, window, sinks), dtype)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_swiglu(dtype):
    rng = np.random.default_rng(5)
    gu = _t(rng.standard_normal((9, 2 * 137)) * 4, DT[dtype])
    g, u = _np(gu)[:, :137], _np(gu)[:, 137:]
    _close(K.swiglu(gu), pm.silu(g) * u, dtype)
    parts = torch.stack([gu.float() * 0.25, gu.float() * 0.75])
    _close(K.swiglu(parts, DT[dtype]), pm.silu(g) * u, dtype)
    _close(K.sum_parts(parts, None, DT[dtype]), _np(gu), dtype)


def test_gather_of_token_ids():
    src = _t([5, 9, 2, 7, 11], torch.int32)
    rows = _t([4, 0, 0, 3], torch.int32)
    dst = torch.full((4,), -1, dtype=torch.int32, device=DEV)
    K.gather_i32(dst, src, rows)
    assert dst.cpu().tolist() == [11, 5, 5, 7]
    K.gather_i32(dst, src, _t([1, 7, -1, 2], torch.int32))               # rows outside the vector give 0, never a fault
    assert dst.cpu().tolist() == [9, 0, 0, 2]
    with pytest.raises(K.KernelError):
        K.gather_i32(dst, src, rows[:3])
    with pytest.raises(K.KernelError):
        K.gather_i32(dst, src.float(), rows)


def test_argmax_first_maximum_wins():
    rng = np.random.default_rng(6)
    x = rng.standard_normal((5, 128257)).astype(np.float32)
    x[1, 4000] = x[1, 90000] = 9.0                                      # a tie: the first wins
    x[2, 128256] = 10.0
    x[3, :] = 0.25                                                      # all equal
    x[4, 0] = 11.0
    got = K.argmax(_t(x)).cpu().tolist()
    assert got == [int(np.argmax(x[0])), 4000, 128256, 0, 0]
    assert K.argmax(_t([[1., 5., 3., 2.]])).item() == 1                 # tests/.../SamplerTests.cs:8-18


def test_kernels_refuse_what_they_cannot_do():
    x = torch.zeros(4, 64, device=DEV)
    with pytest.raises(K.KernelError, match="GPU"):
        K.rmsnorm(torch.zeros(4, 64), torch.ones(64), 1e-6, torch.float32)
    with pytest.raises(K.KernelError, match="weight"):
        K.rmsnorm(x, torch.ones(63, device=DEV), 1e-6, torch.float32)
    with pytest.raises(K.KernelError, match="w must be"):
        K.gemm(x, torch.zeros(8, 65, device=DEV), None, torch.float32)
    with pytest.raises(K.KernelError, match="not supported"):
        K.gemm(x.half(), torch.zeros(8, 64, device=DEV).half(), None, torch.float16)
    with pytest.raises(K.KernelError, match="head_dim"):
        K.qk_rope_cache(torch.zeros(1, 3 * 1024, device=DEV), None, torch.float32, 1, 1, 1024, 2, 0, None, None, 1e-6,
                        torch.zeros(1, 1, 2, device=DEV), None, None, None,
                        torch.zeros(1, dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV))


@pytest.mark.parametrize("M,N,K_", [(1, 4096, 4096), (8, 331, 1000), (16, 100, 72), (17, 4096, 14336), (33, 257, 2048),
                                    (64, 1000, 520), (48, 6144, 4096), (5, 64, 32), (64, 65, 8)])
def test_gemm_on_packed_weights(M, N, K_):
    """The few-row product on the packed copy of the weights (blocks of 64 rows, steps of 32 k,
    zero-padded): every row count class, heights and lengths that fill no block or step, one part
    and several, bias, float32 and bfloat16 results."""
    rng = np.random.default_rng(M * 1000 + N)
    a, w = _t(rng.standard_normal((M, K_)), torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    bias = _t(rng.standard_normal(N))
    want = _np(a) @ _np(w).T
    pw = K.pack_weights(w)
    assert pw.N == N and pw.K == K_ and pw.data.numel() == -(-N // 64) * 64 * -(-K_ // 32) * 32
    for chunk in (128, 256):
        for splits in (1, 2, 5):
            out = K.gemm_packed_bf16(a, pw, None, torch.float32, splits, chunk)
            assert out is not None and out.dtype == torch.float32
            _close(out.sum(0), want, "float32", scale=np.abs(want).max() * 10)        # bfloat16 operands, float32 sums
        out = K.gemm_packed_bf16(a, pw, bias, torch.bfloat16, 1, chunk)
        _close(out[0], want + _np(bias), "bfloat16")
    # through the dispatch, as a part calls it
    out = K.gemm_product(a, w, torch.bfloat16, f32_ok=True, packed=pw)
    _close(K.sum_parts(out, None, torch.float32), want, "float32", scale=np.abs(want).max() * 10)
    _close(K.gemm(a, w, bias, torch.float32, packed=pw), want + _np(bias), "float32", scale=np.abs(want).max() * 10)
    # a row's result does not depend on the other rows of its class
    if M > 1:
        alone = K.gemm_packed_bf16(a[:1].contiguous(), pw, None, torch.float32, 1, 256)
        if (M + 15) // 16 in (1,):
            assert torch.equal(alone[0], K.gemm_packed_bf16(a, pw, None, torch.float32, 1, 256)[0][:1])


@pytest.mark.parametrize("M,N,K_,splits", [(1, 200, 40, 1), (16, 200, 2056, 3), (17, 130, 264, 1), (64, 16384, 520, 1),   # one block a unit
                                           (33, 32840, 264, 1), (17, 32840, 1032, 1),                    # more than two
                                           (64, 28696, 1544, 1), (33, 28696, 2824, 1), (40, 57400, 2568, 1)])   # two strips a wave
def test_packed_product_forms_add_alike(M, N, K_, splits):
    """Every form of the product on packed weights (a ring of loads, one or two strips a wave) gives the bits of the
    row-major product, which adds in the same order: steps and chunks that the ring's length does not divide, the last
    block of a pair missing, several parts."""
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(M, K_, device=DEV, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K_, device=DEV, generator=g) * 0.05).to(torch.bfloat16)
    want = K.gemm_skinny_lds_bf16(a, w, None, torch.float32, splits)
    got = K.gemm_packed_bf16(a, K.pack_weights(w), None, torch.float32, splits, 256)
    assert torch.equal(got, want)
    if splits == 1:                                   # want in parts adds in another order than the gated product
        rows = N // 32 * 32
        y = K.gemm_packed_gated_bf16(a, K.pack_weights(w[:rows].contiguous(), rows // 2), torch.float32, 256)
        gate, up = want[0][:, :rows // 2].double(), want[0][:, rows // 2:rows].double()
        # the hardware's exp2 and reciprocal: 1 ulp each on a factor of at most 1, two more roundings
        assert torch.allclose(y.double(), gate * torch.sigmoid(gate) * up, rtol=2e-6, atol=1e-6)


def test_first_rows_of_packed_weights_and_the_fused_swiglu():
    rng = np.random.default_rng(3)
    I, H = 200, 136
    w = _t(rng.standard_normal((192, H)) * 0.1, torch.bfloat16)
    pw = K.pack_weights(w)
    a = _t(rng.standard_normal((9, H)), torch.bfloat16)
    first = pw.rows(128)
    assert first is not None and first.N == 128 and pw.rows(100) is None and pw.rows(192) is pw
    _close(K.gemm_packed_bf16(a, first, None, torch.float32, 1, 128)[0], (_np(a) @ _np(w).T)[:, :128], "float32", scale=50.0)
    # down product of silu(gate) * up made on the way, from a bfloat16 row [gate | up] and from float32 partial sums
    wd = _t(rng.standard_normal((H, I)) * 0.1, torch.bfloat16)
    pd = K.pack_weights(wd)
    gu = _t(rng.standard_normal((9, 2 * I)), torch.bfloat16)
    g, u = _np(gu)[:, :I], _np(gu)[:, I:]
    act = _np(_t(pm.silu(g) * u, torch.bfloat16))                     # the kernel rounds the product to bfloat16
    want = act @ _np(wd).T
    out = K.gemm_packed_bf16(gu, pd, None, torch.float32, 1, 128, swiglu=True)
    _close(out[0], want, "bfloat16")
    parts = _t(rng.standard_normal((3, 9, 2 * I)))
    tot = _np(parts).sum(0)
    want = _np(_t(pm.silu(tot[:, :I]) * tot[:, I:], torch.bfloat16)) @ _np(wd).T
    out = K.gemm_packed_bf16(parts, pd, None, torch.float32, 2, 128, swiglu=True)
    _close(out.sum(0), want, "bfloat16")


@pytest.mark.parametrize("M,I,H", [(1, 208, 136), (9, 14336, 4096), (16, 64, 72), (33, 1008, 264), (64, 2048, 520), (47, 16, 40)])
def test_gate_up_product_with_the_swiglu_epilogue(M, I, H):
    """The few-row product on a matrix packed as strips of gate rows and up rows in turn gives
    silu(a gate^T) * (a up^T) directly; against the plain functions, every class of row count,
    widths that fill no block."""
    rng = np.random.default_rng(M + I)
    wg, wu = (_t(rng.standard_normal((I, H)) * 0.08, torch.bfloat16) for _ in range(2))
    a = _t(rng.standard_normal((M, H)), torch.bfloat16)
    w = torch.cat([wg, wu]).contiguous()
    pw = K.pack_weights(w, gate_rows=I)
    assert pw.gate_rows == I and pw.rows(64) is None
    want = pm.silu(_np(a) @ _np(wg).T) * (_np(a) @ _np(wu).T)
    for chunk in (128, 256):
        got = K.gemm_packed_gated_bf16(a, pw, torch.float32, chunk)
        assert got is not None and got.shape == (M, I)
        _close(got, want, "float32", scale=np.abs(want).max() * 50)           # hardware exp2 and reciprocal: about 1e-6 relative
    _close(K.gemm_packed_gated_bf16(a, pw, torch.bfloat16, 256), want, "bfloat16")
    # a packed copy in this order serves no other product: the dispatch leaves it aside
    out = K.gemm_product(a, w, torch.bfloat16, packed=pw)
    _close(K.sum_parts(out, None, torch.float32), _np(a) @ _np(w).T, "bfloat16")
    with pytest.raises(K.KernelError):
        K.pack_weights(w, gate_rows=I + 16)


@pytest.mark.parametrize("M,N,K_", [(1, 4096, 4096), (8, 4096, 14336), (16, 48, 200), (5, 80, 8), (13, 5120, 1000), (3, 16, 72), (9, 120, 200),
                                    (2, 7, 16)])
@pytest.mark.parametrize("waves,strips", [(4, 1), (8, 1), (16, 1), (8, 2), (4, 2)])
def test_product_that_adds_itself_to_the_residual_stream(M, N, K_, waves, strips):
    """x += a w^T + bias in one kernel for up to 16 rows, with what it leaves for the norm that follows: the
    sums of squares of the new rows by strips of 16 columns, and x * norm_w rounded to bfloat16.  Against
    float64; rows beyond M stay zero in the sums; a row's result does not depend on the rows beside it."""
    rng = np.random.default_rng(M * 100 + N + waves + strips)
    a, w = _t(rng.standard_normal((M, K_)), torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    bias, norm_w = _t(rng.standard_normal(N)), _t(1 + 0.1 * rng.standard_normal(N))
    x0 = _t(rng.standard_normal((M, N)) * 3)
    pw = K.pack_weights(w)
    want = _np(x0) + _np(a) @ _np(w).T + _np(bias)
    x = x0.clone()
    left = K.gemm_residual_bf16(x, a, pw, bias, waves, norm_w, strips)
    assert isinstance(left, K.RowSquares) and left.width == N and left.norm_w is norm_w
    _close(x, want, "float32", scale=np.abs(want).max() * 10)                    # bfloat16 operands, float32 sums
    n_strips = -(-(-(-N // 16)) // strips)                                        # blocks of 16 * strips columns
    assert left.sums.shape == (n_strips, 16)
    sums = _np(left.sums)
    assert np.all(sums[:, M:] == 0)
    padded = np.zeros((M, n_strips * 16 * strips))
    padded[:, :N] = _np(x)
    by_strip = (padded ** 2).reshape(M, n_strips, 16 * strips).sum(2).T                      # [strips, M] of the x it wrote
    assert np.allclose(sums[:, :M], by_strip, rtol=2e-6, atol=1e-30)
    assert torch.equal(left.unscaled, (x * norm_w).to(torch.bfloat16))           # the same float32 product, rounded once
    # without a bias and without the norm's rows; one row alone gives the same bits
    x1 = x0.clone()
    plain = K.gemm_residual_bf16(x1, a, pw, None, waves, strips=strips)
    assert plain.unscaled is None
    _close(x1, want - _np(bias), "float32", scale=np.abs(want).max() * 10)
    alone = x0[:1].clone()
    K.gemm_residual_bf16(alone, a[:1].contiguous(), pw, None, waves, strips=strips)
    assert torch.equal(alone, x1[:1])
    # refused: two strips a block of 16 waves, whose registers do not fit; more than 16 rows
    with pytest.raises(K.KernelError):
        K.gemm_residual_bf16(x1, a, pw, None, 16, strips=2)
    assert K.gemm_residual_bf16(torch.zeros(17, N, device=DEV), torch.zeros(17, K_, device=DEV, dtype=torch.bfloat16), pw, None, waves) is None


@pytest.mark.parametrize("M,N,K_", [(1, 2048, 8192), (8, 2048, 2048), (16, 1024, 4096), (16, 48, 200), (5, 80, 8), (13, 1000, 1000), (3, 16, 72),
                                    (9, 120, 1032), (2, 7, 16)])
@pytest.mark.parametrize("waves", [8, 16])
def test_product_that_adds_itself_to_the_residual_stream_by_half_strips(M, N, K_, waves):
    """The same with 8 rows of w a block: odd numbers of steps of k and of half strips, parts of them, and rows alone."""
    rng = np.random.default_rng(M * 100 + N + waves)
    a, w = _t(rng.standard_normal((M, K_)), torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    bias, norm_w = _t(rng.standard_normal(N)), _t(1 + 0.1 * rng.standard_normal(N))
    x0 = _t(rng.standard_normal((M, N)) * 3)
    pw = K.pack_weights(w)
    want = _np(x0) + _np(a) @ _np(w).T + _np(bias)
    x = x0.clone()
    left = K.gemm_residual_bf16(x, a, pw, bias, waves, norm_w, 0)
    _close(x, want, "float32", scale=np.abs(want).max() * 10)                    # bfloat16 operands, float32 sums
    blocks = 2 * -(-N // 16)
    sums, padded = _np(left.sums), np.zeros((M, blocks * 8))
    padded[:, :N] = _np(x)
    assert sums.shape == (blocks, 16) and np.all(sums[:, M:] == 0)
    assert np.allclose(sums[:, :M], (padded ** 2).reshape(M, blocks, 8).sum(2).T, rtol=2e-6, atol=1e-30)
    assert torch.equal(left.unscaled, (x * norm_w).to(torch.bfloat16))
    plain, alone = x0.clone(), x0[:1].clone()
    K.gemm_residual_bf16(plain, a, pw, None, waves, strips=0)
    K.gemm_residual_bf16(alone, a[:1].contiguous(), pw, None, waves, strips=0)
    assert torch.equal(alone, plain[:1])


def test_library_product_that_adds_itself_to_the_residual_stream():
    """For prompts that the library's product serves, the sum with the residual stream is the product's
    epilogue: the float32 product added to x, bit for bit; refused for few rows, other element types and where
    the tiled product serves."""
    rng = np.random.default_rng(5)
    for M, N, K_ in ((200, 96, 72), (2048, 4096, 4096), (129, 331, 1000)):
        a, w = _t(rng.standard_normal((M, K_)), torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
        x0 = _t(rng.standard_normal((M, N)) * 3)
        x = x0.clone()
        assert K.gemm_library_add(x, a, w)
        assert torch.equal(x, x0 + torch.mm(a, w.t(), out_dtype=torch.float32))
        _close(x, _np(x0) + _np(a) @ _np(w).T, "float32", scale=np.abs(_np(x)).max() * 10)
    x = x0[:64].clone()
    assert not K.gemm_library_add(x, a[:64].contiguous(), w) and torch.equal(x, x0[:64])
    assert not K.gemm_library_add(x0.clone(), a.float(), w.float())
    a, w = _t(rng.standard_normal((256, 8192)), torch.bfloat16), _t(rng.standard_normal((1024, 8192)) * 0.05, torch.bfloat16)
    pw = K.pack_weights(w)
    if K.tiles_plan(256, 1024, 8192) is not None:                              # much longer than high: the tiled product in parts
        assert not K.gemm_library_add(torch.zeros(256, 1024, device=DEV), a, w, pw)


@pytest.mark.parametrize("M,N,K_", [(1, 6144, 4096), (8, 331, 1000), (16, 96, 72), (7, 64, 4112), (11, 200, 16)])
def test_product_on_norm_rows_without_their_scale(M, N, K_):
    """The few-row product whose activations are x * w of an rmsnorm, with the sums of squares of x beside
    them: the row's scale 1 / sqrt(mean square + eps) is applied to the result.  Against float64 on the same
    bfloat16 rows; parts and a bias; any number of partial sums (also more than 256 and fewer than 16)."""
    rng = np.random.default_rng(M + N)
    eps = 1e-5
    x = _t(rng.standard_normal((M, K_)) * 2)
    norm_w = _t(1 + 0.1 * rng.standard_normal(K_))
    w = _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    bias = _t(rng.standard_normal(N))
    pw = K.pack_weights(w)
    unscaled = (x * norm_w).to(torch.bfloat16)
    inv = 1.0 / np.sqrt((_np(x) ** 2).mean(1) + eps)
    want = (_np(unscaled) @ _np(w).T) * inv[:, None]
    for strips in (K_ // 8, 3, 300):                                               # the sums arrive in parts of any count
        cols = np.array_split(np.arange(K_), strips)
        sums = np.zeros((strips, 16))
        for i, c in enumerate(cols):
            sums[i, :M] = (_np(x)[:, c] ** 2).sum(1)
        left = K.RowSquares(_t(sums), K_, unscaled, norm_w)
        for splits, chunk in ((1, 128), (3, 256)):
            out = K.gemm_packed_unscaled_bf16(left, eps, pw, None, torch.float32, splits, chunk)
            assert out is not None and out.dtype == torch.float32
            _close(out.sum(0), want, "float32", scale=np.abs(want).max() * 10)
        out = K.gemm_packed_unscaled_bf16(left, eps, pw, bias, torch.bfloat16, 1, 128)
        _close(out[0], want + _np(bias), "bfloat16")
    # the norm's own kernel and the product on its output: the same up to one rounding of the activations
    normed = K.rmsnorm(x.clone(), norm_w, eps, torch.bfloat16)
    ref = K.gemm_packed_bf16(normed, pw, None, torch.float32, 1, 128)[0]
    _close(K.gemm_packed_unscaled_bf16(left, eps, pw, None, torch.float32, 1, 128)[0], _np(ref), "bfloat16")


@pytest.mark.parametrize("M,I,H", [(1, 208, 136), (8, 14336, 4096), (16, 64, 72)])
def test_gate_up_product_on_norm_rows_without_their_scale(M, I, H):
    rng = np.random.default_rng(M + I)
    eps = 1e-6
    wg, wu = (_t(rng.standard_normal((I, H)) * 0.08, torch.bfloat16) for _ in range(2))
    pw = K.pack_weights(torch.cat([wg, wu]).contiguous(), gate_rows=I)
    x = _t(rng.standard_normal((M, H)) * 4)
    norm_w = _t(1 + 0.1 * rng.standard_normal(H))
    unscaled = (x * norm_w).to(torch.bfloat16)
    strips = -(-H // 16)
    sums = np.zeros((strips, 16))
    for i in range(strips):
        sums[i, :M] = (_np(x)[:, 16 * i: 16 * i + 16] ** 2).sum(1)
    inv = 1.0 / np.sqrt((_np(x) ** 2).mean(1) + eps)
    a = _np(unscaled)
    want = pm.silu((a @ _np(wg).T) * inv[:, None]) * ((a @ _np(wu).T) * inv[:, None])
    left = K.RowSquares(_t(sums), H, unscaled, norm_w)
    for chunk in (128, 256):
        got = K.gemm_packed_unscaled_bf16(left, eps, pw, None, torch.float32, 1, chunk)
        assert got is not None and got.shape == (M, I)
        _close(got, want, "float32", scale=np.abs(want).max() * 50)
    _close(K.gemm_packed_unscaled_bf16(left, eps, pw, None, torch.bfloat16, 1, 128), want, "bfloat16")


@pytest.mark.parametrize("M,N,K_", [(65, 256, 64), (300, 1000, 512), (2048, 4096, 4096), (129, 6144, 1024), (700, 130, 192),
                                    (1500, 2300, 640), (190, 136, 576), (318, 40, 576)])
@pytest.mark.parametrize("token_tiles", [0, 4, 2])
def test_tiled_product_for_many_rows_on_packed_weights(M, N, K_, token_tiles):
    """The hand-written prompt-size product (tiles of 64 to 256 tokens x 256 rows, 16x16x32 MFMAs on the
    packed copy; the heights that the launch chooses, 256 and 128): token counts and heights that fill no tile, float32 and bfloat16 results, bias, parts of k."""
    rng = np.random.default_rng(M + N)
    a, w = _t(rng.standard_normal((M, K_)), torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    bias = _t(rng.standard_normal(N))
    want = _np(a) @ _np(w).T
    pw = K.pack_weights(w)
    _close(K.gemm_tiles_bf16(a, pw, None, torch.float32, token_tiles=token_tiles), want, "float32", scale=np.abs(want).max() * 10)
    _close(K.gemm_tiles_bf16(a, pw, bias, torch.bfloat16, token_tiles=token_tiles), want + _np(bias), "bfloat16")
    assert K.gemm_tiles_bf16(a[:, :K_ - 8].contiguous(), K.pack_weights(w[:, :K_ - 8].contiguous()), None, torch.float32) is None
    for parts in (2, 3, 4):                                             # (9 stages in 4 parts: 2, 2, 2 and 3, none empty)
        got = K.gemm_tiles_bf16(a, pw, None, torch.bfloat16, parts=parts, token_tiles=token_tiles)
        if K_ // 64 // parts < 2:
            assert got is None                                          # a part would hold less than two stages of 64
            continue
        assert got.shape == (parts, M, N) and got.dtype == torch.float32
        if parts == 2:                                                  # the first part is the product over the first half of k
            half = (K_ // 64) // 2 * 64
            _close(got[0], _np(a)[:, :half] @ _np(w)[:, :half].T, "float32", scale=np.abs(want).max() * 10)
        _close(got.sum(0), want, "float32", scale=np.abs(want).max() * 10)
        _close(K.sum_parts(got, bias, torch.float32), want + _np(bias), "float32", scale=np.abs(want).max() * 10)


def test_tiled_product_cuts_the_last_round_into_smaller_tiles():
    """2,048 tokens by 7,168 rows are 8 x 28 tiles of 256 tokens: on 64 compute units 224 tiles are three
    rounds and a half, and the launch takes the row tiles of the half round in tiles of 128 tokens.  The
    result does not depend on the cut (every element's sum runs over k in the same order)."""
    rng = np.random.default_rng(3)
    M, N, K_ = 2048, 7168, 256
    a, w = _t(rng.standard_normal((M, K_)), torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    pw = K.pack_weights(w)
    lib = K._lib()
    outs = []
    for units in (64, 256, 1):                    # 224 tiles: 3.5 rounds of 64 (cut), less than one round of 256, whole rounds of 1
        out = torch.empty((M, N), dtype=torch.float32, device=a.device)
        code = lib.llogos_gemm_tiles_bf16(K._p(out), K.F32, K._p(a), a.stride(0), K._p(pw.data), None, M, N, K_, N, M * N, 0, 1, 0,
                                          units, -1.0, K._stream())
        assert code == 0
        outs.append(out)
    _close(outs[0], _np(a) @ _np(w).T, "float32", scale=np.abs(_np(a) @ _np(w).T).max() * 10)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("M,I,H", [(200, 1008, 256), (2048, 14336, 4096), (65, 16, 64), (1000, 7200, 320)])
def test_tiled_product_with_the_swiglu_epilogue(M, I, H):
    rng = np.random.default_rng(M + I)
    wg, wu = (_t(rng.standard_normal((I, H)) * 0.08, torch.bfloat16) for _ in range(2))
    a = _t(rng.standard_normal((M, H)) * (0.25 if H > 1000 else 1.0), torch.bfloat16)
    pw = K.pack_weights(torch.cat([wg, wu]).contiguous(), gate_rows=I)
    want = pm.silu(_np(a) @ _np(wg).T) * (_np(a) @ _np(wu).T)
    for token_tiles in (0, 4, 2):
        got = K.gemm_tiles_bf16(a, pw, None, torch.float32, token_tiles=token_tiles)
        assert got.shape == (M, I)
        _close(got, want, "float32", scale=np.abs(want).max() * 50)
        _close(K.gemm_tiles_bf16(a, pw, None, torch.bfloat16, token_tiles=token_tiles), want, "bfloat16")
    with pytest.raises(K.KernelError):
        K.gemm_tiles_bf16(a, pw, None, torch.float32, parts=2)


def test_prompts_through_the_tiled_product(monkeypatch):
    """An engine whose prompt products are the hand-written ones gives the plain logits like the default."""
    import gpu_helpers as H
    monkeypatch.setattr(K, "PROMPT_PRODUCT", "tiles")
    name = "layer_8b"
    eng = H.engine(name, "bfloat16", max_tokens=64 * 8, n_slots=2)
    assert eng.model.layers[0].ffn.gate_up.packed.gate_rows == 14336
    toks = H.tokens(name, 150, 1)
    s = eng.alloc_slot()
    got = eng.step([(s, toks)], want="all").cpu().double().numpy()
    H.close(got, H.plain_logits(name, toks), "bfloat16", "prompt through the tiled product", config=name)


def test_long_prompts_take_the_tiled_gate_up_product_by_default():
    """From TILES_MIN_ROWS tokens on the gate/up product with its SwiGLU epilogue is the hand-written one;
    the logits are the plain ones either way, and the two ways agree within bfloat16 rounding."""
    import gpu_helpers as H
    assert K.PROMPT_PRODUCT == "auto" and K.tiles_serve_gated(K.TILES_MIN_ROWS, 4096) and not K.tiles_serve_gated(K.TILES_MIN_ROWS - 1, 4096)
    name = "layer_8b"
    eng = H.engine(name, "bfloat16", max_tokens=64 * 18, n_slots=1)
    toks = H.tokens(name, K.TILES_MIN_ROWS + 40, 2)
    calls = []
    real = K.gemm_tiles_bf16
    K.gemm_tiles_bf16 = lambda *a, **kw: (calls.append((a[0].shape[0], a[1].gate_rows > 0)), real(*a, **kw))[1]
    try:
        s = eng.alloc_slot()
        got = eng.step([(s, toks)], want=[[0, 100, len(toks) - 1]]).cpu().double().numpy()
    finally:
        K.gemm_tiles_bf16 = real
    assert calls == [(len(toks), True)] * 2                                # the gate/up product of both layers
    want = H.plain_logits(name, toks)[[0, 100, len(toks) - 1]]
    H.close(got, want, "bfloat16", "long prompt, tiled gate/up product", config=name)


@pytest.mark.parametrize("form", ["few", "tiles64", "tiles128", "tiles256"])
@pytest.mark.parametrize("N,K_", [(20, 8), (132, 72), (260, 264), (64, 1320)])
def test_expert_product_at_the_edges_of_its_tiles(form, N, K_, monkeypatch):
    """Segments of no row, one, and around 16, 64, 128 and 256 rows (in the order of many experts, more than a wave has lanes),
    matrices that fill no tile, k of no whole stage, and more of k than the few-row form asks for at once."""
    monkeypatch.setattr(K, "MOE_PRODUCT", form)
    rng = np.random.default_rng(N)
    sizes = [0, 1, 15, 16, 17, 0, 63, 64, 65, 127, 128, 129, 255, 256, 257, 300] + [0, 1] * 40
    seg = _t(np.concatenate([[0], np.cumsum(sizes)]), torch.int32)
    P, E = sum(sizes), len(sizes)
    order = _t(rng.permutation(P), torch.int32)
    a = _t(rng.standard_normal((P, K_)), torch.bfloat16)
    w = _t(rng.standard_normal((E, N, K_)) * 0.1, torch.bfloat16)
    for gather in (True, False):
        rows = a[order.long()] if gather else a
        want = torch.cat([rows[int(seg[e]):int(seg[e + 1])].double() @ w[e].double().t() for e in range(E)])
        got = K.moe_product(a, w, order, seg, 1, gather, torch.float32)
        # (products of bfloat16 are exact in 32 bits; a sum in any order is off by a few roundings of its partial sums)
        assert (got.double() - want).abs().max() <= 2.0 ** -23 * K_ ** 0.5 * 4 * max(1.0, want.abs().max().item())
        half = K.moe_product(a, w, order, seg, 1, gather, torch.bfloat16, relu2=True)
        _close(half, _np(want.clamp(min=0) ** 2), "bfloat16")


@pytest.mark.parametrize("form", ["few", "tiles64", "tiles128", "tiles256", "auto"])
@pytest.mark.parametrize("N,K_", [(64, 64), (192, 96), (320, 1088), (576, 256)])
def test_expert_product_on_packed_matrices(form, N, K_, monkeypatch):
    """The edges of test_expert_product_at_the_edges_of_its_tiles with the matrices packed, every epilogue and type: columns that fill no tile of
    256, k of no whole round of the ring (and of no whole stage, which the tiles leave to the row-major form); the few-row form gives the
    row-major one's bits."""
    monkeypatch.setattr(K, "MOE_PRODUCT", form)
    rng = np.random.default_rng(N)
    sizes = [0, 1, 15, 16, 17, 0, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 300] + [0, 1] * 40
    seg = _t(np.concatenate([[0], np.cumsum(sizes)]), torch.int32)
    P, E = sum(sizes), len(sizes)
    order = _t(rng.permutation(P), torch.int32)
    a = _t(rng.standard_normal((P, K_)), torch.bfloat16)
    w = _t(rng.standard_normal((E, N, K_)) * 0.1, torch.bfloat16)
    packed = K.pack_experts(w)
    pair = _t(rng.uniform(0.1, 1.0, P))
    for gather in (True, False):
        rows = a[order.long()] if gather else a
        want = torch.cat([rows[int(seg[e]):int(seg[e + 1])].double() @ w[e].double().t() for e in range(E)])
        # (products of bfloat16 are exact in 32 bits; a sum in any order is off by a few roundings of its partial sums)
        bound = 2.0 ** -23 * K_ ** 0.5 * 4 * max(1.0, want.abs().max().item())
        got = K.moe_product(a, w, order, seg, 1, gather, torch.float32, packed=packed)
        assert (got.double() - want).abs().max() <= bound
        if form == "few":
            assert torch.equal(got, K.moe_product(a, w, order, seg, 1, gather, torch.float32))
        _close(K.moe_product(a, w, order, seg, 1, gather, torch.bfloat16, relu2=True, packed=packed), _np(want.clamp(min=0) ** 2), "bfloat16")
        weight = pair[order.long()].double()[:, None]
        gate, up = want[:, 0::2] * weight, want[:, 1::2] * weight
        room = 1.2 * bound * (1 + up.abs().max() + gate.abs().max()) + 2e-6 * (gate.abs() * up.abs()).max()
        got = K.moe_product(a, w, order, seg, 1, gather, torch.float32, gated=True, scale=0.5, pair_weight=pair, packed=packed)
        assert (got.double() - 0.5 * torch.nn.functional.silu(gate) * up).abs().max() <= room
        g, u = want[:, 0::2].clamp(max=0.7), want[:, 1::2].clamp(-0.7, 0.7)
        got = K.moe_product(a, w, order, seg, 1, gather, torch.float32, gated=True, limit=0.7, packed=packed)
        assert (got.double() - g * torch.sigmoid(1.702 * g) * (u + 1)).abs().max() <= room
    assert K.pack_experts(w[:, :N - 32].contiguous()) is None and K.pack_experts(w[:, :, :K_ - 8].contiguous()) is None and K.pack_experts(w.float()) is None


@pytest.mark.parametrize("sizes", [[700, 0, 131, 257, 1, 64], [193, 192, 191], [1025]])
@pytest.mark.parametrize("least,most", [(3, 3), (1, 4), (2, 4), (3, 4)])
def test_expert_tiles_of_chosen_heights(sizes, least, most):
    """Tiles whose height the launch's blocks choose among several, on GPUs of several sizes, so that one round of low tiles, several of high ones and what
    lies between are cheapest in turn: grids sized by the lowest height and shared out by the chosen one; tiles of 192 rows forced."""
    N, K_, E, P = 320, 320, len(sizes), sum(sizes)
    rng = np.random.default_rng(P + least)
    seg = _t(np.concatenate([[0], np.cumsum(sizes)]), torch.int32)
    order = _t(rng.permutation(P), torch.int32)
    a = _t(rng.standard_normal((P, K_)), torch.bfloat16)
    w = _t(rng.standard_normal((E, N, K_)) * 0.1, torch.bfloat16)
    packed, rows = K.pack_experts(w), a[order.long()].double()
    want = torch.cat([rows[int(seg[e]):int(seg[e + 1])] @ w[e].double().t() for e in range(E)])
    bound = 2.0 ** -23 * K_ ** 0.5 * 4 * max(1.0, want.abs().max().item())      # as in test_expert_product_on_packed_matrices
    for units in (1, 4, 8, 16, 24, 40, 64, 256):
        out = torch.full((P, N), float("nan"), device=DEV)
        K._check(K._lib().llogos_moe_product_packed_bf16(K._p(out), K.F32, K._p(a), P, K._p(packed.data), K._p(order), K._p(seg), E, 1, 1, P, N, K_, K_, 0,
                                                         ctypes.c_float(1.0), None, ctypes.c_float(0.0), least, most, units, K._stream()), "moe")
        assert (out.double() - want).abs().max() <= bound, units


@pytest.mark.parametrize("M,N,K_", [(1, 64, 64), (129, 320, 192), (700, 1100, 128), (2100, 2900, 64), (4700, 260, 128)])
def test_tiled_product_places_every_tile_and_adds_itself(M, N, K_):
    """One tile, fewer than XCDs, bands of token tiles that are not full, several rounds of blocks, parts of k: every value is
    written once, in every cut into tiles; with the sum in its epilogue the stream gets the same values added once."""
    gen = torch.Generator(device=DEV).manual_seed(M)
    a = torch.randn((M, K_), device=DEV, generator=gen).to(torch.bfloat16)
    w = (torch.randn((N, K_), device=DEV, generator=gen) * 0.1).to(torch.bfloat16)
    pw = K.pack_weights(w)
    want = a.double() @ w.double().t()
    bound = 2.0 ** -22 * K_ ** 0.5 * max(1.0, want.abs().max().item())      # products exact in 32 bits; partial sums rounded
    x = torch.randn((M, N), device=DEV, generator=gen)
    lib = K._lib()
    for token_tiles in (0, 2, 4):
        for parts in (1, 2, 3):
            if K_ // 64 // parts < 2 and parts > 1:
                continue
            got = K.gemm_tiles_bf16(a, pw, None, torch.float32, parts=parts, token_tiles=token_tiles)
            got = got if parts == 1 else got.sum(0)
            assert (got.double() - want).abs().max() <= bound * 2, (token_tiles, parts)
        y = x.clone()
        K._check(lib.llogos_gemm_tiles_bf16(K._p(y), K.F32, K._p(a), a.stride(0), K._p(pw.data), None, M, N, K_, N, 0, 2, 1, token_tiles,
                                            K.compute_units(a.device), -1.0, K._stream()), "tiles")
        assert torch.equal(y, x + K.gemm_tiles_bf16(a, pw, None, torch.float32, token_tiles=token_tiles)), token_tiles


def test_long_products_of_prompts_add_themselves_to_the_stream():
    """Where the plan takes a long product in one part, the stream gets it in the product's epilogue; elsewhere it is untouched."""
    M, N, K_ = 3400, 4096, 16384
    assert K.tiles_plan(M, N, K_) == (1, 0) and K.tiles_plan(2000, N, K_ + 64) == (2, 0) and K.tiles_plan(M + 512, N, K_) is None
    a = torch.randn((M, K_), device=DEV).to(torch.bfloat16)
    w = (torch.randn((N, K_), device=DEV) * 0.02).to(torch.bfloat16)
    pw, x = K.pack_weights(w), torch.randn((M, N), device=DEV)
    y = x.clone()
    assert K.gemm_tiles_add(y, a, pw)
    assert (y - (x + a.float() @ w.float().t())).abs().max() <= 2e-3
    kept = y.clone()
    assert not K.gemm_tiles_add(y[:M - 1000], a[:M - 1000], pw) and not K.gemm_tiles_add(y, a.float(), pw) and not K.gemm_tiles_add(y, a, None)
    assert torch.equal(y, kept)


@pytest.mark.parametrize("M,N,K_", [(1, 1, 64), (65, 300, 128), (64, 256, 192), (130, 515, 448), (191, 2048, 2048), (193, 4160, 320), (70, 64, 4096), (400, 1030, 576)])
def test_short_tiled_product_at_the_edges_of_its_tiles(M, N, K_):
    """Tiles of 64, 128 and 192 tokens: rows and columns at remainders of tiles, one stage of k and several, every split that leaves a
    part two stages; the sums are the larger tiles' bit for bit, in float32 and bfloat16, and right."""
    rng = np.random.default_rng(M + N)
    wide = _t(rng.standard_normal((M, K_ + 8)), torch.bfloat16)
    a, w = wide[:, :K_], _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    pw = K.pack_weights(w)
    want = a.double() @ w.double().t()
    bound = 1e-6 * (a.double().abs() @ w.double().abs().t()).max()      # float32 sums of bfloat16 products: 2^-24 a step of an operand's chain
    for parts in [p for p in range(1, 9) if p == 1 or K_ // 64 // p >= 2]:
        big = K.gemm_tiles_bf16(a, pw, None, torch.float32, parts=parts, token_tiles=2)
        for token_tiles in (1, 2, 3):
            got = K.gemm_tiles_bf16(a, pw, None, torch.float32, parts=parts, token_tiles=token_tiles)
            assert torch.equal(got, big), (parts, token_tiles)
        assert ((got.double().sum(0) if parts > 1 else got.double()) - want).abs().max() <= bound * parts
    for token_tiles in (1, 2, 3):
        assert torch.equal(K.gemm_tiles_bf16(a, pw, None, torch.bfloat16, token_tiles=token_tiles), K.gemm_tiles_bf16(a, pw, None, torch.bfloat16, token_tiles=2))
    assert K.gemm_wide_bf16(a, pw, torch.float32, K_ // 64) is None or K_ == 64                 # parts of one stage
    assert K.gemm_wide_bf16(a.float(), pw, torch.float32, 1) is None


@pytest.mark.parametrize("M,N,K_", [(1, 32, 64), (97, 512, 128), (255, 544, 320), (256, 260, 256), (257, 1024, 576), (161, 96, 1088), (450, 1088, 192)])
def test_tiles_of_every_height_and_epilogue(M, N, K_):
    """Tiles of 64, 96, .. 256 tokens: rows and columns at remainders, one stage of k to several rounds of the ring of four and what is left of one,
    rows of a wider than k, results narrower than whole lines, every epilogue.  Every height gives the same bits; they are right."""
    rng = np.random.default_rng(M * N)
    lib = K._lib()
    wide = _t(rng.standard_normal((M, K_ + 8)), torch.bfloat16)
    a, w = wide[:, :K_], _t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16)
    pw, pg = K.pack_weights(w), (K.pack_weights(w, gate_rows=N // 2) if N % 32 == 0 else None)
    exact = a.double() @ w.double().t()
    bound = 1e-6 * (a.double().abs() @ w.double().abs().t()).max()      # float32 sums of bfloat16 products: 2^-24 a step of an operand's chain
    x = _t(rng.standard_normal((M, N)))
    gate, up = exact[:, :N // 2], exact[:, N // 2:]
    seen = None
    for token_tiles in (1, 6, 2, 10, 3, 14, 4, 0):
        def call(out, packed, epilogue, parts=1, limit=-1.0):
            K._check(lib.llogos_gemm_tiles_bf16(K._p(out), K._DT[out.dtype], K._p(a), a.stride(0), K._p(packed.data), None, M, N, K_, out.shape[-1],
                                                ctypes.c_longlong(M * out.shape[-1]), epilogue, parts, token_tiles, 256, ctypes.c_float(limit), K._stream()), "tiles")
            return out
        empty = lambda *shape, dtype=torch.float32: torch.full(shape, float("nan"), device=DEV, dtype=dtype)
        got = [call(empty(M, N), pw, 0), call(empty(M, N, dtype=torch.bfloat16), pw, 0), call(x.clone(), pw, 2)]
        assert (got[0].double() - exact).abs().max() <= bound and torch.equal(got[1], got[0].bfloat16()) and torch.equal(got[2], x + got[0])
        for parts in (2, 3):
            if K_ // 64 // parts >= 2:
                split = call(empty(parts, M, N), pw, 0, parts)
                assert (split.double().sum(0) - exact).abs().max() <= bound * parts
                got.append(split)
        if pg is not None:
            got += [call(empty(M, N // 2), pg, 1), call(empty(M, N // 2, dtype=torch.bfloat16), pg, 1), call(empty(M, N // 2), pg, 1, limit=0.7)]
            # (the product's own error through silu, whose slope is below 1.1, and a few roundings of the rest)
            room = 1.2 * bound * (1 + up.abs().max() + gate.abs().max()) + 2e-6 * (gate.abs() * up.abs()).max()
            assert (got[-3].double() - torch.nn.functional.silu(gate) * up).abs().max() <= room and torch.equal(got[-2], got[-3].bfloat16())
            g, u = gate.clamp(max=0.7), up.clamp(-0.7, 0.7)
            assert (got[-1].double() - g * torch.sigmoid(1.702 * g) * (u + 1)).abs().max() <= room + 4 * bound
        seen = seen or got
        assert all(torch.equal(p, q) for p, q in zip(seen, got)), token_tiles


@pytest.mark.parametrize("M,N,K_", [(1, 8, 64), (130, 300, 320), (257, 517, 192), (700, 1088, 576)])
def test_tiles_that_activate_their_product(M, N, K_):
    """The activation in the product's epilogue gives the bits of the activation's kernel on the float32 product, in heights of tiles that the launch
    chooses for the sizes, results at remainders of their lines, and for sums that are no number; other kinds are left alone."""
    rng = np.random.default_rng(M + N)
    a, w = _t(rng.standard_normal((M, K_)) * 2, torch.bfloat16), _t(rng.standard_normal((N, K_)) * 0.1, torch.bfloat16)
    a[M // 2, 3], a[M - 1, K_ - 1] = float("inf"), float("nan")
    pw = K.pack_weights(w)
    z = K.gemm_tiles_bf16(a, pw, None, torch.float32)
    for kind, numbers in (("relu2", ()), ("xielu", (0.8, 1.1))):
        got, want = K.gemm_tiles_activated(a, pw, kind, *numbers), K.activation(z, kind, torch.bfloat16, *numbers)
        number = ~torch.isnan(want)
        assert got.dtype == torch.bfloat16 and torch.equal(torch.isnan(got), ~number) and torch.equal(got[number], want[number])
    assert K.gemm_tiles_activated(a, pw, "silu") is None and K.gemm_tiles_activated(a.float(), pw, "relu2") is None


def test_wide_tiles_serve_prompts():
    """What prompt_parts chooses, through the general entry and added to the stream: one part in place, more parts left to the norm that
    adds them, none to the library; matrices and operands that it does not take go the way they went."""
    for M, N, K_ in ((800, 3072, 3072), (2048, 4096, 14336), (300, 512, 4096), (700, 8320, 4096), (1100, 5120, 16384)):
        parts = K.prompt_parts(M, N, K_)
        a, w = torch.randn((M, K_), device=DEV).bfloat16(), (torch.randn((N, K_), device=DEV) * 0.05).bfloat16()
        pw, x0 = K.pack_weights(w), torch.randn((M, N), device=DEV)
        want = a.double() @ w.double().t()
        got = K.gemm_product(a, w, torch.bfloat16, f32_ok=True, packed=pw)
        assert parts and got.dtype == torch.float32 and got.shape == ((M, N) if parts == 1 else (parts, M, N))
        total = got.double() if parts == 1 else got.double().sum(0)
        assert (total - want).abs().max() <= 2e-5 * want.abs().max()
        x = x0.clone()
        adds = K.prompt_parts(M, N, K_, adds=True)
        assert K.gemm_wide_add(x, a, pw) == (adds == 1)
        if adds > 1:
            assert not K.gemm_library_add(x, a, w, pw) and torch.equal(x, x0)
        elif adds == 0:
            assert K.gemm_library_add(x, a, w, pw)
        assert adds > 1 or (x.double() - x0.double() - want).abs().max() <= 2e-5 * want.abs().max()
        x = x0.clone()
        assert not K.gemm_wide_add(x[:, :N - 4], a, pw) and not K.gemm_wide_add(x, a.float(), pw) and not K.gemm_wide_add(x.t(), a, pw) and torch.equal(x, x0)
        odd = torch.randn((M, K_ + 4), device=DEV).bfloat16()[:, 4:]          # rows that are not 16 bytes apart
        assert K.gemm_wide_bf16(odd, pw, torch.float32, 1) is None
        got = K.gemm_product(odd, w, torch.bfloat16, f32_ok=True, packed=pw)
        assert (got.double() - odd.double() @ w.double().t()).abs().max() <= 2e-5 * want.abs().max() * (1 if got.dtype == torch.float32 else 500)


def test_short_tiled_product_serves_prompts_of_some_hundred_rows():
    """What prompt_parts chooses for some hundred rows, through the general entry: in parts or not, with the rows of a product that adds itself left
    to the norm."""
    for M, N, K_ in ((65, 2048, 2048), (128, 8192, 2048), (256, 3072, 2112), (257, 2048, 4096), (1024, 2048, 8192)):
        parts = K.prompt_parts(M, N, K_)
        a, w = torch.randn((M, K_), device=DEV).bfloat16(), (torch.randn((N, K_), device=DEV) * 0.05).bfloat16()
        pw = K.pack_weights(w)
        got = K.gemm_product(a, w, torch.bfloat16, f32_ok=True, packed=pw)
        assert got.dtype == torch.float32 and parts > 1 and got.shape == (parts, M, N)
        want = a.double() @ w.double().t()
        assert (got.double().sum(0) - want).abs().max() <= 2e-5 * want.abs().max()
        x = torch.zeros((M, N), device=DEV)
        assert not K.gemm_tiles_add(x, a, pw) and not K.gemm_library_add(x, a, w, pw) and not x.any()


@pytest.mark.parametrize("M,N,K_", [(129, 2048, 2048), (200, 4096, 4096), (256, 3072, 2112)])
def test_products_that_no_norm_follows_are_added_by_the_library(M, N, K_):
    """Where the tiled product would leave parts for a norm to add and none follows, the library's product adds itself to the stream: the
    float32 product added to x, bit for bit; with a norm behind it, and up to 128 rows, it does not and x stays as it was."""
    base = importlib.import_module("daisi-llogos_amd.parts.base")
    parts = importlib.import_module("daisi-llogos_amd.parts")
    a, w = torch.randn((M, K_), device=DEV).bfloat16(), (torch.randn((N, K_), device=DEV) * 0.05).bfloat16()
    pw, x0 = K.pack_weights(w), torch.randn((M, N), device=DEV)
    assert K.prompt_parts(M, N, K_) > 1
    want = x0 + torch.mm(a, w.t(), out_dtype=torch.float32)
    x = x0.clone()
    assert K.gemm_library_add(x, a, w, pw, norm_adds=False) and torch.equal(x, want)
    x = x0.clone()
    assert not K.gemm_library_add(x, a, w, pw) and not K.gemm_library_add(x[:128], a[:128], w, pw, norm_adds=False) and torch.equal(x, x0)
    lin = parts.Linear(["o"], K_, [N])
    lin.bind(lambda name: w, base.Runtime(torch.device(DEV), torch.bfloat16))
    left = lin.add_to(a, base.Residual(x, None))
    assert isinstance(left, K.RowSquares) and left.sums is None and torch.equal(x, want)
    x = x0.clone()
    norm = parts.RMSNorm("n", N, 1e-5)
    assert lin.add_to(a, base.Residual(x, norm)) is None and torch.equal(x, x0)


@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 16, 33, 64])
@pytest.mark.parametrize("N", [65, 66, 67, 1087])
def test_few_row_results_stored_by_fours_and_one_by_one(N, M, out_dtype):
    """Rows of a multiple of four values are stored four at a time, others (and a row's last few) value by value: the same bits, bias and all."""
    rng = np.random.default_rng(N + M)
    a, w = _t(rng.standard_normal((M, 520)), torch.bfloat16), _t(rng.standard_normal((N + 3, 520)) * 0.05, torch.bfloat16)
    b = _t(rng.standard_normal(N + 3))
    few = K.gemm_packed_bf16(a, K.pack_weights(w[:N].contiguous()), b[:N].contiguous(), out_dtype)
    whole = N + -N % 4
    more = K.gemm_packed_bf16(a, K.pack_weights(w[:whole].contiguous()), b[:whole].contiguous(), out_dtype)
    assert few.shape == (1, M, N) and torch.equal(few, more[:, :, :N])
    _close(few[0], _np(a) @ _np(w[:N]).T + _np(b[:N]), "float32" if out_dtype == torch.float32 else "bfloat16")


@pytest.mark.parametrize("G,M,N,K_", [(4, 1, 64, 8), (4, 8, 256, 1024), (3, 17, 192, 520), (2, 33, 4096, 2048), (4, 64, 128, 4096), (4, 8, 4096, 4096)])
def test_products_of_one_shape_in_one_launch(G, M, N, K_):
    """Each of the group is the product by itself, in the parts that its own plan gives it, bit for bit; the single copies still serve alone."""
    rng = np.random.default_rng(N + M)
    a = _t(rng.standard_normal((G + 1, M, K_)), torch.bfloat16)[1:]
    ws = [_t(rng.standard_normal((N, K_)) * 0.05, torch.bfloat16) for _ in range(G)]
    packed = [K.pack_weights(w) for w in ws]
    data = K.pack_together(packed)
    got = K.gemm_packed_group_bf16(a, data, N)
    splits, chunk = K.packed_plan(M, N, K_)
    for g in range(G):
        alone = K.gemm_packed_bf16(a[g], packed[g], None, torch.float32, splits, chunk)
        assert torch.equal(got[g], alone)
        _close(got[g].sum(0), _np(a[g]) @ _np(ws[g]).T, "float32", scale=np.abs(_np(a[g]) @ _np(ws[g]).T).max() * 10)
    assert K.gemm_packed_group_bf16(torch.zeros((G, 65, K_), device=DEV, dtype=torch.bfloat16), data, N) is None
    assert K.pack_together([packed[0], None]) is None and K.pack_together([K.pack_weights(ws[0][:40])] * 2) is None
