"""Rows, planes and channel counts that are not whole 16-byte vectors, and
operands that are not 16-byte aligned, against the C oracle.

Every call goes through the C entry points with operands inside larger
buffers, so that a store outside the output changes a guard value; offsets of
one element make every pointer misaligned."""
import pytest
import torch

pytestmark = pytest.mark.gpu

GUARD = 64  # elements around every output


class Guarded:
    """A tensor of `shape` at element offset GUARD + shift of a buffer whose
    other elements hold a guard value."""

    def __init__(self, shape, dtype, dev, shift=0):
        n = 1
        for d in shape:
            n *= d
        self.buf = torch.full((n + 2 * GUARD + shift,), 3.0, dtype=dtype, device=dev)
        self.lo, self.hi = GUARD + shift, GUARD + shift + n
        self.t = self.buf[self.lo:self.hi].view(shape)

    def check(self, what):
        assert bool((self.buf[:self.lo] == 3).all()), f"{what}: written before the output"
        assert bool((self.buf[self.hi:] == 3).all()), f"{what}: written past the output"


def place(t, dev, shift):
    """t on the device, `shift` elements off its allocation's alignment."""
    g = Guarded(t.shape, t.dtype, dev, shift)
    g.t.copy_(t)
    return g.t


def lib():
    import hip_oracles
    return hip_oracles.load_library()


def ok(rc):
    assert rc == 0, lib().hipo_last_error()


def close(got, want, rtol, atol, what):
    g, w = got.float().cpu(), want.float()
    assert torch.allclose(g, w, rtol=rtol, atol=atol, equal_nan=True), (
        f"{what}: max |diff| {(g - w).abs().max().item():.3e}")


# One 16-byte group, one value more and one less; the ends of the short-row
# kernel (512) and of its lane counts; ViT and CLIP rows; several waves per
# row; the longest row held in registers is 32768 (past it, the general one).
SOFTMAX_K = [7, 8, 9, 15, 17, 50, 77, 127, 129, 197, 257, 511, 513, 577, 1023, 1025, 1500, 2047,
             4099, 8195]


@pytest.mark.parametrize("k", SOFTMAX_K)
def test_softmax_any_row_length(k, rocm_device):
    """bf16 results: relative 2^-8 is one bf16 ulp, twice that where kernel
    and oracle round to different sides of a boundary."""
    import oracle as ref
    torch.manual_seed(k)
    b, heads, q = 4, 2, 5
    x = torch.randn(b, q, k).to(torch.bfloat16)
    mask = torch.zeros(q, k, dtype=torch.bfloat16)
    mask[torch.arange(k)[None, :] > torch.arange(q)[:, None] + k - q] = float("-inf")
    mask[2, k // 2:] = float("-inf")
    bias = torch.randn(b // heads, q, k).to(torch.bfloat16)
    for shift in (0, 1):
        xd, md, bd = (place(t, rocm_device, shift) for t in (x, mask, bias))
        out = Guarded((b, q, k), torch.bfloat16, rocm_device, shift)
        ok(lib().hipo_scaled_masked_softmax_bf16(xd.data_ptr(), md.data_ptr(), out.t.data_ptr(),
                                                 b, q, k, k, 0.125, None))
        torch.cuda.synchronize()
        out.check(f"masked K={k}")
        close(out.t, ref.scaled_masked_softmax(x, mask, 0.125), 2 ** -7, 1e-6, f"masked K={k}")
        out = Guarded((b, q, k), torch.bfloat16, rocm_device, shift)
        ok(lib().hipo_scaled_bias_softmax_bf16(xd.data_ptr(), bd.data_ptr(), out.t.data_ptr(), b,
                                               q, k, k, q * k, heads, 0.5, None))
        torch.cuda.synchronize()
        out.check(f"bias K={k}")
        close(out.t, ref.scaled_bias_softmax(x, bias, 0.5, heads), 2 ** -7, 1e-6, f"bias K={k}")


# Both sides of the lines where few short rows off the vector path go value by
# value (2048 rows, and 256 of up to 16 values), and every lane count past them.
@pytest.mark.parametrize("b,q,k,shift", [
    (1, 256, 9, 0), (1, 257, 9, 0), (4, 512, 12, 0), (3, 683, 12, 0), (2, 1024, 17, 0),
    (2049, 1, 17, 0), (683, 3, 33, 0), (683, 3, 50, 0), (4, 512, 64, 1), (683, 3, 64, 1),
    (3, 700, 8, 1), (3, 700, 16, 1), (8, 16, 65, 0)])
def test_softmax_few_short_rows(b, q, k, shift, rocm_device):
    import oracle as ref
    torch.manual_seed(b + q + k)
    x = torch.randn(b, q, k).to(torch.bfloat16)
    x[0, 0, k - 1] = float("inf")
    mask = torch.randn(q, k).to(torch.bfloat16)
    mask[q // 2, : k - 1] = float("-inf")
    xd, md = place(x, rocm_device, shift), place(mask, rocm_device, shift)
    out = Guarded((b, q, k), torch.bfloat16, rocm_device, shift)
    ok(lib().hipo_scaled_masked_softmax_bf16(xd.data_ptr(), md.data_ptr(), out.t.data_ptr(), b, q,
                                             k, k, 0.125, None))
    torch.cuda.synchronize()
    out.check(f"[{b}, {q}, {k}]")
    close(out.t, ref.scaled_masked_softmax(x, mask, 0.125), 2 ** -7, 1e-6, f"[{b}, {q}, {k}]")


@pytest.mark.parametrize("k", [9, 197, 577, 1025])
def test_softmax_odd_rows_special_values(k, rocm_device):
    """A row that is -inf throughout is NaN; NaN and +inf scores make their
    row NaN and no other."""
    import hip_oracles
    torch.manual_seed(k)
    x = torch.randn(6, k).to(torch.bfloat16)
    x[1] = float("-inf")
    x[2, k - 1] = float("nan")
    x[3, k - 2] = float("inf")
    x[4, : k - 1] = float("-inf")
    got = hip_oracles.softmax_lastdim(x.to(rocm_device)).float().cpu()
    assert bool(got[1:4].isnan().all())
    want = torch.softmax(x.double(), -1).to(torch.bfloat16).float()
    for r in (0, 4, 5):
        close(got[r], want[r], 2 ** -7, 1e-6, f"row {r}")


def test_softmax_zero_row_is_one_and_ready_for_every_stream(rocm_device, monkeypatch):
    """softmax_lastdim's mask row: one per device whatever row lengths come,
    filled before any other stream can use it (the first call waits for the
    stream that fills it, here behind other work), longer ones on demand."""
    import hip_oracles
    monkeypatch.setattr(hip_oracles, "_zero_rows", {})
    monkeypatch.setattr(hip_oracles, "_old_zero_rows", [])
    x = torch.randn(64, 500).to(torch.bfloat16).to(rocm_device)
    want = torch.softmax(x.double(), -1).to(torch.bfloat16).float().cpu()
    a = torch.randn(4096, 4096, device=rocm_device)
    torch.cuda.synchronize()
    side = torch.cuda.Stream(rocm_device)
    with torch.cuda.stream(side):
        for _ in range(8):
            a = a @ a
            a = a / a.abs().max()
        event = torch.cuda.Event()
        event.record()
        first = hip_oracles.softmax_lastdim(x)
    assert event.query(), "the zero row was published before it was filled"
    close(hip_oracles.softmax_lastdim(x), want, 2 ** -7, 1e-6, "another stream")
    torch.cuda.synchronize()
    close(first, want, 2 ** -7, 1e-6, "the filling stream")
    for k in (1, 7, 197, 32768):
        hip_oracles.softmax_lastdim(torch.zeros(2, k, dtype=torch.bfloat16, device=rocm_device))
    assert [r.numel() for r in hip_oracles._zero_rows.values()] == [32768]
    assert not hip_oracles._old_zero_rows
    x = torch.randn(2, 33000).to(torch.bfloat16)
    close(hip_oracles.softmax_lastdim(x.to(rocm_device)),
          torch.softmax(x.double(), -1).to(torch.bfloat16).float(), 2 ** -7, 1e-6, "33000")
    assert [r.numel() for r in hip_oracles._zero_rows.values()] == [65536]
    assert [r.numel() for r in hip_oracles._old_zero_rows] == [32768]


# (channels, positions): one block each way, one value more, odd planes, more
# block columns than a tile's 8 and fewer rows, thin output rows, fewer values
# than a block (the one-element kernel).  One image, and 2^19 and 2^21 elements:
# past the tile kernel's minimum, and with enough ragged images for it to pay
# (from 65 x 49 on; smaller images go one element per thread at every count).
BIAS_GELU_CP = [(8, 8), (9, 8), (8, 9), (65, 49), (64, 196), (100, 25), (16, 1001), (230, 77),
                (513, 17), (7, 500), (300, 7)]


@pytest.mark.parametrize("c,hw", BIAS_GELU_CP)
def test_bias_gelu_any_plane(c, hw, rocm_device):
    """Both sides hold the correctly rounded bf16: equal bit for bit."""
    import oracle as ref
    torch.manual_seed(c * 1000 + hw)
    for n in (1, (1 << 19) // (c * hw) + 2, (1 << 21) // (c * hw) + 2):
        x = torch.randn(n, c, 1, hw).to(torch.bfloat16) * 3
        bias = torch.randn(c).to(torch.bfloat16)
        want = ref.bias_gelu_nchw_to_nhwc(x, bias).permute(0, 2, 3, 1)
        for shift in (0, 1):
            xd, bd = place(x, rocm_device, shift), place(bias, rocm_device, shift)
            out = Guarded((n, 1, hw, c), torch.bfloat16, rocm_device, shift)
            ok(lib().hipo_bias_gelu_nchw_to_nhwc_bf16(xd.data_ptr(), bd.data_ptr(),
                                                      out.t.data_ptr(), n, c, hw, None))
            torch.cuda.synchronize()
            out.check(f"[{n}, {c}, {hw}]")
            assert torch.equal(out.t.cpu(), want), f"[{n}, {c}, {hw}] shift {shift}"


# Matrices past the whole-matrix kernel's 32 KiB: sides of exactly one block,
# one element more, odd on either side or both, thin ones (general kernel).
TRANSPOSE_RC = [(8, 4096), (4096, 8), (9, 2500), (2500, 9), (197, 768), (768, 197), (333, 129),
                (129, 333), (1001, 65), (3, 20000), (20000, 3), (200, 200)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["b16", "b32"])
@pytest.mark.parametrize("r,c", TRANSPOSE_RC)
def test_transpose_any_matrix(r, c, dtype, rocm_device):
    torch.manual_seed(r * 7 + c)
    x = torch.randn(3, r, c).to(dtype)
    for shift in (0, 1):
        xd = place(x, rocm_device, shift)
        out = Guarded((3, c, r), dtype, rocm_device, shift)
        ok(lib().hipo_transpose_last2(xd.data_ptr(), out.t.data_ptr(), 3, r, c,
                                      x.element_size(), None))
        torch.cuda.synchronize()
        out.check(f"[{r}, {c}]")
        assert torch.equal(out.t.cpu(), x.transpose(1, 2).contiguous()), f"[{r}, {c}]"


# Every cache policy of the register-block transposes: rows of whole cache lines
# both ways up to 32 MB read and written and beyond 160 MB (non-temporal; in
# plain workgroup order where four tiles cover the output rows, XCD order
# otherwise), between the two (non-temporal stores), and rows that are not whole
# lines beyond 160 MB (cached).
@pytest.mark.parametrize("batch,r,c,dtype", [
    (2, 512, 384, torch.bfloat16), (2, 256, 192, torch.float32), (40, 512, 512, torch.bfloat16),
    (161, 256, 1024, torch.bfloat16), (161, 128, 1024, torch.float32),
    (81, 1024, 512, torch.bfloat16), (161, 520, 500, torch.bfloat16),
    # output rows of whole 16, 32 and 64 bytes, the second below and beyond 32 MB
    (3, 500, 72, torch.float32), (62, 1000, 64, torch.float32), (63, 1000, 64, torch.float32),
    (70, 2000, 66, torch.float32), (5, 4968, 64, torch.bfloat16)])
def test_transpose_cache_policies(batch, r, c, dtype, rocm_device):
    g = torch.Generator(device=rocm_device).manual_seed(r + c)
    bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
    x = torch.randint(-2 ** 15, 2 ** 15, (batch, r, c), generator=g, device=rocm_device).to(bits)
    out = Guarded((batch, c, r), bits, rocm_device)
    ok(lib().hipo_transpose_last2(x.data_ptr(), out.t.data_ptr(), batch, r, c, x.element_size(),
                                  None))
    torch.cuda.synchronize()
    out.check(f"[{batch}, {r}, {c}]")
    assert torch.equal(out.t, x.transpose(1, 2)), f"[{batch}, {r}, {c}]"


# (n, c, hw): planes of whole float4s and not, value by value (below 9), one
# vector a thread and many, the 1024-thread kernel from 16385 values on (both
# kinds, its largest), split-K past it, with one plane and with many.
BN_TRAIN = [(3, 5, 7), (3, 5, 9), (4, 5, 12), (26, 9, 49), (334, 3, 49), (335, 3, 49), (128, 40, 196),
            (146, 33, 196), (147, 33, 196), (1820, 2, 9), (2000, 3, 13), (17, 6, 1295), (5, 3, 9999),
            (1, 4, 50001), (60, 2, 1023), (9000, 2, 3), (700, 2, 70),
            # 9 vectors a thread: split-K for few channels of long planes only
            (16, 3, 2209), (16, 32, 2209), (900, 2, 41)]


@pytest.mark.parametrize("n,c,hw", BN_TRAIN)
def test_batchnorm_train_any_plane(n, c, hw, rocm_device):
    """fp32 statistics of exact two-pass pieces merged by Chan's formula:
    1e-5 holds with a margin of over ten."""
    import hip_oracles
    import oracle as ref
    torch.manual_seed(n + c + hw)
    x = torch.randn(n, c, 1, hw) * 2 + 0.5
    gamma, beta = torch.randn(c), torch.randn(c)
    for shift, relu in ((0, True), (1, False)):
        rm, rv = torch.randn(c), torch.rand(c) + 0.5
        want = ref.batchnorm_train(x, gamma, beta, rm.clone(), rv.clone(), momentum=0.1, eps=1e-5,
                                   relu=relu)
        xd = place(x, rocm_device, shift)
        y = Guarded(x.shape, torch.float32, rocm_device, shift)
        side = [t.to(rocm_device) for t in (gamma, beta, rm, rv)]
        mean, invstd = (torch.empty(c, device=rocm_device) for _ in range(2))
        need = hip_oracles.batchnorm_workspace_bytes(n, c, hw)
        ws = torch.zeros(need, dtype=torch.uint8, device=rocm_device)
        ok(lib().hipo_batchnorm_train_fwd_f32(
            xd.data_ptr(), *(t.data_ptr() for t in side), y.t.data_ptr(), mean.data_ptr(),
            invstd.data_ptr(), n, c, hw, 0.1, 1e-5, int(relu), ws.data_ptr(), need, None))
        torch.cuda.synchronize()
        y.check(f"[{n}, {c}, {hw}]")
        got = (y.t, mean, invstd, side[2], side[3])
        for name, a, b in zip(("y", "mean", "invstd", "running_mean", "running_var"), got, want):
            close(a, b, 1e-5, 1e-5, f"[{n}, {c}, {hw}] shift {shift} {name}")


@pytest.mark.parametrize("hw", [28672, 28671], ids=["whole", "ragged"])
def test_batchnorm_train_large_channels_merge_in_fp64(hw, rocm_device):
    """The 1024-thread register kernel: each of its 16 waves (wave w holds the
    float4s i with i % 1024 // 64 == w) sees one 18-bit value only, so its sum,
    its mean and its merge over the lanes are exact and the waves' fp64 merge
    is the one that rounds: every statistic is the fp64 one rounded to fp32."""
    import hip_oracles
    import numpy as np
    c = 64
    g = torch.Generator().manual_seed(7)
    per_wave = (torch.randint(1 << 17, 1 << 18, (c, 16), generator=g).double()
                * 2.0 ** torch.randint(-20, -8, (c, 16), generator=g).double()
                * (torch.randint(0, 2, (c, 16), generator=g) * 2 - 1))
    wave = torch.arange(hw) // 4 % 1024 // 64
    x = per_wave[:, wave].float().view(1, c, 1, hw)
    assert torch.equal(x.double().view(c, hw), per_wave[:, wave])
    rm, rv = torch.zeros(c, device=rocm_device), torch.zeros(c, device=rocm_device)
    ones = torch.ones(c, device=rocm_device)
    _, mean, invstd = hip_oracles.batchnorm_train(x.to(rocm_device), ones, rm.clone(), rm, rv,
                                                  momentum=0.5, eps=1e-5, relu=False)
    x64 = x.double().view(c, hw).numpy()
    mean64, var64 = x64.mean(1), x64.var(1)
    assert np.array_equal(mean.cpu().numpy(), mean64.astype(np.float32))
    assert np.array_equal(rm.cpu().numpy(), (0.5 * mean64).astype(np.float32))
    assert np.array_equal(rv.cpu().numpy(), (0.5 * var64 * hw / (hw - 1)).astype(np.float32))
    # var and var + eps rounded to fp32, then one square root and one division
    want = 1 / np.sqrt(var64.astype(np.float32) + np.float32(1e-5))
    assert np.abs(invstd.cpu().numpy() / want - 1).max() < 2.0 ** -22


@pytest.mark.parametrize("n", [1, 3])
def test_batchnorm_train_infinity_in_the_first_split(n, rocm_device):
    """An infinite value gives an infinite channel mean where the merges
    inside a workgroup keep it (it comes last in their order; in any other
    place Chan's formula meets inf - inf), and NaN elsewhere, never a finite
    one: the merge of the splits loses neither, also for the first split.  256
    channels have it in one each of a workgroup's 256 threads, in the first
    plane."""
    import hip_oracles
    c, hw = 256, 50001
    x = torch.randn(n, c, 1, hw, device=rocm_device)
    for t in range(c):  # vector 12032 + t: thread t's, the last one for t > 212
        x[0, t, 0, 4 * (12032 + t)] = float("inf")
    rm, rv = torch.zeros(c, device=rocm_device), torch.ones(c, device=rocm_device)
    y, mean, invstd = hip_oracles.batchnorm_train(
        x, torch.ones_like(rm), torch.zeros_like(rm), rm, rv, momentum=0.1, eps=1e-5, relu=False)
    assert not bool(torch.isfinite(mean).any())
    assert bool((mean == float("inf")).any())
    assert bool(((rm == float("inf")) == (mean == float("inf"))).all())
    assert bool(torch.isnan(invstd).all()) and bool(torch.isnan(rv).all())


# One group, one value more and less; the ends of the lane counts and of the
# short-row kernels (512, 1536); several waves and groups per row; value by
# value (below 8).
NORM_COLS = [7, 8, 9, 63, 64, 65, 100, 128, 180, 257, 511, 512, 513, 769, 1025, 1535, 2530, 4096,
             4796, 7842, 16385]


@pytest.mark.parametrize("cols", NORM_COLS)
def test_norms_any_row_length(cols, rocm_device):
    """Statistics 1e-5; bf16 results within 2^-7 (two ulps where kernel and
    oracle round to different sides twice), 1e-2 near zero for LayerNorm,
    whose terms cancel there."""
    import oracle as ref
    torch.manual_seed(cols)
    L = lib()
    for rows in ((3, 16400) if cols in (513, 769, 1535) else (1, 37)):
        x, r = (torch.randn(rows, cols).to(torch.bfloat16) for _ in range(2))
        g, b = (1 + 0.1 * torch.randn(cols)).to(torch.bfloat16), torch.randn(cols).to(torch.bfloat16)
        hw, yw, mw, sw = ref.residual_layernorm(x, r, g, b, 1e-5)
        for shift in (0, 1):
            what = f"[{rows}, {cols}] shift {shift}"
            xd, rd, gd, bd = (place(t, rocm_device, shift) for t in (x, r, g, b))
            h, y = (Guarded((rows, cols), torch.bfloat16, rocm_device, shift) for _ in range(2))
            mean, rstd = (Guarded((rows,), torch.float32, rocm_device) for _ in range(2))
            ok(L.hipo_residual_layernorm_bf16(
                xd.data_ptr(), rd.data_ptr(), gd.data_ptr(), bd.data_ptr(), h.t.data_ptr(),
                y.t.data_ptr(), mean.t.data_ptr(), rstd.t.data_ptr(), rows, cols, 1e-5, None))
            torch.cuda.synchronize()
            for o in (h, y, mean, rstd):
                o.check("layernorm " + what)
            assert torch.equal(h.t.cpu(), hw), what
            close(y.t, yw, 2 ** -7, 1e-2, "layernorm y " + what)
            close(mean.t, mw, 1e-5, 1e-5, "mean " + what)
            close(rstd.t, sw, 1e-5, 1e-5, "rstd " + what)
            for mode, scale, res in ((0, 1.0, None), (1, 0.125, rd), (0, 0.5, rd), (1, 1.0, None)):
                want = ref.rmsnorm_ex(x, g, 1e-6, residual=None if res is None else r,
                                      scale=scale, mode=mode)
                h, y = (Guarded((rows, cols), torch.bfloat16, rocm_device, shift)
                        for _ in range(2))
                ok(L.hipo_rmsnorm_ex_bf16(
                    xd.data_ptr(), None if res is None else res.data_ptr(), gd.data_ptr(),
                    None if res is None else h.t.data_ptr(), y.t.data_ptr(), rstd.t.data_ptr(),
                    rows, cols, 1e-6, scale, mode, None))
                torch.cuda.synchronize()
                for o in (h, y, rstd):
                    o.check(f"rmsnorm mode {mode} " + what)
                if res is not None:
                    assert torch.equal(h.t.cpu(), hw), what
                close(y.t, want[0], 2 ** -6 if mode else 2 ** -7, 1e-6, f"rmsnorm {mode} " + what)


# (n, c, hw): one group, one channel more and less, channel counts over several
# blocks of groups, one position, fewer positions than rows per instruction.
SPATIAL = [(2, 7, 9), (2, 8, 9), (3, 9, 1), (3, 15, 49), (4, 29, 3190), (2, 61, 700), (130, 1001, 49),
           (6, 1759, 196), (1, 514, 50), (2, 8193, 4), (300, 33, 100),
           # ragged plan and thread per output, on both sides of the line
           (2100, 500, 1), (3000, 9, 4), (1500, 250, 9), (600, 250, 9), (2, 8200, 7),
           # whole groups: as many rows as give a thread its loads, one row, two.
           # Powers of two positions: the sum times 1 / P is exact and rounds
           # once, as in the oracle; other counts round twice, and among as many
           # outputs some lie an ulp off, 2^-7 of a value just above a power of 2
           # ([3, 1000, 13]: 2^-9 at 0.27).
           (3, 168, 4), (3, 168, 8), (5, 232, 64), (3, 1000, 8), (3, 1000, 16), (767, 1240, 16),
           (768, 1240, 16), (769, 1000, 64)]


@pytest.mark.parametrize("n,c,hw", SPATIAL)
def test_spatial_mean_any_channels(n, c, hw, rocm_device):
    """fp32 sums of up to 3190 bf16 values rounded once: one bf16 ulp, 2^-8,
    and 1e-5 near zero."""
    import oracle as ref
    torch.manual_seed(n + c + hw)
    x = torch.randn(n, hw, c).to(torch.bfloat16)
    want = ref.spatial_mean_nhwc(x.view(n, hw, 1, c).permute(0, 3, 1, 2)).reshape(n, c)
    for shift in (0, 1):
        xd = place(x, rocm_device, shift)
        out = Guarded((n, c), torch.bfloat16, rocm_device, shift)
        need = lib().hipo_spatial_mean_workspace_bytes(n, hw, c)
        ws = torch.empty(max(need, 1), dtype=torch.uint8, device=rocm_device)
        ok(lib().hipo_spatial_mean_nhwc_bf16(xd.data_ptr(), out.t.data_ptr(), n, hw, c,
                                             ws.data_ptr() if need else None, need, None))
        torch.cuda.synchronize()
        out.check(f"[{n}, {c}, {hw}]")
        close(out.t, want, 2 ** -8, 1e-5, f"[{n}, {c}, {hw}] shift {shift}")


# (n, c, h, w, pad): one group, a channel more and less, several groups with a
# remainder, one row a workgroup and many, more groups than threads.
BN_NHWC = [(2, 7, 3, 3, 1), (2, 8, 3, 3, 0), (3, 9, 5, 4, 1), (2, 28, 20, 21, 1), (4, 103, 9, 9, 0),
           (2, 664, 6, 5, 1), (3, 2049, 3, 2, 1), (40, 33, 31, 30, 0), (1, 8200, 2, 2, 0),
           # 39 and 40 rows: one thread per channel, and workgroups
           (3, 237, 13, 1, 1), (4, 237, 5, 2, 1), (4, 9, 2, 5, 0),
           # 127 128-row slices, halved, and 128 of them, a partial last one
           (1, 40, 127, 128, 0), (1, 40, 128, 128, 1), (1, 9, 131, 127, 0)]


@pytest.mark.parametrize("n,c,h,w,pad", BN_NHWC)
def test_batchnorm_nhwc_any_channels(n, c, h, w, pad, rocm_device):
    """Statistics 1e-5.  y = act(t), t rounded to bf16, where kernel and oracle
    may land on neighbouring values: one ulp, up to 2^-7 of t; 1e-5 near zero,
    where the affine form cancels.  SiLU carries that ulp at a relative slope
    of at most 1.1 for t > 0 and rounds again, two ulps, 2^-6; for t < 0 the
    ulp moves it by at most 2^-7 max |t silu'(t)| = 2^-7 * 0.25 = 2e-3."""
    import oracle as ref
    torch.manual_seed(n * c + h)
    x = torch.randn(n, h, w, c).to(torch.bfloat16)
    gamma, beta, rm, rv = torch.randn(c), torch.randn(c), torch.randn(c), torch.rand(c) + 0.5
    for shift, act, code in ((0, "silu", 2), (1, "relu", 1), (1, "none", 0)):
        sm, sr, yw, rmw, rvw = ref.batchnorm_nhwc_act_pad(
            x.permute(0, 3, 1, 2), gamma, beta, rm, rv, momentum=0.1, eps=1e-3, var_scale=1.25,
            act=act, pad_bottom=pad, pad_right=pad)
        xd = place(x, rocm_device, shift)
        out = Guarded((n, h + pad, w + pad, c), torch.bfloat16, rocm_device, shift)
        side = [t.to(rocm_device) for t in (gamma, beta, rm, rv)]
        mean, rstd = (Guarded((c,), torch.float32, rocm_device) for _ in range(2))
        need = lib().hipo_batchnorm_nhwc_workspace_bytes(n, h, w, c)
        ws = Guarded((need // 4,), torch.float32, rocm_device)
        ok(lib().hipo_batchnorm_nhwc_act_pad_bf16(
            xd.data_ptr(), *(t.data_ptr() for t in side), mean.t.data_ptr(), rstd.t.data_ptr(),
            out.t.data_ptr(), n, h, w, c, pad, pad, 0.1, 1e-3, 1.25, code, ws.t.data_ptr(), need,
            None))
        torch.cuda.synchronize()
        what = f"[{n}, {c}, {h}, {w}] {act}"
        for o in (out, mean, rstd, ws):
            o.check(what)
        rtol, atol = (2 ** -6, 2e-3) if act == "silu" else (2 ** -7, 1e-5)
        close(out.t, yw.permute(0, 2, 3, 1), rtol, atol, what)
        for a, b in ((mean.t, sm), (rstd.t, sr), (side[2], rmw), (side[3], rvw)):
            close(a, b.reshape(-1), 1e-5, 1e-5, what)


# (n, c, h, w): the small-plane kernel with a channel block moved back and with
# misaligned x (the one-launch kernel needs C % 4 == 0), planes over 128 values
# at the ends of the lane counts (256, 512, 1024) and in several chunks,
# fewer channels than a block, fewer values than a group, a partial slice.
BN_NCHW = [(5, 9, 5, 5), (6, 15, 8, 16), (3, 125, 7, 7), (2, 3, 3, 2), (2, 3, 3, 3), (5, 6, 3, 43),
           (4, 8, 16, 16), (9, 11, 1, 257), (7, 10, 16, 32), (3, 5, 1, 513), (2, 9, 28, 28),
           (1, 2, 32, 32), (6, 7, 25, 41), (2, 3, 60, 61), (300, 2, 12, 12),
           # a lane per channel, several slices of images and a partial last
           # one, and the neighbours of its lines
           (9, 3, 2, 2), (301, 7, 1, 7), (47, 1001, 1, 3), (49, 1001, 1, 3), (255, 1025, 1, 1),
           (33, 2049, 2, 3), (33, 2047, 2, 3)]


@pytest.mark.parametrize("n,c,h,w", BN_NCHW)
def test_batchnorm_nchw_mean_any_plane(n, c, h, w, rocm_device):
    """Statistics 1e-5.  A mean of up to 3660 activations, each of which may
    sit one bf16 ulp off the oracle's at a rounding boundary (rarely, and up
    or down alike), rounded once more: 2^-7, and 1e-4 near zero.  Planes of a
    few values average no such flip away: one value t of the plane whose bf16
    pre-activation falls to the other side moves its activation (slopes up to
    1.1) by 1.1 ulps of t, at most 1.1 * 2^-7 |t|, and that rounds once more:
    2^-6 max |t| over the plane, divided by its size, on top."""
    import oracle as ref
    torch.manual_seed(n + c + h)
    x = torch.randn(n, c, h, w).to(torch.bfloat16)
    gamma, beta, rm, rv = torch.randn(c), torch.randn(c), torch.randn(c), torch.rand(c) + 0.5
    for shift, act, code in ((0, "silu", 2), (1, "relu", 1), (1, "none", 0)):
        sm, sr, yw, rmw, rvw = ref.batchnorm_nchw_act_mean(
            x, gamma, beta, rm, rv, momentum=0.1, eps=1e-5, var_scale=1.25, act=act)
        xd = place(x, rocm_device, shift)
        out = Guarded((n, c), torch.bfloat16, rocm_device, shift)
        side = [Guarded((c,), torch.float32, rocm_device) for _ in range(4)]
        for g, t in zip(side, (gamma, beta, rm, rv)):
            g.t.copy_(t)
        mean, rstd = (Guarded((c,), torch.float32, rocm_device) for _ in range(2))
        need = lib().hipo_batchnorm_nchw_mean_workspace_bytes(n, c, h * w)
        ws = Guarded((need // 4,), torch.float32, rocm_device)
        ok(lib().hipo_batchnorm_nchw_act_mean_bf16(
            xd.data_ptr(), *(g.t.data_ptr() for g in side), mean.t.data_ptr(), rstd.t.data_ptr(),
            out.t.data_ptr(), n, c, h * w, 0.1, 1e-5, 1.25, code, ws.t.data_ptr(), need, None))
        torch.cuda.synchronize()
        what = f"[{n}, {c}, {h}, {w}] {act}"
        for o in (out, mean, rstd, ws, *side):
            o.check(what)
        if h * w < 9:
            v = [1, c, 1, 1]
            t = (x.float() - sm.view(v)) * sr.view(v) * gamma.view(v) + beta.view(v)
            tol = 2 ** -7 * yw.float().abs() + 1e-4 + 2 ** -6 * t.abs().amax((2, 3)) / (h * w)
            assert bool(((out.t.float().cpu() - yw.float()).abs() <= tol).all()), what
        else:
            close(out.t, yw, 2 ** -7, 1e-4, what)
        for a, b in ((mean.t, sm), (rstd.t, sr), (side[2].t, rmw), (side[3].t, rvw)):
            close(a, b.reshape(-1), 1e-5, 1e-5, what)


# Rows per block rounded up from 65..96 and 33..63 rows, the last block and
# the last pass of a block partly filled; 97 rows, as planned.
@pytest.mark.parametrize("rows,cols", [(25000, 3072), (5001, 6144), (1025, 4104), (24901, 4096)])
def test_gelu_bwd_row_blocks(rows, cols, rocm_device):
    """y is one fp32 product of the same operands, the column sum one rounding
    of an fp64 sum that is exact here: bit for bit."""
    import hip_oracles
    import oracle as ref
    torch.manual_seed(rows)
    g, x = (torch.randn(rows, cols).to(torch.bfloat16) for _ in range(2))
    yw, cw = ref.gelu_erf_bwd_colsum(g, x)
    y, colsum = hip_oracles.gelu_erf_bwd_colsum(g.to(rocm_device), x.to(rocm_device))
    assert torch.equal(y.cpu(), yw)
    assert torch.equal(colsum.cpu(), cw)


# Below a vector, one vector, one value more and less, several waves per row
# and more than one sweep; a row stride past the row.
@pytest.mark.parametrize("cols", [1, 3, 4, 5, 7, 8, 9, 255, 257, 333, 511, 513, 777, 1025, 4097,
                                  8707, 33000])
def test_row_mean_any_row_length(cols, rocm_device):
    """fp32 sums in another order: 1e-5.  bf16: one rounding of an fp32 mean,
    one ulp, 2^-7, and 1e-5 near zero."""
    import oracle as ref
    torch.manual_seed(cols)
    rows = 11
    x = torch.randn(rows, cols + 3)
    xb = torch.randn(rows, cols).to(torch.bfloat16)
    for shift in (0, 1):
        xd = place(x, rocm_device, shift)
        out = Guarded((rows,), torch.float32, rocm_device)
        ok(lib().hipo_row_mean_f32(xd.data_ptr(), out.t.data_ptr(), rows, cols, cols + 3, None))
        torch.cuda.synchronize()
        out.check(f"f32 {cols}")
        close(out.t, ref.row_mean(x[:, :cols].contiguous()), 1e-5, 1e-5, f"f32 {cols}")
        xd = place(xb, rocm_device, shift)
        for relu in (0, 1):
            out = Guarded((rows,), torch.bfloat16, rocm_device)
            ok(lib().hipo_row_mean_bf16(xd.data_ptr(), out.t.data_ptr(), rows, cols, relu, None))
            torch.cuda.synchronize()
            out.check(f"bf16 {cols}")
            close(out.t, ref.row_mean_bf16(xb, relu=bool(relu)), 2 ** -7, 1e-5, f"bf16 {cols}")


# (rows, cols, elements off alignment): both sides of the lines where short
# rows off alignment leave the wave per row for the short-row kernel (24000
# rows, up to 256 values), and whole longer ones the rows kernel for one wave
# each, by waves a row and how full they are; partial last workgroups.
@pytest.mark.parametrize("rows,cols,shift", [
    (23999, 256, 1), (24000, 256, 1), (24013, 9, 3), (24001, 257, 1), (70, 400, 1), (9, 512, 5),
    (2559, 520, 0), (2560, 520, 0), (2563, 1032, 0), (4095, 2056, 0), (4097, 2056, 0),
    (4099, 4104, 0), (4097, 8200, 0), (2561, 1024, 0),
    (2048, 520, 0), (2049, 1000, 0), (16384, 1000, 0), (16385, 1000, 0), (16385, 520, 0),
    (32768, 704, 0), (32769, 704, 0),
    (3, 1096, 0), (3, 1112, 0), (1536, 1448, 0), (1537, 1448, 0), (4095, 1736, 0), (4096, 1736, 0),
    (2815, 2056, 0), (2816, 2056, 0), (3583, 3080, 0), (3584, 3080, 0), (4099, 3592, 0),
    (2048, 3001, 0), (2049, 3001, 0), (2047, 4095, 3), (2053, 4095, 0), (999, 1500, 1)])
def test_row_mean_bf16_many_rows(rows, cols, shift, rocm_device):
    """One rounding of an fp32 mean: one ulp, 2^-7, and 1e-5 near zero."""
    import oracle as ref
    torch.manual_seed(rows + cols)
    x = torch.randn(rows, cols).to(torch.bfloat16)
    xd = place(x, rocm_device, shift)
    for relu in (0, 1):
        out = Guarded((rows,), torch.bfloat16, rocm_device)
        ok(lib().hipo_row_mean_bf16(xd.data_ptr(), out.t.data_ptr(), rows, cols, relu, None))
        torch.cuda.synchronize()
        out.check(f"[{rows}, {cols}]")
        close(out.t, ref.row_mean_bf16(x, relu=bool(relu)), 2 ** -7, 1e-5, f"[{rows}, {cols}]")


# fp32 rows off the vector path: both sides of the lines between one wave and
# several waves per row.
@pytest.mark.parametrize("rows,cols", [(1023, 1025), (1024, 1025), (1024, 1535), (1025, 1537),
                                       (2047, 1537), (2048, 1537), (1000, 1023)])
def test_row_mean_f32_ragged_lines(rows, cols, rocm_device):
    """fp32 sums in another order: 1e-5."""
    import oracle as ref
    torch.manual_seed(rows + cols)
    x = torch.randn(rows, cols)
    xd = place(x, rocm_device, 1)
    out = Guarded((rows,), torch.float32, rocm_device)
    ok(lib().hipo_row_mean_f32(xd.data_ptr(), out.t.data_ptr(), rows, cols, cols, None))
    torch.cuda.synchronize()
    out.check(f"[{rows}, {cols}]")
    close(out.t, ref.row_mean(x), 1e-5, 1e-5, f"[{rows}, {cols}]")
