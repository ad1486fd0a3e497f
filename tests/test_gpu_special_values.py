"""NaN and infinite inputs of the reductions: in their own row or channel the
results are NaN (a mean may be the infinity where a merge keeps it), and every
other row and channel is what the C oracle gives."""
import pytest
import torch

pytestmark = pytest.mark.gpu

NAN, INF = float("nan"), float("inf")


def with_specials(x):
    """Channels 1 to 4 of [n, c, ...]: a NaN, +inf, -inf, both infinities."""
    n = x.shape[0]
    x = x.clone()
    x[n // 2, 1].view(-1)[0] = NAN
    x[0, 2].view(-1)[-1] = INF
    x[n - 1, 3].view(-1)[0] = -INF
    x[0, 4].view(-1)[0] = INF
    x[n - 1, 4].view(-1)[-1] = -INF
    return x


def check_channels(got, want, outs, want_outs, rtol, atol, what):
    """got / want: (mean, rstd, running mean, running var) per channel; outs:
    the outputs with the channel first."""
    got = [t.float().cpu().reshape(-1) for t in got]
    want = [t.float().reshape(-1) for t in want]
    bad = slice(1, 5)
    good = [c for c in range(got[0].numel()) if not 1 <= c <= 4]
    mean, rstd, rm, rv = got
    assert not bool(torch.isfinite(mean[bad]).any()), what
    assert not bool(torch.isfinite(rm[bad]).any()), what
    assert bool(mean[1].isnan()) and bool(mean[4].isnan()), what
    assert bool(rstd[bad].isnan().all()) and bool(rv[bad].isnan().all()), what
    assert bool(outs[bad].isnan().all()), what
    for a, b in zip(got, want):
        assert torch.allclose(a[good], b[good], rtol=1e-5, atol=1e-5), what
    assert torch.allclose(outs[good], want_outs[good], rtol=rtol, atol=atol), what


def params(c):
    return torch.randn(c), torch.randn(c), torch.zeros(c), torch.ones(c)


# Value by value; planes with the last vector moved back and whole ones, 256 and
# 1024 threads; split-K; the single-pass kernel.
@pytest.mark.parametrize("n,c,hw", [(3, 5, 7), (26, 9, 49), (400, 9, 49), (4, 8, 196), (128, 40, 196),
                                    (1100, 5, 49), (16, 8, 3136)])
def test_batchnorm_train(n, c, hw, rocm_device):
    import hip_oracles
    import oracle as ref
    torch.manual_seed(n + c)
    x = with_specials(torch.randn(n, c, 1, hw))
    gm, bt, rm, rv = params(c)
    want = ref.batchnorm_train(x, gm, bt, rm, rv, momentum=0.1, eps=1e-5, relu=True)
    d = [t.to(rocm_device) for t in (x, gm, bt, rm, rv)]
    y, mean, rstd = hip_oracles.batchnorm_train(*d, momentum=0.1, eps=1e-5, relu=True)
    check_channels((mean, rstd, d[3], d[4]), want[1:], y.cpu().transpose(0, 1),
                   want[0].transpose(0, 1), 1e-5, 1e-5, f"[{n}, {c}, {hw}]")


# 16-byte groups, the last one moved back, and one thread per channel.
@pytest.mark.parametrize("c", [5, 8, 9, 103])
@pytest.mark.parametrize("act", ["relu", "silu", None])
def test_batchnorm_nhwc(c, act, rocm_device):
    """Outputs within one bf16 ulp of a pre-activation that may fall to its
    neighbour: 2^-6 of it covers both roundings, 1e-2 where it cancels."""
    import hip_oracles
    import oracle as ref
    torch.manual_seed(c)
    x = with_specials(torch.randn(6, c, 13, 11)).to(torch.bfloat16)
    x = x.contiguous(memory_format=torch.channels_last)
    gm, bt, rm, rv = params(c)
    kw = dict(momentum=0.1, eps=1e-5, var_scale=1.0, act=act, pad_bottom=0, pad_right=0)
    sm, sr, yw, rmw, rvw = ref.batchnorm_nhwc_act_pad(x, gm, bt, rm, rv, **kw)
    d = [t.to(rocm_device) for t in (x, gm, bt, rm, rv)]
    mean, rstd, y = hip_oracles.batchnorm_nhwc_act_pad(*d, **kw)
    check_channels((mean, rstd, d[3], d[4]), (sm, sr, rmw, rvw), y.float().cpu().transpose(0, 1),
                   yw.float().transpose(0, 1), 2 ** -6, 1e-2, f"C {c} {act}")


# A wave per channel (32 and 64 lanes a plane, several chunks), a wave per 8
# channels (all of them its own, and the last ones moved back), a channel in
# registers, a lane per channel.
@pytest.mark.parametrize("n,c,h,w", [(5, 6, 10, 20), (6, 7, 25, 21), (5, 7, 40, 41), (300, 8, 7, 7),
                                     (300, 9, 7, 7), (8, 8, 7, 7), (9, 5, 2, 2)])
def test_batchnorm_nchw_mean(n, c, h, w, rocm_device):
    """A mean of activations, each at most one bf16 ulp off: 2^-6, and 1e-2
    where a small plane's values cancel."""
    import hip_oracles
    import oracle as ref
    torch.manual_seed(n + c)
    x = with_specials(torch.randn(n, c, h, w)).to(torch.bfloat16)
    gm, bt, rm, rv = params(c)
    kw = dict(momentum=0.1, eps=1e-5, var_scale=1.0, act="relu")
    sm, sr, yw, rmw, rvw = ref.batchnorm_nchw_act_mean(x, gm, bt, rm, rv, **kw)
    d = [t.to(rocm_device) for t in (x, gm, bt, rm, rv)]
    mean, rstd, out = hip_oracles.batchnorm_nchw_act_mean(*d, **kw)
    check_channels((mean, rstd, d[3], d[4]), (sm, sr, rmw, rvw), out.float().cpu().T,
                   yw.float().reshape(n, c).T, 2 ** -6, 1e-2, f"[{n}, {c}, {h}, {w}]")


# Finite values whose squares overflow: the variance is infinite, rstd 0, and the
# outputs are act(beta).  Every route as above but the kernels that sum about one
# of the channel's values, and shapes whose huge value is the only one of a
# thread's first merge.
@pytest.mark.parametrize("n,c,hw", [(3, 5, 7), (26, 9, 49), (400, 9, 49), (4, 8, 196), (21, 5, 961),
                                    (128, 40, 196), (3, 40, 8836), (1100, 5, 49), (2, 5, 9999),
                                    (7, 5, 8649)])
@pytest.mark.parametrize("where", [0, 1, 4097, -1])
def test_batchnorm_train_overflowing_squares(n, c, hw, where, rocm_device):
    import hip_oracles
    torch.manual_seed(n + c)
    x = torch.randn(n, c, 1, hw)
    flat = x.transpose(0, 1).reshape(c, -1)
    at = where % flat.shape[1]
    x[at // hw, 1, 0, at % hw] = 3e38
    x[at // hw, 2, 0, at % hw] = -3e38
    gm, bt, rm, rv = params(c)
    d = [t.to(rocm_device) for t in (x, gm, bt, rm, rv)]
    y, mean, rstd = hip_oracles.batchnorm_train(*d, momentum=0.1, eps=1e-5, relu=False)
    for ch, v in ((1, 3e38), (2, -3e38)):
        assert float(mean[ch]) == pytest.approx(v / (n * hw), rel=1e-5)
        assert float(rstd[ch]) == 0 and float(d[4][ch]) == INF
        assert bool((y[:, ch] == d[2][ch]).all())
    assert bool(torch.isfinite(y).all())


@pytest.mark.parametrize("n,c,h,w", [(5, 6, 10, 20), (6, 7, 25, 21), (5, 7, 40, 41), (5, 36, 85, 85),
                                     (300, 8, 7, 7), (300, 9, 7, 7)])
@pytest.mark.parametrize("where", [0, 1, -1])
def test_batchnorm_nchw_mean_overflowing_squares(n, c, h, w, where, rocm_device):
    import hip_oracles
    torch.manual_seed(n + c)
    x = torch.randn(n, c, h, w).to(torch.bfloat16)
    at = where % (n * h * w)
    x[at // (h * w), 1].view(-1)[at % (h * w)] = 3e38
    gm, bt, rm, rv = params(c)
    d = [t.to(rocm_device) for t in (x, gm, bt, rm, rv)]
    mean, rstd, out = hip_oracles.batchnorm_nchw_act_mean(*d, momentum=0.1, eps=1e-5, var_scale=1.0,
                                                          act="relu")
    big = float(torch.tensor(3e38).to(torch.bfloat16))
    assert float(mean.view(-1)[1]) == pytest.approx(big / (n * h * w), rel=1e-5)
    assert float(rstd.view(-1)[1]) == 0 and float(d[4][1]) == INF
    want = torch.relu(bt[1]).to(torch.bfloat16).float()
    assert torch.allclose(out[:, 1].float().cpu(), want.expand(n), rtol=2 ** -7, atol=1e-6)


# Short rows aligned and not, a wave per row, several waves per row in one sweep
# and in several, whole and ragged; fp32: the vector kernel, its ragged form,
# single values.
@pytest.mark.parametrize("rows,cols,shift", [(40, 49, 0), (40, 49, 1), (24003, 50, 1), (40, 300, 1),
                                             (2600, 520, 0), (40, 777, 0), (40, 1024, 0),
                                             (40, 9001, 0), (40, 16400, 0)])
def test_row_means(rows, cols, shift, rocm_device):
    import hip_oracles
    import oracle as ref
    torch.manual_seed(rows + cols)
    x = torch.randn(rows, cols)
    x[3, cols - 1] = NAN
    x[5, 0] = INF
    x[7, cols // 2] = -INF
    x[9, 0], x[9, cols - 1] = INF, -INF
    xb = x.to(torch.bfloat16)
    buf = torch.zeros(x.numel() + shift, dtype=torch.bfloat16, device=rocm_device)
    xd = buf[shift:].view(rows, cols)
    xd.copy_(xb)
    for relu in (False, True):
        got = hip_oracles.row_mean_bf16(xd, relu=relu).float().cpu()
        want = ref.row_mean_bf16(xb, relu=relu).float()
        assert torch.allclose(got, want, rtol=2 ** -7, atol=1e-5, equal_nan=True), relu
    got = hip_oracles.row_mean(x.to(rocm_device)).cpu()
    assert torch.allclose(got, ref.row_mean(x), rtol=1e-5, atol=1e-5, equal_nan=True)
