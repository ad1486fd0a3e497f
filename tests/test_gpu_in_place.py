"""Calls whose output is one of the inputs, through the C entry points: the
results are those of the same call with a separate output, bit for bit."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def lib():
    import hip_oracles
    return hip_oracles.load_library()


def ok(rc):
    assert rc == 0, lib().hipo_last_error()


def same(got, want, what):
    torch.cuda.synchronize()
    assert torch.equal(got.cpu(), want.cpu()), what


# Value by value; register-held planes of whole vectors and not, 256 and 1024
# threads; the single-pass kernel; split-K with whole vectors (x off alignment)
# and with planes whose last vector is moved back.
@pytest.mark.parametrize("n,c,hw,shift", [
    (3, 5, 7, 0), (26, 9, 49, 0), (335, 3, 49, 0), (128, 40, 196, 0), (16, 8, 3136, 0),
    (16, 8, 3136, 1), (60, 2, 1023, 0), (1, 4, 50001, 0), (700, 2, 70, 0), (400, 4, 131, 1)])
def test_batchnorm_train_in_place(n, c, hw, shift, rocm_device):
    torch.manual_seed(n + c + hw)
    x = torch.randn(n * c * hw + shift, device=rocm_device) * 2 + 0.5
    gamma, beta = torch.randn(c, device=rocm_device), torch.randn(c, device=rocm_device)
    outs = []
    for in_place in (False, True):
        xd = x.clone()[shift:]
        y = xd if in_place else torch.empty_like(x)[shift:]
        rm, rv = torch.zeros(c, device=rocm_device), torch.ones(c, device=rocm_device)
        mean, invstd = torch.empty_like(rm), torch.empty_like(rm)
        need = lib().hipo_batchnorm_workspace_bytes(n, c, hw)
        ws = torch.zeros(need, dtype=torch.uint8, device=rocm_device)
        ok(lib().hipo_batchnorm_train_fwd_f32(
            xd.data_ptr(), gamma.data_ptr(), beta.data_ptr(), rm.data_ptr(), rv.data_ptr(),
            y.data_ptr(), mean.data_ptr(), invstd.data_ptr(), n, c, hw, 0.1, 1e-5, 1,
            ws.data_ptr(), need, None))
        torch.cuda.synchronize()
        outs.append((y.clone(), mean, invstd, rm, rv))
    for name, a, b in zip(("y", "mean", "invstd", "running_mean", "running_var"), *outs):
        same(b, a, f"[{n}, {c}, {hw}] {name}")


@pytest.mark.parametrize("c", [5, 8, 72, 103, 1001])
@pytest.mark.parametrize("shift", [0, 1])
def test_batchnorm_nhwc_in_place(c, shift, rocm_device):
    """No padding: out has x's shape."""
    n, h, w = 6, 20, 31
    torch.manual_seed(c)
    x = (torch.randn(n * h * w * c + shift, device=rocm_device) * 2 + 0.5).to(torch.bfloat16)
    gamma, beta = torch.randn(c, device=rocm_device), torch.randn(c, device=rocm_device)
    outs = []
    for in_place in (False, True):
        xd = x.clone()[shift:]
        y = xd if in_place else torch.empty_like(x)[shift:]
        rm, rv = torch.zeros(c, device=rocm_device), torch.ones(c, device=rocm_device)
        mean, rstd = torch.empty_like(rm), torch.empty_like(rm)
        need = lib().hipo_batchnorm_nhwc_workspace_bytes(n, h, w, c)
        ws = torch.empty(need, dtype=torch.uint8, device=rocm_device)
        ok(lib().hipo_batchnorm_nhwc_act_pad_bf16(
            xd.data_ptr(), gamma.data_ptr(), beta.data_ptr(), rm.data_ptr(), rv.data_ptr(),
            mean.data_ptr(), rstd.data_ptr(), y.data_ptr(), n, h, w, c, 0, 0, 0.1, 1e-5, 1.0, 1,
            ws.data_ptr(), need, None))
        torch.cuda.synchronize()
        outs.append((y.clone(), mean, rstd, rm, rv))
    for name, a, b in zip(("out", "mean", "rstd", "running_mean", "running_var"), *outs):
        same(b, a, f"C {c} shift {shift} {name}")


# Value by value; one row to a part of a wave, with one and two groups a lane;
# several waves a row with the last group moved back over a wave's first
# values (cols % 512 in 1..7), over its own wave's, and not at all; rows longer
# than the registers hold.
@pytest.mark.parametrize("cols", [5, 64, 197, 513, 769, 1543, 2049, 2055, 4096, 4097, 8195, 33001])
def test_norms_in_place(cols, rocm_device):
    """h over x and over the residual, y over x: as with separate outputs."""
    rows, bf = 37, torch.bfloat16
    torch.manual_seed(cols)
    x, r = (torch.randn(rows, cols, device=rocm_device).to(bf) for _ in range(2))
    gamma, beta = (torch.randn(cols, device=rocm_device).to(bf) for _ in range(2))

    def run(op, where):
        xd, rd = x.clone(), r.clone()
        spare = [torch.empty_like(x) for _ in range(2)]
        h, y = {"apart": spare, "h=x": (xd, spare[0]), "h=res": (rd, spare[0]),
                "y=x": (spare[0], xd)}[where]
        mean, rstd = (torch.empty(rows, device=rocm_device) for _ in range(2))
        if op == "layernorm":
            ok(lib().hipo_residual_layernorm_bf16(
                xd.data_ptr(), rd.data_ptr(), gamma.data_ptr(), beta.data_ptr(), h.data_ptr(),
                y.data_ptr(), mean.data_ptr(), rstd.data_ptr(), rows, cols, 1e-5, None))
        else:
            ok(lib().hipo_rmsnorm_ex_bf16(
                xd.data_ptr(), rd.data_ptr(), gamma.data_ptr(), h.data_ptr(), y.data_ptr(),
                rstd.data_ptr(), rows, cols, 1e-5, 0.5, 1, None))
        torch.cuda.synchronize()
        return h, y, rstd

    for op in ("layernorm", "rmsnorm"):
        want = run(op, "apart")
        for where in ("h=x", "h=res", "y=x"):
            for name, a, b in zip(("h", "y", "rstd"), run(op, where), want):
                same(a, b, f"{op} cols {cols} {where} {name}")
