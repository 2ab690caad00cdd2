"""What the fused TimeMix pieces refuse: parameters of another length or device than the
kernels read, which they take by pointer."""
import pytest
import torch

from theseus import fused

C = 256


@pytest.mark.parametrize("p", [torch.ones(8), torch.ones(1, 1, 8), torch.ones(8, dtype=torch.bfloat16),
                               torch.ones(2 * C), torch.ones(8, requires_grad=True)])
def test_vec_refuses_another_length(p):
    with pytest.raises(RuntimeError, match="invalid for input of size"):
        fused._vec(p, C)


def test_vec_hands_out_a_row():
    row = torch.ones(3, C)[1]
    assert fused._vec(row, C) is row
    assert fused._vec(torch.ones(1, 1, C), C).shape == (C,)


@pytest.mark.parametrize("bad", [torch.ones(8), torch.ones(1, 1, C - 1, dtype=torch.bfloat16), torch.ones(C, 2),
                                 torch.ones(C, device="meta")])
@pytest.mark.parametrize("at", [1, 2])
def test_pack_params_refuses_another_length_or_device(bad, at):
    ps = [torch.ones(C), torch.ones(1, 1, C, dtype=torch.bfloat16)]
    ps.insert(at, bad)
    with pytest.raises(RuntimeError, match="pack_params: expected parameters of 256 elements on cpu"):
        fused.pack_params(ps, C)


@pytest.mark.parametrize("coefs", [torch.ones(5, C), torch.ones(6, C - 1), torch.ones(6 * C),
                                   [torch.ones(C)] * 5, torch.ones(6, 8, dtype=torch.bfloat16),
                                   torch.ones(6, 2 * C)[:, ::2][:5]])
def test_coefficients_of_another_shape(coefs):
    with pytest.raises(RuntimeError, match="six coefficients|invalid for input of size"):
        fused._coef_matrix(coefs, C)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float64])
def test_coefficient_matrix_of_any_type_and_stride(dtype):
    rows = torch.rand(6, C).to(dtype)
    for m in (rows, rows.t().contiguous().t(), rows.unsqueeze(1), [r.reshape(1, 1, C) for r in rows]):
        cf = fused._coef_matrix(m, C)
        assert cf.dtype == torch.float32 and cf.is_contiguous() and torch.equal(cf, rows.float())


def test_kernels_inputs_on_the_device_of_x():
    x, shift = torch.zeros(1, 2, C, dtype=torch.bfloat16, device="meta"), torch.zeros(1, C, device="meta")
    with pytest.raises(RuntimeError, match="coefficients on cpu, x on meta"):
        fused._shift_lerp_fwd(x, shift, torch.ones(6, C))


@pytest.mark.parametrize("shape", [(1, 2, C - 64), (1, 1, C), (2, 2, C)])
def test_decay_input_like_k(shape):
    k = torch.zeros(1, 2, C, dtype=torch.bfloat16)
    v = torch.ones(C)
    with pytest.raises(RuntimeError, match="decay input like k"):
        fused.kk_kmod_w(k, k, v, v, v, torch.zeros(shape, dtype=torch.bfloat16), v, 64, torch.bfloat16)


def test_direct_calls():
    """A call goes past its autograd function only when nothing that the function answers is on."""
    x, p, seen = torch.ones(2), torch.ones(2, requires_grad=True), []
    assert fused._direct(x, x) and not fused._direct(x, p)
    with torch.no_grad():
        assert fused._direct(x, p)
        torch.jit.trace(lambda t: (seen.append(fused._direct(t)), t * 2)[1], x, check_trace=False)
        torch.func.vmap(lambda t: (seen.append(fused._direct(t)), t)[1])(x)
        with torch.autograd.forward_ad.dual_level():
            seen.append(fused._direct(x))
    assert seen == [False] * len(seen) and len(seen) >= 3
