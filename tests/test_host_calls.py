"""The native operator calls' checks, which need no GPU: each wrong call raises the exception type that the operators document,
before anything is launched."""
import pytest
import torch


def _t(*shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype)


@pytest.mark.parametrize("call,error", [
    (lambda o: o.gemm_ksteps("NN", [], []), ValueError),
    (lambda o: o.gemm_ksteps("NN", [_t(2, 3)], []), ValueError),
    (lambda o: o.gemm_ksteps("XX", [_t(2, 3)], [_t(3, 2)]), ValueError),
    (lambda o: o.gemm_ksteps("NN", [_t(2, 3)], [_t(3, 2)]), RuntimeError),
    # step operands and addends may be one stacked tensor, as any sequence: it gets as far as the device check
    (lambda o: o.gemm_ksteps("NN", _t(2, 2, 3), _t(2, 3, 2)), RuntimeError),
    (lambda o: o.gemm_ksteps("NN", [_t(2, 3)], [_t(3, 2)], addends=_t(1, 2, 2)), RuntimeError),
    (lambda o: o.gemm_ksteps("NN", [3], [_t(3, 2)]), TypeError),
    (lambda o: o.gemm_ksteps("NN", [_t(2, 3)], [_t(3, 2)], _t(2), "swish"), KeyError),
    (lambda o: o.colsum(_t(2, 3)), RuntimeError),
    (lambda o: o.act_bwd_colsum("relu", _t(2, 3), _t(2, 3)), RuntimeError),
    (lambda o: o.ln_forward_fused(_t(2, 3), 1e-5), RuntimeError),
    (lambda o: o.ln_backward_fused(_t(2, 3), _t(2, 3), _t(2, 2)), RuntimeError),
])
def test_wrong_calls_raise(call, error):
    from cubework_amd import ops

    with pytest.raises(error):
        call(ops)
