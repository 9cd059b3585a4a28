"""The cached plans of the kernel spectra, built on the CPU here: every stream and thread reads them, so on a GPU they come from
copies that wait, and nothing of them is computed on the device."""
import numpy as np
import torch
from torch.utils._python_dispatch import TorchDispatchMode


class _Operations(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func.overloadpacket._qualified_op_name)
        return func(*args, **(kwargs or {}))


def test_plans_are_computed_on_the_host():
    import s2cnn_amd
    from s2cnn_amd import s2_real, so3_real, wigner
    cpu = torch.device("cpu")
    with _Operations() as ops:
        idx, E, Et, dtab = so3_real._setup_so3_rft_plan.__wrapped__(5, s2cnn_amd.so3_near_identity_grid(), cpu)
        F, Ft = s2_real._setup_s2_rft_plan.__wrapped__(5, s2cnn_amd.s2_near_identity_grid(), cpu)
    assert set(ops.names) <= {"aten::lift_fresh", "aten::detach", "aten::detach_", "aten::_to_copy"}, ops.names      # uploads
    assert all(t.is_contiguous() for t in (idx, E, Et, dtab, F, Ft))
    assert idx.dtype == torch.int32 and torch.equal(Et, E.transpose(1, 2)) and torch.equal(Ft, F.t())
    want = wigner.so3_rft_plan(5, s2cnn_amd.so3_near_identity_grid())
    for got, w in zip((idx, E, dtab), want):
        assert np.array_equal(got.numpy(), w.astype(got.numpy().dtype))
    assert torch.equal(F, s2_real._setup_s2_ft_real.__wrapped__(5, s2cnn_amd.s2_near_identity_grid(), cpu))
