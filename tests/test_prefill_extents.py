"""prefill()'s host checks: a tensor smaller than its step describes is refused before its
pointer goes down, also where a size does not fit the description's 32-bit fields (stand-in
tensors; no GPU needed)."""
import pytest
import torch

from apertura_amd.prefill import PrefillStep, prefill


class _Tensor:
    """What prefill() reads of a contiguous bf16 GPU tensor of n elements."""
    dtype, is_cuda, device = torch.bfloat16, True, "cuda"

    def __init__(self, n):
        self._n = n

    def untyped_storage(self):
        return self

    def nbytes(self):
        return 2 * self._n

    def storage_offset(self):
        return 0

    def data_ptr(self):
        return 0


@pytest.mark.parametrize("field,value,name", [
    ("seq_q", 2 ** 32 + 8, "q"), ("seq_k", 2 ** 32 + 8, "k"), ("num_q_heads", 2 ** 32 + 4, "q"),
    ("num_kv_heads", 2 ** 32 + 2, "k"), ("seq_q", 9, "q"), ("seq_k", 9, "k"),
])
def test_sizes_past_the_tensors_are_refused(field, value, name):
    """The tensors hold 4 / 2 heads of 8 rows; the step's sizes wrap to exactly those in 32 bits,
    or are one row more."""
    D = 128
    sizes = dict(num_q_heads=4, num_kv_heads=2, seq_q=8, seq_k=8)
    sizes[field] = value
    step = PrefillStep(head_dim=D, q_head_stride=8 * D, q_row_stride=D, kv_head_stride=8 * D,
                       out_row_stride=4 * D, out_head_stride=D, **sizes)
    with pytest.raises(ValueError, match=f"{name} is smaller"):
        prefill(step, _Tensor(4 * 8 * D), _Tensor(2 * 8 * D), _Tensor(2 * 8 * D), _Tensor(8 * 4 * D))
