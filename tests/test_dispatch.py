"""Which kernels the entry points launch, without a GPU (dispatch.py)."""
import pytest

from dispatch import kernel, launched


def names(step):
    return [kernel(n) for n, _, _ in step]


# The batched step's q|k|v sums in the order of the calls one by one, whatever
# the width of q: the same kernels, in one launch or with q in one of its own.
@pytest.mark.parametrize("fp8", [True, False])
def test_multi_step_qkv_takes_the_kernels_of_separate_calls(fp8):
    shapes = [(hq, rows) for hq in (32, 36, 40, 64, 72) for rows in (1, 3, 4, 16)]
    steps = []
    for hq, rows in shapes:
        steps += [("multi_step", 4096, 12800, hq, hq // 4, rows, fp8), ("gemm", fp8, rows, hq * 128, 4096),
                  ("gemm", fp8, rows, hq // 4 * 128, 4096)]
    got = launched(steps)
    for i, (hq, rows) in enumerate(shapes):
        q, kv = names(got[3 * i + 1]), names(got[3 * i + 2])
        step = [n for n, _, _ in got[3 * i]]
        append = next(j for j, n in enumerate(step) if "rope_append" in n)
        qkv = [k for k in map(kernel, step[:append]) if k[0].startswith("gemm_")]
        assert kv[0][0] == "gemm_skinny_kernel"  # k and v, or all three, in one launch
        assert qkv == (q if q == kv else q + kv), (hq, rows)


# A key-split attention whose scratch pool cannot be made runs unsplit, and the
# next call tries again; under capture it never splits.
def test_prefill_attn_scratch_pool_failure_lasts_one_call():
    step = ("prefill_attn", 17, 50000)
    got = [names(s) for s in launched([("fail_pool_create", 1), step, step, ("capturing", 1), step,
                                       ("capturing", 0), step])]
    split = ["attn_prefill_kernel", "attn_prefill_combine_kernel"]
    assert [[n for n, _ in s] for s in got if s] == [split[:1], split, split[:1], split]
