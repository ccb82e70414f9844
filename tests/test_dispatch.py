"""Which kernels the entry points launch, without a GPU (dispatch.py)."""
import pytest

import gemm_tile_shapes as shapes
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


# Where the tile kernel is the slower one (a K too short for its pipeline, or a
# last round of tiles nearly empty; by the factor given), the call takes the
# kernel that is faster; layer shapes keep the tile.
FASTER = [  # FP8 (None: SwiGLU), rows, columns, K, kernel
    (True, 128, 1024, 256, "gemm_fp8_kernel"),      # 2.4
    (True, 700, 4096, 512, "gemm_fp8_kernel"),      # 1.5
    (True, 1000, 2560, 1024, "gemm_fp8_kernel"),    # 1.3
    (True, 96, 7168, 1280, "gemm_fp8_kernel"),      # 1.1
    (True, 32, 25600, 2048, "gemm_fp8_kernel"),     # 1.15
    (True, 300, 4096, 1792, "gemm_fp8_kernel"),     # 1.07
    (True, 4, 8192, 1280, "gemm_skinny_kernel"),    # 1.7
    (True, 16, 8192, 512, "gemm_skinny_kernel"),    # 2.1
    (True, 1, 25600, 2048, "gemm_skinny_kernel"),   # 1.2
    (True, 4, 6144, 4096, "gemm_skinny_kernel"),    # 1.1 (weights from memory)
    (False, 128, 1024, 128, "gemm_bf16w_kernel"),   # 2.1
    (False, 700, 2560, 256, "gemm_bf16w_kernel"),   # 1.4
    (False, 300, 1024, 640, "gemm_bf16w_kernel"),   # 1.1
    (False, 4, 8192, 1152, "gemm_skinny_kernel"),   # 2.9
    (False, 8, 6144, 512, "gemm_skinny_kernel"),    # 1.2
    (None, 300, 2048, 256, "gemm_fp8_kernel"),      # 2.1
    (None, 300, 8192, 2560, "gemm_fp8_kernel"),     # 1.1
    (None, 300, 9600, 2560, "gemm_fp8_kernel"),     # 1.1
    (None, 8, 8192, 4096, "gemm_skinny_kernel"),    # 1.2
    # weights from memory
    (None, 8, 16384, 4096, "gemm_skinny_kernel"),   # 1.13
    (None, 8, 12288, 4096, "gemm_skinny_kernel"),   # 1.08
    (None, 1, 20480, 5120, "gemm_skinny_kernel"),   # 1.4
    (None, 16, 12288, 8192, "gemm_skinny_kernel"),  # 1.2
    (None, 8, 5120, 2048, "gemm_skinny_kernel"),    # 1.09
    (None, 8, 6144, 8192, "gemm_skinny_kernel"),    # 1.08
    (True, 4, 16384, 4096, "gemm_skinny_kernel"),   # 1.09
    (True, 8, 16384, 8192, "gemm_skinny_kernel"),   # 1.15
    (True, 4, 6144, 8192, "gemm_skinny_kernel"),    # 1.06
    (False, 2, 9216, 6144, "gemm_skinny_kernel"),   # 1.09
    (None, 16, 16384, 6144, "gemm_tile_kernel"), (None, 8, 12800, 4096, "gemm_tile_kernel"),
    (None, 16, 6144, 4096, "gemm_tile_kernel"), (True, 4, 12800, 4096, "gemm_tile_kernel"),
    (True, 12, 16384, 7168, "gemm_tile_kernel"), (False, 2, 12800, 6144, "gemm_tile_kernel"),
    (True, 2561, 6144, 4096, "gemm_fp8_kernel"),    # 1.3
    (None, 832, 12800, 4096, "gemm_fp8_kernel"),    # 1.08
    (True, 512, 4096, 12800, "gemm_tile_kernel"), (True, 8192, 6144, 4096, "gemm_tile_kernel"),
    (True, 16, 6144, 4096, "gemm_tile_kernel"), (False, 1000, 6144, 4096, "gemm_tile_kernel"),
    (False, 17, 4096, 4096, "gemm_tile_kernel"), (False, 16, 100352, 4096, "gemm_tile_kernel"),
    (None, 8192, 12800, 4096, "gemm_tile_kernel"), (None, 1, 12800, 4096, "gemm_tile_kernel"),
    (True, 8, 4096, 12800, "gemm_skinny_kernel"), (False, 16, 4096, 4096, "gemm_skinny_kernel"),
]


def test_gemm_takes_the_faster_kernel():
    got = launched([("gemm_swiglu", m, n, k) if fp8 is None else ("gemm", fp8, m, n, k)
                    for fp8, m, n, k, _ in FASTER])
    assert [(*f[:4], names(s)[0][0]) for f, s in zip(FASTER, got)] == FASTER


def prefill_plan(step):
    """(positions per workgroup, key splits) of a prefill attention's launches."""
    _, (_, _, blocks, _, ksp) = kernel(step[0][0])
    assert len(step) == (1 if step[0][1][2] == 1 else 2)
    return 16 if ksp == 2 else 32 * blocks, step[0][1][2]


# Behind a window most workgroups are as long as the longest: their mean length
# is not half of it (us with the plan of a chunk that grows throughout / this one).
@pytest.mark.parametrize("rows,base,window,hk,plan", [
    (1300, 0, 1024, 8, (32, 1)),    # 50.0 / 42.1
    (2000, 0, 1024, 8, (64, 1)),    # 69.6 / 57.9
    (900, 0, 256, 8, (32, 1)),      # 24.1 / 17.2 (split before)
    (4096, 0, 1024, 2, (32, 1)),    # 52.3 / 38.4
    (2000, 0, 0, 8, (32, 1)), (2000, 0, 4096, 8, (32, 1))])
def test_prefill_plan_behind_a_window(rows, base, window, hk, plan):
    assert prefill_plan(launched([("prefill_attn", rows, base, window, hk)])[0]) == plan


# Key splits only where the call gains by them: its scratch and its two launches
# take the host 20 us, and the partials their share of the memory's time (us
# split / whole).
@pytest.mark.parametrize("rows,base,hk,plan", [
    (1, 700, 8, (16, 1)),       # 33.1 / 19.5
    (64, 700, 8, (16, 1)),      # 26.8 / 20.3
    (128, 500, 1, (16, 1)),     # 25.3 / 17.7
    (1000, 1000, 8, (32, 1)),   # 79.2 / 63
    (2000, 500, 4, (16, 1)),    # 84.5 / 71.9
    (8, 3000, 8, (16, 10)), (17, 50000, 8, (64, 61)), (500, 20000, 8, (64, 4))])
def test_prefill_plan_splits_keys_where_they_gain(rows, base, hk, plan):
    assert prefill_plan(launched([("prefill_attn", rows, base, 0, hk)])[0]) == plan


# The shapes of the tile GEMM's test run the configurations that they name, as
# many tiles per workgroup as they say; the K padded copies that they are
# compared with, and the short K, run the other kernels.
def test_gemm_tile_shapes_run_the_named_tiles():
    todo = ([(True, *s) for s in shapes.FP8] + [(False, *s) for s in shapes.BF16] +
            [(None, *s) for s in shapes.SWIGLU])

    def step(fp8, m, n, k):
        return ("gemm_swiglu", m, n, k) if fp8 is None else ("gemm", fp8, m, n, k)

    for (fp8, m, n, k, fragments, turns), got in zip(todo, launched([step(*t[:4]) for t in todo])):
        (name, args), grid = kernel(got[0][0]), got[0][1][0]
        assert (name, tuple(args[2:4])) == ("gemm_tile_kernel", fragments), (fp8, m, n, k)
        count = shapes.tiles(m, n, fragments, fp8 is None)
        assert grid == min(count, 256) and -(-count // grid) == turns, (fp8, m, n, k, count)
    along_n = [t for t, o in zip(todo, launched([step(*t[:4]) for t in todo], "orders")) if o[0][3]]
    assert along_n == [(True, *s) for s in shapes.FP8[-3:]] + [(False, *s) for s in shapes.BF16[-3:]] + [
        (None, *s) for s in shapes.SWIGLU[-2:]]
    other = [step(t[0], t[1], t[2], t[3] + (32 if t[0] is False else 128)) for t in todo]
    other += [step(f, *s) for f, l in ((True, shapes.FP8_OTHER), (False, shapes.BF16_OTHER),
                                       (None, shapes.SWIGLU_OTHER)) for s in l]
    for s, got in zip(other, launched(other)):
        assert kernel(got[0][0])[0] != "gemm_tile_kernel", s


# Where an XCD would run every 8th tile of a column with an odd number of them,
# and so read all of A, tiles are numbered along N (us plain / along N).
@pytest.mark.parametrize("fp8,m,n,k,order", [
    (True, 6337, 1024, 4096, (25, 8, True, True)),      # 40 / 29
    (True, 7936, 3072, 4096, (31, 24, True, True)),     # 129 / 91
    (False, 7936, 4096, 12800, (31, 16, True, True)),   # 602 / 578
    (True, 8192, 4096, 12800, (32, 16, False, False)),  # an eighth of the M tiles per XCD
    (True, 6337, 25600, 4096, (25, 100, False, False)),  # along N as much of W as of A before
    (True, 512, 4096, 12800, (4, 64, True, False))])
def test_gemm_tile_order(fp8, m, n, k, order):
    assert [tuple(o) for o in launched([("gemm", fp8, m, n, k)], "orders")[0]] == [order]


# The bf16 general kernel's two residual forms: loaded at a tile's start, or
# after its K loop where tiles outnumber the resident workgroups.
def test_prefill_gemm_residual_forms():
    got = launched([("gemm", False, 200, 256, 480, 2), ("gemm", False, 2100, 4096, 128, 2)])
    assert [names(s) for s in got] == [[("gemm_bf16w_kernel", [2, 0])], [("gemm_bf16w_kernel", [2, 1])]]
