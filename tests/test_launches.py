"""Kernel and launch shape of calls, recorded without a GPU (launches.py)."""

import pytest

from launches import (LdsLimit, Launch, a8_gemm, a8_tiled, built, kernels, moe, padded, pointers, q4_gemm, q8_prefill,
                      record)
import test_gpu_prefill_tilings as tilings

DEFAULT_LDS = 64 * 1024


def q8(entry, tokens, n, k, dtype, slots=False):
    x, codes, scales, out, workspace = pointers(5)
    return entry, [x, codes, scales, out, tokens, n, k, padded(k), dtype, *((workspace, 1 << 30) if slots else ()), None]


# Calls whose kernels need more LDS than a launch may have by default: the prefill GEMMs' forms, the decode forms that
# stage long activations, the canonical-order route and the few-token MoE.
CALLS = {
    "q8 prefill, cooperative": q8_prefill(2048, 34816, 5120),
    "q8 prefill, split": q8_prefill(200, 4096, 5120),
    "q8 prefill, long rows": q8_prefill(64, 128, (1 << 22) + 8),
    "a8 prefill, cooperative": a8_gemm(2048, 34816, 5120, 1),
    "a8 prefill, split": a8_gemm(200, 4096, 5120, 2),
    "a8 decode, staged": a8_tiled(16, 4096, 5120, 2),
    "q4 prefill, cooperative": q4_gemm(512, 7168, 5120),
    "q4 prefill, split": q4_gemm(64, 7168, 5120),
    "q4 prefill, wide": q4_gemm(2048, 34816, 5120),
    "q8 decode": q8("venturi_q8_tiled_run", 1, 4096, 40960, 0, slots=True),
    "q8 exact": q8("venturi_q8_head_run", 2, 7168, 17408, 0),
    "q8 exact, slab": q8("venturi_q8_head_run", 64, 7168, 17408, 1),
    "moe, few tokens": moe(16, 2048, 128, 8, 768),
}


@pytest.mark.parametrize("name", CALLS)
def test_lds_limit_is_raised_on_every_device(name):
    """A process that drives two devices: the attribute belongs to a device, so each kernel's limit is raised on the
    one that it is launched on, before the launch."""
    entry, args = CALLS[name]
    limits, large = {}, 0
    for events in record([(device, entry, args) for device in (0, 1, 0, 70)]):
        for e in events:
            if isinstance(e, LdsLimit):
                limits[e.kernel, e.device] = e.bytes
            elif e.shared > DEFAULT_LDS:
                large += 1
                assert limits.get((e.kernel, e.device), 0) >= e.shared, e
        assert any(isinstance(e, Launch) for e in events)
    assert large, "the call no longer needs the limit raised"


def rows_of_a_pass(k):
    """Activation rows that the few-token MoE form stages: 67584 bytes of rows of whole 256-column chunks and 8 halves."""
    return min(16, 67584 // (2 * ((padded(k) + 255) // 256 * 256 + 8)))


@pytest.mark.parametrize("hidden,experts,top_k,inter", [(2048, 128, 8, 768), (4096, 64, 4, 1408), (2880, 32, 4, 2880),
                                                        (1024, 32, 16, 512), (776, 8, 1, 4104), (8, 1024, 2, 8)])
def test_moe_few_token_form_takes_at_most_two_passes(hidden, experts, top_k, inter):
    """However the routing shares experts among the tokens, no expert takes more than two passes of the form's rows;
    past that, gate/up and down each run the grouped form."""
    gate_up, down = 2 * rows_of_a_pass(hidden), 2 * rows_of_a_pass(inter)
    tokens = sorted({1, 8, 16, gate_up, gate_up + 1, down, down + 1, 33, 64})
    for t, events in zip(tokens, record([(0, *moe(t, hidden, experts, top_k, inter)) for t in tokens])):
        forms = [e.kernel.split("<")[0] for e in events if isinstance(e, Launch)]
        assert forms[:2] == ["q4_few" if t <= gate_up else "q4_grouped", "q4_few" if t <= down else "q4_grouped"], (t, forms)


def reached(calls):
    return {kernel for launched in kernels([(0, *call) for call in calls]) for kernel in launched}


def test_q8_prefill_tests_reach_every_tiling():
    calls = [q8_prefill(*shape) for shape in tilings.Q8_SHAPES]
    calls += [q8_prefill(t, n, k, scales_offset=2 * shift) for t, n, k, shift in tilings.Q8_OUTSIDE_SPLIT]
    assert built("q8_prefill") | built("q8_prefill_split") == reached(calls)


def test_q8_prefill_of_short_rows_shares_the_cus():
    """Where K is a few hundred columns and the grid fills the chip, the prologue and the output are the time: such calls
    take a tiling without a K split, of which two or four workgroups share a CU."""
    shapes = [(100, 34816, 136), (128, 34816, 256), (1024, 16384, 136), (8192, 16384, 256), (2048, 34816, 64)]
    for shape, launched in zip(shapes, kernels([(0, *q8_prefill(*shape)) for shape in shapes])):
        assert launched[0].startswith(("q8_prefill<1, 4, 1, 8, 2,", "q8_prefill<1, 4, 1, 4, 2,")), (shape, launched)


def test_a8_prefill_tests_reach_every_tiling():
    calls = [a8_gemm(*shape) for shape in tilings.A8_SHAPES]
    calls += [a8_gemm(*shape, scales_offset=2) for shape in tilings.A8_TWO_BYTE_SCALES]
    assert built("a8_prefill") | built("a8_prefill_split") == reached(calls)


def test_a8_prefill_tests_reach_two_passes_with_partial_and_whole_stages():
    """Both passes' partial stages come first, then the whole ones of each: on every cooperative tiling that can have a
    partial stage (K split over two or four waves, one 32-column group per wave and stage)."""
    want = {name for name in built("a8_prefill") if int(name.split(",")[2]) > 1 and "unsigned int" in name}
    seen = set()
    for shape, launched in zip(tilings.A8_SHAPES, kernels([(0, *a8_gemm(*shape)) for shape in tilings.A8_SHAPES])):
        if shape[3] == 2 and launched[0] in want:
            groups, waves = (shape[2] + 31) // 32, int(launched[0].split(",")[2])
            if groups > waves and groups % waves:
                seen.add(launched[0])
    assert seen == want


def test_a8_prefill_of_short_rows_shares_the_cus():
    shapes = [(100, 34816, 136, 1), (128, 34816, 256, 1), (1024, 16384, 136, 1), (8192, 16384, 256, 1), (2048, 34816, 64, 1)]
    for shape, launched in zip(shapes, kernels([(0, *a8_gemm(*shape)) for shape in shapes])):
        assert launched[0].startswith(("a8_prefill<1, 4, 1, 8, 2,", "a8_prefill<1, 4, 1, 4, 2,")), (shape, launched)


def test_q4_prefill_tests_reach_every_tiling():
    names = built("q4_prefill") | built("q4_prefill_split") | {k for k in built("row_prefill") if k.startswith("row_prefill<0,")}
    assert names == reached([q4_gemm(*shape) for shape in tilings.Q4_SHAPES])


def test_q4_prefill_of_short_rows_and_of_rows_past_the_lane_offsets_takes_the_tiles_that_win_there():
    """Short rows on a full grid, and, below 256 tokens, rows past the 32-bit lane offsets: 128 x 128 tiles with the whole
    K in one wave, two workgroups to a CU. Those rows in longer prompts: the 256-token tiles."""
    short = [(100, 34816, 1024), (128, 151936, 1024), (200, 65536, 512), (100, 250000, 136), (33, 151936, 64),
             (100, 64, (1 << 22) + 8)]
    for shape, launched in zip(short, kernels([(0, *q4_gemm(*shape)) for shape in short])):
        assert launched == ["row_prefill<0, 4, 2, 2, 4, 2, 1>"], (shape, launched)
    assert kernels([(0, *q4_gemm(256, 64, (1 << 22) + 8))])[0][0].startswith("row_prefill<0, 4, 2, 4, ")


def a8_tiled_linear(tokens, n, k, passes):
    x, workspace, codes, scales, out, slots = pointers(6)
    return "venturi_q8_a8_tiled_linear_run", [x, workspace, 1 << 35, codes, scales, out, tokens, n, k, padded(k), passes,
                                              slots, 1 << 30, None]


def test_a8_tiled_tests_reach_every_form_without_an_lds_copy():
    assert built("a8_tiled_split") | built("a8_tiled_decode") <= reached([a8_tiled(*shape) for shape in tilings.A8_TILED_SHAPES])


def test_a8_projection_keeps_the_one_launch_order():
    """Quantizing and projecting in one launch or in two gives the same bytes where the workgroup shape is the same:
    wherever the one-launch form serves run(), project() takes the staged form, in its shape unless it splits K (long rows
    of 257-384 row blocks)."""
    shapes = [(t, n, k, p) for t in (1, 3, 8, 9, 16) for n in (16, 4096, 4097, 8176, 8192, 8208, 12288, 12300, 17000, 34816)
              for k in (8, 128, 1000, 2048, 4096, 6144, 9000, 14336, 17408, 30000) for p in (1, 2)]
    one = record([(0, *a8_tiled_linear(*shape)) for shape in shapes])
    two = record([(0, *a8_tiled(*shape)) for shape in shapes])
    served = 0
    for shape, run, project in zip(shapes, one, two):
        run, project = ([e for e in events if isinstance(e, Launch)] for events in (run, project))
        assert len(project) == 1
        if len(run) == 1:  # no separate quantizer
            served += 1
            fused, staged = (e.kernel.split("<")[1].replace(" ", "").split(",") for e in (run[0], project[0]))
            assert run[0].kernel.startswith("a8_tiled_lds<") and project[0].kernel.startswith("a8_tiled_lds<"), shape
            if not staged[5].startswith("2"):  # workgroups that share a row block's K
                assert fused[:4] == staged[:4], shape
                assert (run[0].blocks, run[0].threads) == (project[0].blocks, project[0].threads), shape
    assert served > 100
