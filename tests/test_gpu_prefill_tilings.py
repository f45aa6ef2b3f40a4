"""Every tiling of the prefill GEMMs at ragged edges, against FP64 on the GPU.

The dispatch chooses a tiling per shape by a time model; the shapes below reach
each candidate (largest tiles down to the smallest) with partial token tiles,
partial row tiles, K that is not whole stages or chunks, and the fallbacks of
operands that the split form does not take. Bound per output (fp32 sums of
exact products, one fp16 rounding): 0.5 ulp16(exact) + 2^-19 sum_k |x_k w_k|.
"""

import pytest
import torch

from helpers import guarded_out, random_q8
from venturi_amd import Q8RowSplitWeight, prepare_q8_dp4a
from venturi_amd.weights import Q4RowSplitWeight

pytestmark = pytest.mark.gpu


def ulp16(v):
    return torch.exp2(torch.floor(torch.log2(v.abs().clamp_min(2.0**-14))) - 10)


def assert_bound(got, x, w):
    """got [T, N] fp16 against x [T, K] @ w[N, K]^T in FP64 (all on the GPU)."""
    exact, magnitude = x @ w.T, x.abs() @ w.abs().T
    error = (got.double() - exact).abs()
    assert bool((error <= 0.5 * ulp16(exact) + 2.0**-19 * magnitude).all())


def values(codes, scales, k):
    n, padded = codes.shape
    group = padded // scales.shape[1]
    return (codes.view(n, -1, group).double() * scales.double().unsqueeze(-1)).view(n, padded)[:, :k]


def activations(tokens, k, device, seed):
    return torch.randn(tokens, k, generator=torch.Generator().manual_seed(seed)).half().to(device)


# (tokens, rows, columns): 256 x 128, 128 x 128 and 64 x 128 tiles (the latter two with and without a K split), 80 x 64,
# 64 x 64, 48 x 64, 32 x 64 and 32 x 32 tiles; test_launches.py checks that every tiling is reached.
Q8_SHAPES = [(257, 14003, 136), (513, 7001, 136), (1025, 7001, 136), (300, 10001, 264), (97, 14003, 136),
             (33, 20001, 520), (129, 7001, 1032), (81, 14003, 1000), (160, 4100, 1032), (113, 7001, 1032),
             (79, 14003, 136), (300, 4100, 136), (33, 14003, 136), (65, 10001, 200), (33, 257, 136), (97, 31, 3976),
             (700, 7001, 520), (2047, 2049, 520), (257, 10001, 520), (300, 20001, 264), (1025, 14003, 72), (129, 7001, 2056),
             (33, 10001, 264), (33, 4100, 136), (47, 4100, 264)]


@pytest.mark.parametrize("tokens,n,k", Q8_SHAPES)
def test_q8_tilings(backend, device, tokens, n, k):
    print(f"case q8 prefill tiling tokens={tokens} n={n} k={k}", flush=True)
    codes, scales = (t.to(device) for t in random_q8(n, k, 31 + n + tokens))
    x = activations(tokens, k, device, tokens)
    plan = backend.upload_linear(Q8RowSplitWeight(codes, scales, k), dtype=torch.float16, device=device).prepare(
        tokens=tokens, route="mfma")
    guard, out = guarded_out(tokens, n, torch.float16, device)
    plan.run(x, out=out)
    assert guard[0] == 47 and guard[-1] == 47
    assert_bound(out, x.double(), values(codes, scales, k))
    aligned = torch.empty(tokens, n, dtype=torch.float16, device=device)
    plan.run(x, out=aligned)  # 16-byte stores where n allows them: the same bits
    assert torch.equal(aligned, out)


Q8_OUTSIDE_SPLIT = [(40, 70, 8, 0), (70, 33, 40, 0), (33, 64, 120, 0), (40, 300, 1000, 1), (130, 64, 4096, 1),
                    (33, 3, (1 << 22) + 8, 0)]


@pytest.mark.parametrize("tokens,n,k,shift", Q8_OUTSIDE_SPLIT)
def test_q8_operands_outside_the_split_form(backend, device, tokens, n, k, shift):
    # Fewer than 128 columns, scales aligned to 2 bytes only, rows past the 32-bit lane offsets.
    print(f"case q8 prefill fallback tokens={tokens} n={n} k={k} shift={shift}", flush=True)
    codes, scales = (t.to(device) for t in random_q8(n, k, 5 + n + tokens))
    padded = codes.shape[1]
    moved = torch.empty(scales.numel() + shift, dtype=torch.float16, device=device)[shift:].view(scales.shape)
    moved.copy_(scales)
    x = activations(tokens, k, device, 9)
    guard, out = guarded_out(tokens, n, torch.float16, device)
    lib = backend._native
    lib.check(lib.venturi_q8_prefill_run(x.data_ptr(), codes.data_ptr(), moved.data_ptr(), out.data_ptr(), tokens, n, k,
                                         padded, 0, torch.cuda.current_stream(device).cuda_stream))
    assert guard[0] == 47 and guard[-1] == 47
    assert_bound(out, x.double(), values(codes, scales, k))


def integers(shape, low, high, device, seed):
    gen = torch.Generator().manual_seed(seed)
    return torch.randint(low, high + 1, shape, dtype=torch.int8, generator=gen).to(device)


def powers(shape, device, seed):
    """Group scales 1/2, 1 and 2."""
    return torch.exp2(integers(shape, -1, 1, device, seed).float())


def assert_exact(got, x, w):
    """Sums of small integers times powers of two: every association gives the same fp16 value."""
    exact = x @ w.T
    assert bool((exact.half().double() == exact).all())
    assert torch.equal(got.double(), exact)


@pytest.mark.parametrize("tokens,n,k", Q8_SHAPES)
def test_q8_tilings_place_every_product(backend, device, tokens, n, k):
    print(f"case q8 prefill exact sums tokens={tokens} n={n} k={k}", flush=True)
    p = (k + 127) // 128 * 128
    codes, scales = integers((n, p), -1, 1, device, n + k), powers((n, p // 32), device, n).half()
    x = integers((tokens, k), -1, 1, device, tokens)
    plan = backend.upload_linear(Q8RowSplitWeight(codes, scales, k), dtype=torch.float16, device=device).prepare(
        tokens=tokens, route="mfma")
    out = torch.empty(tokens, n, dtype=torch.float16, device=device)
    plan.run(x.half(), out=out)
    assert_exact(out, x.double(), values(codes, scales, k))


def represented(workspace, tokens, k, passes):
    """FP64 values of the quantized activations in an A8 workspace."""
    groups = (k + 31) // 32
    count = tokens * groups
    codes = workspace[: count * 32 * passes].view(torch.int8).view(passes, tokens, groups, 32).double()
    scales = workspace[count * 32 * passes :].view(torch.float32).view(passes, tokens, groups, 1).double()
    return (codes * scales).sum(0).view(tokens, groups * 32)[:, :k]


# 256 x 128, 128 x 128 and 64 x 128 (with and without a K split), 32 x 128, 64 x 64 (eight and four K waves), 48 x 64 (four
# and eight), 32 x 64 and 32 x 32 tiles (test_launches.py checks that every tiling is reached); whole and partial stages
# and chunks (K % 128), K below one chunk, one and two passes, two passes that each have a partial and whole stages.
A8_SHAPES = [(257, 14003, 136, 1), (513, 7001, 128, 2), (129, 14003, 136, 1), (257, 7001, 300, 1), (65, 10001, 136, 1),
             (33, 14003, 256, 1), (97, 7001, 520, 1), (160, 4100, 520, 2), (97, 14003, 4104, 1), (200, 7001, 2056, 2),
             (65, 10001, 1032, 1), (79, 10001, 519, 2), (33, 14003, 136, 2), (97, 4100, 520, 1), (33, 4100, 1032, 1),
             (47, 4100, 520, 2), (65, 257, 136, 1), (33, 257, 129, 2), (81, 31, 3971, 1), (65, 70, 31, 2), (40, 33, 127, 1),
             (700, 7001, 520, 1), (700, 7001, 264, 2), (257, 7001, 264, 1), (257, 7001, 136, 2), (200, 7001, 264, 1),
             (200, 7001, 136, 2), (700, 10001, 136, 1), (700, 7001, 136, 2), (129, 7001, 72, 1), (513, 7001, 130, 2),
             (97, 4100, 136, 1), (160, 4100, 2056, 2), (47, 4100, 1032, 2), (97, 4100, 2056, 1),
             (33, 3, (1 << 22) + 8, 1)]  # the last: rows past the 32-bit lane offsets


@pytest.mark.parametrize("tokens,n,k,passes", A8_SHAPES)
def test_a8_tilings(backend, device, tokens, n, k, passes):
    print(f"case a8 prefill tiling tokens={tokens} n={n} k={k} passes={passes}", flush=True)
    codes, scales = (t.to(device) for t in random_q8(n, k, 57 + n + tokens))
    x = activations(tokens, k, device, tokens + 1)
    x[3, min(k - 1, 40)] = float("inf")  # that group: zero codes, NaN scale; the token's outputs are NaN
    plan = prepare_q8_dp4a(backend.upload_linear(Q8RowSplitWeight(codes, scales, k), dtype=torch.float16, device=device),
                           tokens=tokens, residual_compensation=passes == 2, route="mfma")
    workspace = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=device)
    guard, out = guarded_out(tokens, n, torch.float16, device)
    plan.run(x, out=out, workspace=workspace)
    assert guard[0] == 47 and guard[-1] == 47
    keep = torch.arange(tokens, device=device) != 3
    assert bool(torch.isnan(out[3]).all())
    assert_bound(out[keep], represented(workspace, tokens, k, passes)[keep], values(codes, scales, k))
    aligned = torch.empty(tokens, n, dtype=torch.float16, device=device)
    plan.project(out=aligned, workspace=workspace)  # 16-byte stores where n allows them: the same bits
    assert torch.equal(aligned[keep], out[keep])


@pytest.mark.parametrize("tokens,n,k,passes", A8_SHAPES[:-1])  # (sums of four million products exceed fp16's integers)
def test_a8_tilings_place_every_product(backend, device, tokens, n, k, passes):
    print(f"case a8 prefill exact sums tokens={tokens} n={n} k={k} passes={passes}", flush=True)
    p, groups = (k + 127) // 128 * 128, (k + 31) // 32
    codes, scales = integers((n, p), -1, 1, device, n + k), powers((n, p // 32), device, n).half()
    acts = integers((passes, tokens, groups * 32), -1, 1, device, tokens)
    acts[:, :, k:] = 0
    ascales = powers((passes, tokens, groups), device, tokens + 1)
    workspace = torch.cat((acts.flatten().view(torch.uint8), ascales.flatten().view(torch.uint8)))
    lib, stream = backend._native, torch.cuda.current_stream(device).cuda_stream
    out = torch.empty(tokens, n, dtype=torch.float16, device=device)
    lib.check(lib.venturi_q8_a8_gemm_run(workspace.data_ptr(), workspace.numel(), codes.data_ptr(), scales.data_ptr(),
                                         out.data_ptr(), tokens, n, k, p, passes, stream))
    assert_exact(out, represented(workspace, tokens, k, passes), values(codes, scales, k))


A8_TWO_BYTE_SCALES = [(130, 300, 1000, 1), (70, 64, 4096, 2), (70, 64, 4104, 2)]


@pytest.mark.parametrize("tokens,n,k,passes", A8_TWO_BYTE_SCALES)
def test_a8_scales_aligned_to_two_bytes(backend, device, tokens, n, k, passes):
    print(f"case a8 prefill fallback tokens={tokens} n={n} k={k}", flush=True)
    codes, scales = (t.to(device) for t in random_q8(n, k, 5 + n + tokens))
    moved = torch.empty(scales.numel() + 1, dtype=torch.float16, device=device)[1:].view(scales.shape)
    moved.copy_(scales)
    x = activations(tokens, k, device, 9)
    lib, stream = backend._native, torch.cuda.current_stream(device).cuda_stream
    workspace = torch.empty(lib.venturi_q8_dp4a_bytes(tokens, k, passes), dtype=torch.uint8, device=device)
    lib.check(lib.venturi_q8_dp4a_quantize(x.data_ptr(), workspace.data_ptr(), workspace.numel(), tokens, k, passes, stream))
    guard, out = guarded_out(tokens, n, torch.float16, device)
    lib.check(lib.venturi_q8_a8_gemm_run(workspace.data_ptr(), workspace.numel(), codes.data_ptr(), moved.data_ptr(),
                                         out.data_ptr(), tokens, n, k, codes.shape[1], passes, stream))
    assert guard[0] == 47 and guard[-1] == 47
    assert_bound(out, represented(workspace, tokens, k, passes), values(codes, scales, k))


# 128 x 128 (with and without a K split), 64 x 128, 64 x 64 (eight and four K waves), 48 x 64 (four and eight), 32 x 64 and
# 32 x 32 tiles, the wide tiles of the large grids (test_launches.py checks that every tiling is reached), K below one
# chunk, and the first token count of the route.
Q4_SHAPES = [(300, 10001, 264), (129, 7001, 520), (97, 7001, 1032), (113, 14003, 2056), (65, 14003, 520),
             (97, 4100, 1032), (47, 4100, 1032), (65, 257, 136), (32, 33, 3976), (33, 70, 40), (40, 300, 120),
             (1025, 14003, 264), (513, 14003, 136), (1025, 10001, 136), (700, 7001, 2056), (65, 10001, 136), (200, 2049, 1000), (513, 1000, 2056),
             (65, 20001, 136), (200, 10001, 2056), (513, 7001, 4104), (2047, 4100, 136), (513, 14003, 2056),
             (2047, 7001, 136), (33, 3, (1 << 22) + 8)]  # the last: rows past the 32-bit lane offsets


@pytest.mark.parametrize("tokens,n,k", Q4_SHAPES)
def test_q4_tilings(backend, device, tokens, n, k):
    print(f"case q4 prefill tiling tokens={tokens} n={n} k={k}", flush=True)
    gen = torch.Generator().manual_seed(3 + n + tokens)
    padded = (k + 127) // 128 * 128
    codes = torch.randint(0, 256, (n, padded // 2), dtype=torch.uint8, generator=gen).to(device)
    scales = (torch.rand(n, padded // 64, generator=gen) * 0.05).half().to(device)
    low, high = codes & 15, codes >> 4
    signed = torch.stack((low, high), -1).view(n, padded).to(torch.int8)
    signed = torch.where(signed > 7, signed - 16, signed)
    x = activations(tokens, k, device, tokens + 2)
    plan = backend.upload_linear(Q4RowSplitWeight(codes, scales, k), dtype=torch.float16, device=device).prepare(
        tokens=tokens, route="mfma")
    guard, out = guarded_out(tokens, n, torch.float16, device)
    plan.run(x, out=out)
    assert guard[0] == 47 and guard[-1] == 47
    weights = values(signed, scales, k).half().double()  # the contract's fp16(q * scale)
    assert_bound(out, x.double(), weights)
    aligned = torch.empty(tokens, n, dtype=torch.float16, device=device)
    plan.run(x, out=aligned)  # 16-byte stores where n allows them: the same bits
    assert torch.equal(aligned, out)


@pytest.mark.parametrize("tokens,n,k", Q4_SHAPES[:-1])  # (sums of four million products exceed fp16's integers)
def test_q4_tilings_place_every_product(backend, device, tokens, n, k):
    print(f"case q4 prefill exact sums tokens={tokens} n={n} k={k}", flush=True)
    p = (k + 127) // 128 * 128
    signed, scales = integers((n, p), -1, 1, device, n + k), powers((n, p // 64), device, n).half()
    nibbles = signed.view(torch.uint8) & 15
    x = integers((tokens, k), -1, 1, device, tokens)
    plan = backend.upload_linear(Q4RowSplitWeight(nibbles[:, 0::2] | (nibbles[:, 1::2] << 4), scales, k),
                                 dtype=torch.float16, device=device).prepare(tokens=tokens, route="mfma")
    out = torch.empty(tokens, n, dtype=torch.float16, device=device)
    plan.run(x.half(), out=out)
    assert_exact(out, x.double(), values(signed, scales, k))


# The split form over the tiled planes: one, two and three row blocks per workgroup, four K waves past 768 blocks (past
# 1024 at up to 16 tokens); K below one chunk, partial chunks, odd group counts; up to 16 tokens where the activations
# exceed the decode LDS, and there the register form at 513-768 row blocks (test_launches.py checks what is reached).
A8_TILED_SHAPES = [(17, 4096, 1000, 1), (32, 70, 31, 2), (31, 33, 97, 1), (20, 500, 4000, 2), (24, 5120, 519, 1),
                   (32, 7167, 2056, 2), (17, 11702, 391, 2), (32, 12300, 136, 1), (25, 20001, 264, 2),
                   (16, 300, 16392, 2), (12, 5000, 17408, 2), (16, 13000, 5120, 2), (9, 17000, 12296, 1),
                   (16, 17000, 5128, 2), (13, 16999, 12296, 2), (12, 300, 30000, 2), (12, 9001, 15240, 2), (16, 9001, 30001, 1)]


@pytest.mark.parametrize("tokens,n,k,passes", A8_TILED_SHAPES)
def test_a8_tiled_split(backend, device, tokens, n, k, passes):
    print(f"case a8 tiled split tokens={tokens} n={n} k={k} passes={passes}", flush=True)
    codes, scales = (t.to(device) for t in random_q8(n, k, 91 + n + tokens))
    x = activations(tokens, k, device, tokens + 4)
    x[1, min(k - 1, 40)] = float("nan")  # that group: zero codes, NaN scale; the token's outputs are NaN
    plan = prepare_q8_dp4a(backend.upload_linear(Q8RowSplitWeight(codes, scales, k), dtype=torch.float16, device=device),
                           tokens=tokens, residual_compensation=passes == 2)
    assert plan.kernel == "tiled"
    workspace = torch.empty(plan.workspace_bytes, dtype=torch.uint8, device=device)
    guard, out = guarded_out(tokens, n, torch.float16, device)
    plan.run(x, out=out, workspace=workspace)
    assert guard[0] == 47 and guard[-1] == 47
    keep = torch.arange(tokens, device=device) != 1
    assert bool(torch.isnan(out[1]).all())
    assert_bound(out[keep], represented(workspace, tokens, k, passes)[keep], values(codes, scales, k))
    again = torch.empty(tokens, n, dtype=torch.float16, device=device)
    plan.project(out=again, workspace=workspace)
    assert torch.equal(again[keep], out[keep])
