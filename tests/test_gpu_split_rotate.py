"""Rotated K ranges and the split Basic down, on integer-valued operands whose sums are exact: every
result must be the float64 product rounded once, whatever the order of the sum.

Rotation (rows <= 256, a padded depth whose pitch is a multiple of 4 KiB, 64 MiB of weights or more):
a K tail then lands in the middle of a tile's iterations, and every tile column starts elsewhere.  Split Basic: given a
workspace the tiles are split along H and finished in the launch; without one they run whole.
"""
import ctypes
import sys

import pytest
import torch

from ffn_optim_amd import _lib
from gpu_workspace import counters_are_zero, poisoned_workspace

pytestmark = pytest.mark.gpu


def say(*args):
    print("[split-rotate]", *args, file=sys.stderr, flush=True)


def _align(v, unit):
    return (v + unit - 1) // unit * unit


def _operands(m, h, n, hp, np_, dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    mp = _align(m, 64)
    hid = torch.zeros((mp, hp), dtype=dtype)
    w2 = torch.zeros((np_, hp), dtype=dtype)
    hid[:m, :h] = torch.randint(-2, 3, (m, h), generator=gen, dtype=torch.int8).to(dtype)
    w2[:n, :h] = torch.randint(-2, 3, (n, h), generator=gen, dtype=torch.int8).to(dtype)
    # integer sums below 2^24 are exact in float32
    golden = torch.zeros((mp, np_), dtype=dtype)
    golden[:m] = (hid[:m].float() @ w2.float().T).to(dtype)
    return hid, w2, golden


# depths with and without a K tail (2000 = 31 x 64 + 16, 8176 = 63 x 128 + 112)
@pytest.mark.parametrize("m, h, n, dtype", [
    (1, 2048, 16384, torch.bfloat16),
    (16, 8176, 4100, torch.bfloat16),
    (65, 2000, 16500, torch.float16),
    (256, 65536, 512, torch.bfloat16),
    (257, 2048, 16384, torch.float16),   # one row too many: in step
    (65, 2000, 192, torch.float16),      # too few weights: in step, split
])
def test_rotated_down_is_exact_on_all_variants(m, h, n, dtype):
    lib = _lib.load()
    hp, np_ = _align(h, 2048), _align(n, 64)
    hid, w2, golden = _operands(m, h, n, hp, np_, dtype, m)
    code = _lib.BF16 if dtype == torch.bfloat16 else _lib.FP16
    hid_d, w2_d = hid.cuda(), w2.cuda()
    stream = torch.cuda.current_stream().cuda_stream
    ran = 0
    for variant in range(lib.ffn_mi355x_num_variants()):
        for down in ("basic", "streamk"):
            try:
                plan = _lib.make_plan(hid.shape[0], 64, hp, np_, code, down, "erf", 256, 0, variant, m=m)
            except ValueError:
                continue
            _lib.set_operands(plan, 64, h, n, 64, 64, hp)
            for ws in (poisoned_workspace(plan), None):
                if ws is None and down == "streamk":
                    continue
                say(m, h, n, dtype, variant, down, "split" if plan.down_sk_tiles and ws is not None else "whole")
                out = torch.full(golden.shape, float("nan"), dtype=dtype, device="cuda")
                _lib.check(lib.ffn_mi355x_down(ctypes.byref(plan), hid_d.data_ptr(), w2_d.data_ptr(), out.data_ptr(),
                                               ws.data_ptr() if ws is not None else None, stream))
                torch.cuda.synchronize()
                assert torch.equal(out.cpu()[:m].view(torch.int16), golden[:m].view(torch.int16)), (variant, down)
                assert ws is None or counters_are_zero(plan, ws), (variant, down)
                ran += 1
    assert ran > 2 * lib.ffn_mi355x_num_variants()


@pytest.mark.parametrize("m, k, h", [(16, 2048, 16384), (100, 16368, 2200)])
def test_rotated_up_matches_gelu(m, k, h):
    """hidden is the erf GELU of the exact sum, to one unit in the last place (float64 GELU)."""
    lib = _lib.load()
    kp, hp = _align(k, 2048), _align(h, 64)
    x, w1, z = _operands(m, k, h, kp, hp, torch.bfloat16, k)
    z64 = x[:m].double() @ w1.double().T
    truth = (0.5 * z64 * torch.special.erfc(-z64 / 2 ** 0.5)).to(torch.bfloat16)
    xd, wd = x.cuda(), w1.cuda()
    stream = torch.cuda.current_stream().cuda_stream

    def ordinal(bits16):
        b = bits16.int() & 0xFFFF
        return torch.where(b >= 0x8000, -(b & 0x7FFF), b)

    for variant in range(lib.ffn_mi355x_num_variants()):
        plan = _lib.make_plan(x.shape[0], kp, hp, 64, _lib.BF16, "basic", "erf", 256, variant, -1, m=m)
        _lib.set_operands(plan, k, h, 64, kp, kp, hp)
        say("up", m, k, h, variant, plan.up_sk_tiles)
        hidden = torch.full((x.shape[0], hp), float("nan"), dtype=torch.bfloat16, device="cuda")
        ws = poisoned_workspace(plan)
        _lib.check(lib.ffn_mi355x_up(ctypes.byref(plan), xd.data_ptr(), wd.data_ptr(), hidden.data_ptr(),
                                     ws.data_ptr(), stream))
        torch.cuda.synchronize()
        ulps = (ordinal(hidden.cpu()[:m].view(torch.int16)) - ordinal(truth.view(torch.int16))).abs()
        assert int(ulps.max()) <= 1, variant


def test_split_basic_in_place_operands_match_their_copies():
    """ffn() on operands read in place and the prepared copies run the same split and the same
    rotated order: bit-identical, and equal on a second call on the same workspace."""
    from ffn_optim_amd import ffn, prepare_ffn
    gen = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn((100, 2040), generator=gen, device="cuda").bfloat16()
    w1 = (torch.randn((16384, 2040), generator=gen, device="cuda") / 45).bfloat16()
    w2 = (torch.randn((2100, 16384), generator=gen, device="cuda") / 128).bfloat16()
    prepared = prepare_ffn(x, w1, w2)
    assert prepared.plan.native.down_sk_tiles > 0 and prepared.plan.native.down_dp_tiles == 0
    first = prepared.run().clone()
    assert torch.equal(first, prepared.run())
    assert torch.equal(first, ffn(x, w1, w2))


@pytest.mark.parametrize("m, h, n", [
    (1, 6161, 512),     # 49 iterations in four pieces: all but the first straddle two tiles
    (32, 9088, 3072),   # 71 iterations in two
    (65, 2560, 192),    # the shallowest depth that splits, in even pieces
    (65, 2496, 192),    # one step shallower: whole
])
def test_split_basic_down_by_depth(m, h, n):
    """The automatic Basic down at the edges of its split: pieces that do not cut a tile evenly, and
    the depth below which tiles stay whole; exact against the float product, run after run."""
    lib = _lib.load()
    hp, np_ = _align(h, 64), _align(n, 64)
    hid, w2, golden = _operands(m, h, n, hp, np_, torch.bfloat16, h)
    hid_d, w2_d = hid.cuda(), w2.cuda()
    plan = _lib.make_plan(hid.shape[0], 64, hp, np_, _lib.BF16, "basic", "erf", 256, m=m)
    assert (plan.down_sk_tiles > 0) == (h >= 2560)
    ws = poisoned_workspace(plan)
    say("depth", m, h, n, plan.down_variant, plan.down_tiles, plan.down_grid)
    for _ in range(3):
        out = torch.full(golden.shape, float("nan"), dtype=torch.bfloat16, device="cuda")
        _lib.check(lib.ffn_mi355x_down(ctypes.byref(plan), hid_d.data_ptr(), w2_d.data_ptr(), out.data_ptr(),
                                       ws.data_ptr(), torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        assert torch.equal(out.cpu()[:m].view(torch.int16), golden[:m].view(torch.int16))
        assert counters_are_zero(plan, ws)


GUARD = 0x5A5A5A5A


def _ffn_operands(m, k, h, n, plan):
    gen = torch.Generator(device="cuda").manual_seed(k)
    mp, kp, hp, np_ = plan.mp, plan.kp, plan.hp, plan.np
    x = torch.zeros((mp, kp), dtype=torch.bfloat16, device="cuda")
    w1 = torch.zeros((hp, kp), dtype=torch.bfloat16, device="cuda")
    w2 = torch.zeros((np_, hp), dtype=torch.bfloat16, device="cuda")
    for t, rows, cols, std in ((x, m, k, 1.0), (w1, h, k, k ** -0.5), (w2, n, h, h ** -0.5)):
        t[:rows, :cols] = (torch.randn((rows, cols), generator=gen, device="cuda") * std).bfloat16()
    hidden = torch.empty((mp, hp), dtype=torch.bfloat16, device="cuda")
    return x, w1, w2, hidden


def _run_ffn(plan, x, w1, w2, hidden, ws_ptr):
    out = torch.full((plan.mp, plan.np), float("nan"), dtype=torch.bfloat16, device="cuda")
    hidden.fill_(float("nan"))
    _lib.check(_lib.load().ffn_mi355x_run(ctypes.byref(plan), x.data_ptr(), w1.data_ptr(), w2.data_ptr(),
                                          hidden.data_ptr(), out.data_ptr(), ws_ptr,
                                          torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return out


def _plain_plan(m, k, h, n):
    return _lib.make_plan(_align(m, 64), _align(k, 16), _align(h, 64), _align(n, 64), _lib.BF16, "basic", "erf", 256,
                          m=m, split_down=False)


@pytest.mark.parametrize("m, k, h, n", [(8, 6784, 11648, 320), (3, 4832, 7232, 640), (128, 4096, 16384, 4096)])
def test_plain_basic_plan_leaves_ws_alone(m, k, h, n):
    """A Basic plan nobody asked to split ignores `ws`: a 64-byte block of a larger buffer, a block whose
    words are no counters, and NULL give the same bits, and the buffer keeps every word."""
    plan = _plain_plan(m, k, h, n)
    assert plan.workspace_bytes == 0 and plan.down_sk_tiles == 0
    x, w1, w2, hidden = _ffn_operands(m, k, h, n, plan)
    say("plain", m, k, h, n)
    expected = _run_ffn(plan, x, w1, w2, hidden, None)
    pool = torch.full((32 << 20,), GUARD, dtype=torch.int32, device="cuda")   # room for any split of these shapes
    got = _run_ffn(plan, x, w1, w2, hidden, pool.data_ptr())
    assert torch.equal(got, expected) and bool((pool == GUARD).all())
    # the two stages on their own, the up without a workspace
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream
    out = torch.full_like(expected, float("nan"))
    _lib.check(lib.ffn_mi355x_up(ctypes.byref(plan), x.data_ptr(), w1.data_ptr(), hidden.data_ptr(), None, stream))
    _lib.check(lib.ffn_mi355x_down(ctypes.byref(plan), hidden.data_ptr(), w2.data_ptr(), out.data_ptr(),
                                   pool.data_ptr(), stream))
    torch.cuda.synchronize()
    assert torch.equal(out, expected) and bool((pool == GUARD).all())


def test_plain_basic_plan_with_split_up_takes_the_ups_workspace():
    """A plain Basic plan with a split up GEMM needs the up's bytes alone, and stays inside them."""
    m, k, h, n = 3, 7552, 3328, 3712
    plan = _plain_plan(m, k, h, n)
    assert plan.up_sk_tiles > 0 and plan.down_sk_tiles == 0
    x, w1, w2, hidden = _ffn_operands(m, k, h, n, plan)
    clean = poisoned_workspace(plan)
    expected = _run_ffn(plan, x, w1, w2, hidden, clean.data_ptr())
    pool = torch.full((32 << 20,), GUARD, dtype=torch.int32, device="cuda")
    words = plan.workspace_bytes // 4
    pool[:words] = poisoned_workspace(plan).view(torch.int32)
    say("up-sized", plan.workspace_bytes)
    for _ in range(3):
        assert torch.equal(_run_ffn(plan, x, w1, w2, hidden, pool.data_ptr()), expected)
        assert bool((pool[words:] == GUARD).all()) and counters_are_zero(plan, pool)


@pytest.mark.parametrize("m, k, h, n", [
    (8, 6784, 11648, 320),
    (1, 512, 6161, 512),        # uneven pieces, two slots a workgroup
    (128, 4096, 16384, 4096),
    (3, 7552, 3328, 3712),      # both GEMMs split
])
def test_split_basic_down_from_dirty_counters(m, k, h, n):
    """A split Basic down through ffn_mi355x_run starts right from whatever its counters held (the up
    launch clears them), stays inside plan.workspace_bytes and leaves the counters zero."""
    plan = _lib.make_plan(_align(m, 64), _align(k, 16), _align(h, 64), _align(n, 64), _lib.BF16, "basic", "erf", 256,
                          m=m)
    assert plan.down_sk_tiles > 0
    x, w1, w2, hidden = _ffn_operands(m, k, h, n, plan)
    clean = poisoned_workspace(plan)
    expected = _run_ffn(plan, x, w1, w2, hidden, clean.data_ptr())
    assert not bool(expected[:m, :n].isnan().any())
    pool = torch.full((32 << 20,), GUARD, dtype=torch.int32, device="cuda")
    words = plan.workspace_bytes // 4
    pool[:words] = poisoned_workspace(plan).view(torch.int32)
    stride = 32 if (plan.up_sk_tiles + plan.down_sk_tiles) * 32 * 4 <= 64 << 10 else 1
    down_words = plan.down_sk_tiles * stride
    say("dirty", m, k, h, n, plan.up_sk_tiles, plan.down_sk_tiles)
    for garbage in (1, 0x7FFFFFFF, -1):
        pool[:down_words] = garbage
        assert torch.equal(_run_ffn(plan, x, w1, w2, hidden, pool.data_ptr()), expected)
        assert bool((pool[words:] == GUARD).all()) and counters_are_zero(plan, pool)
    # and without a workspace: whole tiles of the same size.  Both round an FP32 sum to bf16 (half an ulp,
    # 2^-9 of the value, each), and the sums' own difference is far below that: 2^-7 of the largest value
    if plan.up_sk_tiles == 0:
        whole = _run_ffn(plan, x, w1, w2, hidden, None)
        scale = expected[:m, :n].float().abs().max()
        assert float((whole[:m, :n].float() - expected[:m, :n].float()).abs().max()) <= float(scale) * 2 ** -7
