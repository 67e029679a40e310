"""GPU parity of the whole-K few-row GEMM over activations in fragment order (dflash_pack_xf,
dflash_gemm_fewrow_xf): against float64 of the oracle's dequant (<= 1e-2 relative, f32 accumulation), and
against dflash_gemm_fewrow on the same weights, which streams the larger ones (same operands rounded the same way: the two may
differ only in the order of the f32 sums) and takes the same kernels, with the rows brought in by themselves, for the others."""
import numpy as np
import pytest

import qwen_llm_amd as dfl

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = dfl.Context(0)
    yield c
    c.close()


def dev(a):
    import torch

    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def check(y, ref, label):
    y = y.astype(np.float64)
    assert np.all(np.isfinite(y)), f"{label}: non-finite output"
    rel_l2 = np.linalg.norm(y - ref) / max(np.linalg.norm(ref), 1e-30)
    rms = np.sqrt(np.mean(ref ** 2))
    elem = np.max(np.abs(y - ref) / np.maximum(np.abs(ref), rms))
    assert rel_l2 <= 2e-3 and elem <= 1e-2, f"{label}: rel_l2 {rel_l2:.3e} elem {elem:.3e}"


# (n_in, n_out, rows): one stage per wave (n_in <= 4096), two (up to 8192), ragged tile and row counts, two tiles per wave
SHAPES = [(256, 16, 16), (256, 40, 1), (1024, 272, 16), (2048, 5120, 16), (2048, 1000, 7), (4096, 2048, 16), (6144, 2048, 16),
          (5120, 6144, 16), (2048, 12288, 16), (3072, 100, 3), (8192, 48, 16)]
# of those and of these the public operator streams what has more than 24 super-blocks (and what is 17 to 24 in more than one round of tiles)
STREAMED_SHAPES = [(6656, 1000, 16), (6656, 17, 3), (7168, 2047, 5), (8192, 4096, 16)]


def upload(ctx, qtype, n_in, n_out, seed, extreme=False):
    """(device weight, type tag for the GEMM, host blocks in GGUF row order)."""
    if extreme:
        blocks = dfl.synth.extreme_blocks(qtype, n_out * n_in // 256, seed=seed).reshape(n_out, -1)
    else:
        blocks = dfl.synth.random_weight(qtype, n_out, n_in, seed=seed)
    wd = dev(blocks)
    if qtype == dfl.synth.Q4_K:
        return ctx.repack_q4k_tiled(wd, n_in, n_out), dfl.TYPE_Q4_K_TILED, blocks, wd
    return wd, ctx.checked_type(dfl.TYPE_Q6_K, wd), blocks, wd


def reductions(ctx, w, w_type, x, n_in, n_out):
    """Split-K reductions launched by one call of the public operator: one on the streaming kernels, none in one launch."""
    ctx.set_kernel_timing(1)
    ctx.gemm_fewrow(w, w_type, x, n_in, n_out)
    n = ctx.kernel_timing(4)[1]
    ctx.set_kernel_timing(0)
    return n


@pytest.mark.parametrize("qtype", [dfl.synth.Q4_K, dfl.synth.Q6_K])
@pytest.mark.parametrize("n_in,n_out,rows", SHAPES + STREAMED_SHAPES)
@pytest.mark.parametrize("x_dtype", [np.float32, np.float16])
def test_whole_k_gemm_matches_oracle_and_streaming_kernels(ctx, oracle, canaries, qtype, n_in, n_out, rows, x_dtype):
    w, w_type, blocks, w_rows = upload(ctx, qtype, n_in, n_out, seed=n_in + n_out)
    kind = ctx.xf_kind(w_type, n_in, n_out)
    assert kind == (dfl.XF_Q4K if qtype == dfl.synth.Q4_K else dfl.XF_Q6K)
    x = np.random.default_rng(rows).standard_normal((rows, n_in)).astype(x_dtype)
    xd = dev(x)
    xf = ctx.pack_xf(xd, kind)
    y = ctx.gemm_fewrow_xf(w, w_type, xf, rows, n_in, n_out).cpu().numpy()
    canaries.check()
    wf = oracle.dequant(qtype, blocks, n_in * n_out).reshape(n_out, n_in).astype(np.float64)
    ref = x.astype(np.float16).astype(np.float64) @ wf.T  # every few-row kernel rounds its activations to f16
    check(y, ref, f"{n_in}->{n_out} x{rows}")
    # the public operator on the same operands, for the longer K the streaming kernels: same products, other order of the f32 sums
    assert n_in <= 6144 or reductions(ctx, w, w_type, xd, n_in, n_out) == 1
    y2 = ctx.gemm_fewrow(w, w_type, xd, n_in, n_out).cpu().numpy()
    assert np.max(np.abs(y - y2)) <= 2e-5 * max(np.max(np.abs(ref)), 1.0) + 1e-4 * np.sqrt(np.mean(ref ** 2))


@pytest.mark.parametrize("qtype", [dfl.synth.Q4_K, dfl.synth.Q6_K])
def test_whole_k_gemm_extreme_blocks(ctx, oracle, qtype):
    """The reference's extreme blocks (metal/mat_mat.rs:4228-4265: largest scales and codes) within the kernels' range."""
    n_in, n_out, rows = 2048, 320, 16
    w, w_type, blocks, _ = upload(ctx, qtype, n_in, n_out, seed=5, extreme=True)
    x = np.random.default_rng(6).standard_normal((rows, n_in)).astype(np.float32)
    xf = ctx.pack_xf(dev(x), ctx.xf_kind(w_type, n_in, n_out))
    y = ctx.gemm_fewrow_xf(w, w_type, xf, rows, n_in, n_out).cpu().numpy()
    wf = oracle.dequant(qtype, blocks, n_in * n_out).reshape(n_out, n_in).astype(np.float64)
    check(y, x.astype(np.float16).astype(np.float64) @ wf.T, "extreme")


@pytest.mark.parametrize("n_in,n_out,rows", SHAPES)
def test_q6k_tiled_order_is_bit_identical(ctx, n_in, n_out, rows):
    """The tiled, field-planar Q6_K order holds the same blocks in other places: the one-launch GEMM on it equals the same
    GEMM on the GGUF row order bit for bit (ragged tile and row counts, one and two stages per wave, two tiles per wave)."""
    blocks = dfl.synth.random_weight(dfl.synth.Q6_K, n_out, n_in, seed=n_in * 3 + n_out)
    wd = dev(blocks)
    row_type = ctx.checked_type(dfl.TYPE_Q6_K, wd)
    kind = ctx.xf_kind(row_type, n_in, n_out)
    assert kind == dfl.XF_Q6K and ctx.xf_kind(dfl.TYPE_Q6_K_TILED, n_in, n_out) == dfl.XF_Q6K
    wt = ctx.repack_q6k_tiled(wd, n_in, n_out)
    x = dev(np.random.default_rng(rows + 1).standard_normal((rows, n_in)).astype(np.float32))
    xf = ctx.pack_xf(x, kind)
    a = ctx.gemm_fewrow_xf(wd, row_type, xf, rows, n_in, n_out).cpu().numpy()
    b = ctx.gemm_fewrow_xf(wt, dfl.TYPE_Q6_K_TILED, xf, rows, n_in, n_out).cpu().numpy()
    assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_q6k_tiled_guards(ctx):
    import torch

    n_in, n_out = 2048, 512
    blocks = dfl.synth.random_weight(dfl.synth.Q6_K, n_out, n_in, seed=3)
    wt = ctx.repack_q6k_tiled(dev(blocks), n_in, n_out)
    x = torch.zeros((16, n_in), device="cuda")
    with pytest.raises(dfl.DFlashError) as e:   # the streaming kernels do not read this order
        ctx.gemm_fewrow(wt, dfl.TYPE_Q6_K_TILED, x, n_in, n_out)
    assert e.value.kind == "Unsupported" and "gemm_fewrow_xf" in str(e.value)
    bad = dfl.synth.extreme_blocks(dfl.synth.Q6_K, n_out * n_in // 256, seed=1).reshape(n_out, -1).copy()
    bad.view(np.uint8).reshape(-1, 210)[0, 208:210] = np.array([np.float16(128.0)]).view(np.uint8)   # |d| = 128: outside the f16 range
    with pytest.raises(dfl.DFlashError) as e:
        ctx.repack_q6k_tiled(dev(bad), n_in, n_out)
    assert e.value.kind == "Unsupported"


@pytest.mark.parametrize("qtype,tiled", [(dfl.synth.Q4_K, True), (dfl.synth.Q6_K, True), (dfl.synth.Q6_K, False)])
@pytest.mark.parametrize("n_in,n_out,rows", [(2048, 20000, 16), (1024, 9001, 5), (4096, 6000, 16)])
def test_many_rounds_of_tiles_take_the_looping_kernel(ctx, oracle, qtype, tiled, n_in, n_out, rows):
    """A matrix of many more tiles than one round of the chip (an output head) with K of at most 16 super-blocks: the
    looping kernel against f64 of the oracle's dequant, and - the same sums in the same order - bit for bit against
    the one-round kernel on the matrix's first rows."""
    blocks = dfl.synth.random_weight(qtype, n_out, n_in, seed=n_out)
    wd = dev(blocks)
    if qtype == dfl.synth.Q4_K:
        w, w_type = ctx.repack_q4k_tiled(wd, n_in, n_out), dfl.TYPE_Q4_K_TILED
    elif tiled:
        w, w_type = ctx.repack_q6k_tiled(wd, n_in, n_out), dfl.TYPE_Q6_K_TILED
    else:
        w, w_type = wd, ctx.checked_type(dfl.TYPE_Q6_K, wd)
    kind = ctx.xf_kind(w_type, n_in, n_out)
    assert kind != dfl.XF_NONE
    x = np.random.default_rng(rows).standard_normal((rows, n_in)).astype(np.float32)
    xf = ctx.pack_xf(dev(x), kind)
    y = ctx.gemm_fewrow_xf(w, w_type, xf, rows, n_in, n_out).cpu().numpy()
    wf = oracle.dequant(qtype, blocks, n_in * n_out).reshape(n_out, n_in).astype(np.float64)
    check(y, x.astype(np.float16).astype(np.float64) @ wf.T, f"loop {n_in}->{n_out} x{rows}")
    head_rows = 2048   # a matrix of the first rows alone fits one round
    hb = np.ascontiguousarray(blocks[:head_rows])
    hd = dev(hb)
    if qtype == dfl.synth.Q4_K:
        hw, ht = ctx.repack_q4k_tiled(hd, n_in, head_rows), dfl.TYPE_Q4_K_TILED
    elif tiled:
        hw, ht = ctx.repack_q6k_tiled(hd, n_in, head_rows), dfl.TYPE_Q6_K_TILED
    else:
        hw, ht = hd, ctx.checked_type(dfl.TYPE_Q6_K, hd)
    y1 = ctx.gemm_fewrow_xf(hw, ht, xf, rows, n_in, head_rows).cpu().numpy()
    assert np.array_equal(y1.view(np.uint32), y[:, :head_rows].view(np.uint32))


def test_rows_are_independent(ctx):
    """A row of the product depends on its own activation row only: a 16-row block and each row alone agree bit for
    bit (what makes a packed verify equal to token-by-token decoding through the same kernel)."""
    n_in, n_out = 2048, 5120
    for qtype in (dfl.synth.Q4_K, dfl.synth.Q6_K):
        w, w_type, _, _ = upload(ctx, qtype, n_in, n_out, seed=9)
        kind = ctx.xf_kind(w_type, n_in, n_out)
        x = dev(np.random.default_rng(3).standard_normal((16, n_in)).astype(np.float32))
        y = ctx.gemm_fewrow_xf(w, w_type, ctx.pack_xf(x, kind), 16, n_in, n_out).cpu().numpy()
        for r in (0, 7, 15):
            y1 = ctx.gemm_fewrow_xf(w, w_type, ctx.pack_xf(x[r:r + 1].contiguous(), kind), 1, n_in, n_out).cpu().numpy()
            assert np.array_equal(y1[0].view(np.uint32), y[r].view(np.uint32))


@pytest.mark.parametrize("qtype,tiled", [(dfl.synth.Q4_K, True), (dfl.synth.Q6_K, True), (dfl.synth.Q6_K, False)])
@pytest.mark.parametrize("n_in,n_out", [(2048, 1000), (4096, 5120), (6144, 2048), (5120, 6144)])
def test_several_blocks_in_a_call_equal_block_by_block(ctx, canaries, qtype, tiled, n_in, n_out):
    """More than sixteen rows, their blocks' fragment orders one behind the other: one and two stages per wave, one and two
    tiles, a last block that is not full."""
    import torch

    w, w_type, _, _ = upload(ctx, qtype, n_in, n_out, seed=n_in + 7)
    if qtype == dfl.synth.Q6_K and tiled:
        w, w_type = ctx.repack_q6k_tiled(w, n_in, n_out), dfl.TYPE_Q6_K_TILED
    kind = ctx.xf_kind(w_type, n_in, n_out)
    x = dev(np.random.default_rng(37).standard_normal((37, n_in)).astype(np.float32))
    blocks = [ctx.pack_xf(x[i:i + 16].contiguous(), kind) for i in (0, 16, 32)]
    got = ctx.gemm_fewrow_xf(w, w_type, torch.cat(blocks), 37, n_in, n_out)
    want = torch.cat([ctx.gemm_fewrow_xf(w, w_type, b, n, n_in, n_out) for b, n in zip(blocks, (16, 16, 5))])
    canaries.check()
    assert torch.equal(got, want)
    xf = torch.zeros(3 * blocks[0].numel() + 37 * n_out * 4, dtype=torch.uint8, device="cuda")
    with pytest.raises(dfl.DFlashError) as e:  # the result over the third block of rows
        ctx.gemm_fewrow_xf(w, w_type, xf, 37, n_in, n_out, y=xf[2 * blocks[0].numel():])
    assert e.value.kind == "Alias"


def test_shapes_outside_the_path_are_declined(ctx):
    import torch

    assert ctx.xf_kind(dfl.TYPE_Q4_K_TILED, 17408, 5120) == dfl.XF_NONE      # more than two stages per wave
    assert ctx.xf_kind(dfl.TYPE_Q6_K | dfl.TYPE_RANGE_CHECKED, 5120, 151936) == dfl.XF_NONE  # many rounds of the chip and K over 16 super-blocks
    assert ctx.xf_kind(dfl.TYPE_Q6_K | dfl.TYPE_RANGE_CHECKED, 2048, 151936) == dfl.XF_Q6K   # many rounds, short K: the looping kernel
    assert ctx.xf_kind(dfl.TYPE_Q6_K | dfl.TYPE_RANGE_CHECKED, 2048, 2048) == dfl.XF_Q6K
    assert ctx.xf_kind(dfl.TYPE_Q6_K, 2048, 2048) == dfl.XF_NONE             # not range-checked: these kernels scale in f16
    assert ctx.xf_kind(dfl.TYPE_Q4_K, 2048, 2048) == dfl.XF_NONE             # GGUF row order Q4_K: streaming kernels only
    assert ctx.xf_kind(dfl.TYPE_Q8_0, 2048, 2048) == dfl.XF_NONE
    buf = torch.zeros(1 << 20, dtype=torch.uint8, device="cuda")
    y = torch.zeros((16, 5120), dtype=torch.float32, device="cuda")
    with pytest.raises(dfl.DFlashError) as e:
        ctx.gemm_fewrow_xf(buf, dfl.TYPE_Q4_K_TILED, buf, 16, 17408, 5120, y=y)
    assert e.value.kind == "Unsupported"
    with pytest.raises(dfl.DFlashError) as e:
        ctx.pack_xf(torch.zeros((16, 300), device="cuda"), dfl.XF_Q4K)
    assert e.value.kind == "BadShape"


# one super-block and one tile; a last tile and a last super-block slice that are ragged; both sides of one round of tiles at
# one tile a wave, of two tiles a wave (Q4_K), and of the widest K taken (24 super-blocks; 16 for two tiles)
DIRECT_SHAPES = [(256, 5), (2048, 512), (1280, 4097), (4096, 4096), (4096, 4097), (4096, 8192), (4096, 8193), (4352, 130), (6144, 2047), (6400, 64)]


@pytest.mark.parametrize("qtype", [dfl.synth.Q4_K, dfl.synth.Q6_K])
@pytest.mark.parametrize("n_in,n_out", DIRECT_SHAPES)
@pytest.mark.parametrize("rows,x_dtype", [(1, "f32"), (2, "f16"), (15, "f32"), (16, "f16")])
def test_rows_in_row_order_give_the_bits_of_packed_rows(ctx, oracle, canaries, qtype, n_in, n_out, rows, x_dtype):
    """The public operator on small matrices is one launch that brings the caller's rows in itself: the bits of pack_xf +
    gemm_fewrow_xf on the same operands (where both run, the same products in the same order), f16 rows at an 8-byte
    boundary included, and the same bits for either order of the weights and for a row alone."""
    import torch

    w, w_type, blocks, w_rows = upload(ctx, qtype, n_in, n_out, seed=n_in + n_out)
    tag = ctx.checked_type(qtype, w_rows)
    x = dev(np.random.default_rng(rows).standard_normal((rows, n_in)).astype(np.float32))
    if x_dtype == "f16":
        x = torch.cat([torch.zeros(4, device="cuda", dtype=torch.float16), x.half().flatten()])[4:].view(rows, n_in)
        assert x.data_ptr() % 16 == 8
    y = ctx.gemm_fewrow(w_rows, tag, x, n_in, n_out)
    canaries.check()
    assert torch.equal(ctx.gemm_fewrow(w, w_type, x, n_in, n_out).view(torch.int32), y.view(torch.int32))
    alone = x[rows - 1:].clone()
    assert torch.equal(ctx.gemm_fewrow(w_rows, tag, alone, n_in, n_out).view(torch.int32), y[rows - 1:].view(torch.int32))
    tiles = (n_out + 15) // 16
    one_round = 256 * (16 // min(n_in // 256, 16))
    if n_in <= 6144 and (tiles <= one_round or (qtype == dfl.synth.Q4_K and n_in <= 4096 and tiles <= 2 * one_round)):
        xf = ctx.pack_xf(x, ctx.xf_kind(w_type, n_in, n_out))
        assert torch.equal(ctx.gemm_fewrow_xf(w, w_type, xf, rows, n_in, n_out).view(torch.int32), y.view(torch.int32))
    cols = np.unique(np.concatenate([np.arange(min(n_out, 40)), np.arange(max(0, n_out - 40), n_out)]))
    wf = oracle.dequant(qtype, np.ascontiguousarray(blocks[cols]), len(cols) * n_in).reshape(len(cols), n_in).astype(np.float64)
    ref = x.half().cpu().numpy().astype(np.float64) @ wf.T
    check(y[:, torch.from_numpy(cols).cuda()].cpu().numpy(), ref, f"{n_in}->{n_out} x{rows}")


@pytest.mark.parametrize("n_in,n_out,streamed", [(5632, 512, 0), (5888, 512, 1), (6144, 1024, 1), (6144, 2032, 1), (6144, 2033, 0), (6144, 4096, 0),
                                                 (6400, 4096, 1)])
def test_q6k_of_many_super_blocks_and_few_tiles_streams(ctx, oracle, n_in, n_out, streamed):
    """Beyond 22 super-blocks one launch pays from half a round of tiles on; both sides of the line against the f64 product."""
    w, w_type, blocks, _ = upload(ctx, dfl.synth.Q6_K, n_in, n_out, seed=n_out)
    x = np.random.default_rng(n_in).standard_normal((16, n_in)).astype(np.float32)
    assert reductions(ctx, w, w_type, dev(x), n_in, n_out) == streamed
    y = ctx.gemm_fewrow(w, w_type, dev(x), n_in, n_out).cpu().numpy()
    cols = np.unique(np.concatenate([np.arange(40), np.arange(n_out - 40, n_out)]))
    wf = oracle.dequant(dfl.synth.Q6_K, np.ascontiguousarray(blocks[cols]), len(cols) * n_in).reshape(len(cols), n_in).astype(np.float64)
    check(y[:, cols], x.astype(np.float16).astype(np.float64) @ wf.T, f"{n_in}->{n_out}")


# (type, tiled order, n_in, n_out): one round of tiles, in both orders of Q4_K, many rounds in both, Q6_K
SWITCHED = [(dfl.synth.Q4_K, True, 4096, 4096), (dfl.synth.Q4_K, False, 4096, 4096), (dfl.synth.Q4_K, True, 2560, 16384), (dfl.synth.Q4_K, False, 2560, 16384),
            (dfl.synth.Q6_K, False, 2048, 1024)]


def switched_routes(ctx):
    """For each of SWITCHED the split-K reductions of a call."""
    routes = []
    for qtype, tiled, n_in, n_out in SWITCHED:
        w, w_type, _, w_rows = upload(ctx, qtype, n_in, n_out, seed=1)
        if not tiled:
            w, w_type = w_rows, ctx.checked_type(qtype, w_rows)
        routes.append(reductions(ctx, w, w_type, dev(np.ones((5, n_in), np.float32)), n_in, n_out))
    return routes


@pytest.mark.parametrize("qtype,tiled,n_in,n_out,stamps", [(*s, [1, 0] if s[0] == dfl.synth.Q4_K else [0, 0]) for s in SWITCHED] +
                         [(dfl.synth.Q4_K, True, 8192, 528, [1, 1])])
def test_dispatch_stamps_of_a_q4k_product(ctx, qtype, tiled, n_in, n_out, stamps):
    """Stamps of single dispatches: the kernel of a Q4_K product whichever it is, and the tiled order's reduction where it has one."""
    w, w_type, _, w_rows = upload(ctx, qtype, n_in, n_out, seed=1)
    if not tiled:
        w, w_type = w_rows, ctx.checked_type(qtype, w_rows)
    ctx.set_kernel_timing(2)
    ctx.gemm_fewrow(w, w_type, dev(np.ones((5, n_in), np.float32)), n_in, n_out)
    got = [ctx.kernel_timing(slot) for slot in (5, 6)]
    ctx.set_kernel_timing(0)
    assert [n for _, n in got] == stamps and all((ms > 0) == (n > 0) for ms, n in got)


_SWITCH_PROBE = """
import sys
sys.path.insert(0, "tests")
import qwen_llm_amd as dfl
import test_gpu_gemm_whole as t
print(t.switched_routes(dfl.Context(0)))
"""


@pytest.mark.parametrize("name,value,streamed", [
    ("DFLASH_GEMM_WHOLE", "0", [1, 1, 1, 1, 1]), ("DFLASH_GEMM_WHOLE_LOOP", "0", [0, 0, 1, 1, 0]), ("DFLASH_GEMM_WGS", "200", [1, 1, 1, 1, 1]),
    ("DFLASH_GEMM_WAVES", "8", [1, 1, 1, 1, 1]), ("DFLASH_Q4K_SLAB", "0", [0, 1, 0, 1, 0])])
def test_switches_of_the_streaming_kernels_reach_the_public_operator(ctx, name, value, streamed):
    """What a switch says of a matrix holds for the public operator's call on it: with the whole-K kernels off, or with a launch geometry
    of the streaming kernels asked for, the matrix streams.  (The switches are read once per process.)"""
    import os
    import subprocess
    import sys

    assert switched_routes(ctx) == [0, 0, 0, 0, 0]
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root + os.pathsep + os.environ.get("PYTHONPATH", ""), **{name: value})
    r = subprocess.run([sys.executable, "-c", _SWITCH_PROBE], env=env, cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.split("\n")[-2] == str(streamed)


# many rounds of tiles: K of one super-block (sixteen tiles a workgroup), of one and two super-blocks a wave, an odd split of K
# (17: nine waves, one of them with one super-block), the widest (24); a ragged last tile, a last round that few workgroups have
WIDE_SHAPES = [(256, 140001), (768, 45000), (1024, 33000), (2048, 16400), (2560, 8200), (4096, 8193), (4352, 12300), (5120, 17408), (6144, 12289)]


@pytest.mark.parametrize("n_in,n_out", WIDE_SHAPES)
@pytest.mark.parametrize("rows,x_dtype", [(1, "f32"), (7, "f16"), (9, "f32"), (16, "f16"), (16, "f32")])
def test_rows_in_row_order_against_many_rounds_of_tiles(ctx, oracle, canaries, n_in, n_out, rows, x_dtype):
    """The looping product of the public operator: against the f64 product on columns of every round, the same bits for either
    order of the weights and for a row alone, twice in a row, rows whose sub-block sums pass the f16 range included."""
    import torch

    blocks = dfl.synth.random_blocks(dfl.synth.Q4_K, n_out * n_in // 256, seed=n_in + n_out).reshape(n_out, -1)
    w_rows = dev(blocks)
    tag = ctx.checked_type(dfl.synth.Q4_K, w_rows)
    wt = ctx.repack_q4k_tiled(w_rows, n_in, n_out)
    x = np.random.default_rng(rows).standard_normal((rows, n_in)).astype(np.float32)
    x[rows // 2] += 2500.0
    xd = dev(x.astype(np.float16 if x_dtype == "f16" else np.float32))
    y = ctx.gemm_fewrow(w_rows, tag, xd, n_in, n_out)
    canaries.check()
    for other in (ctx.gemm_fewrow(wt, dfl.TYPE_Q4_K_TILED, xd, n_in, n_out), ctx.gemm_fewrow(w_rows, tag, xd, n_in, n_out)):
        assert torch.equal(other.view(torch.int32), y.view(torch.int32))
    alone = ctx.gemm_fewrow(wt, dfl.TYPE_Q4_K_TILED, xd[rows - 1:].clone(), n_in, n_out)
    assert torch.equal(alone.view(torch.int32), y[rows - 1:].view(torch.int32))
    cols = np.unique(np.concatenate([np.arange(16), np.random.default_rng(n_out).integers(0, n_out, 500), np.arange(n_out - 20, n_out)]))
    wf = oracle.dequant(dfl.synth.Q4_K, np.ascontiguousarray(blocks[cols]), len(cols) * n_in).reshape(len(cols), n_in).astype(np.float64)
    ref = x.astype(np.float16).astype(np.float64) @ wf.T
    got = y[:, torch.from_numpy(cols).cuda()].cpu().numpy()
    for r in range(rows):
        check(got[r:r + 1], ref[r:r + 1], f"{n_in}->{n_out} row {r}")
