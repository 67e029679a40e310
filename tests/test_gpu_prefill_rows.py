"""The grouped prefill's many-row products (csrc/gemm_rows.hip) against the block-by-block verify, whose own products
are the oracle-checked ones: captured residuals bit for bit.

The row counts are those where a launch changes its shape: two blocks (one of a single row); the whole-K kernel's last
and the split's first count (64 | 80 rows narrow, 192 | 200 experts); tiles of every number of row blocks with a last
tile that is not full; several rounds of the chip.  K and the column counts bring each kind of cut: 5120 (whole-K slices, twenty super-blocks), 17408 (stream-K
ranges that differ from tile group to tile group), 1024 (fewer super-blocks than slices), Q6_K projections, experts
with one to four blocks per tile."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

import qwen_llm_amd as dfl

pytestmark = pytest.mark.gpu

SHAPES = {
    "wide": (dfl.ModelConfig(n_layers=2, hidden=5120, n_q=32, n_kv=8, head_dim=128, ffn=17408, vocab=2048), dfl.synth.Q4_K),
    "narrow": (dfl.ModelConfig(n_layers=2, hidden=1024, n_q=16, n_kv=8, head_dim=128, ffn=3072, vocab=2048), dfl.synth.Q4_K),
    "experts": (dfl.ModelConfig(n_layers=2, hidden=2048, n_q=16, n_kv=2, head_dim=256, ffn=0, vocab=2048, n_expert=32, n_expert_used=4,
                                ffn_expert=768, ffn_shared=768), dfl.synth.Q6_K),
}
SHAPES["experts128"] = (dfl.ModelConfig(n_layers=2, hidden=2048, n_q=16, n_kv=2, head_dim=256, ffn=0, vocab=2048, n_expert=128, n_expert_used=8,
                                        ffn_expert=768, ffn_shared=768), dfl.synth.Q6_K)
# (Q6_K projections whose weights the whole-K kernel does not hold, two tiles of a super-block or two super-blocks a wave)
SHAPES["q6k4096"] = (dfl.ModelConfig(n_layers=2, hidden=4096, n_q=32, n_kv=8, head_dim=128, ffn=3072, vocab=2048), dfl.synth.Q6_K)
SHAPES["q6k5120"] = (dfl.ModelConfig(n_layers=2, hidden=5120, n_q=32, n_kv=8, head_dim=128, ffn=3072, vocab=2048), dfl.synth.Q6_K)
SHAPES["heads64"] = (dfl.ModelConfig(n_layers=2, hidden=1024, n_q=24, n_kv=2, head_dim=64, ffn=3072, vocab=2048), dfl.synth.Q4_K)
SHAPES["heads64x12"] = (dfl.ModelConfig(n_layers=2, hidden=1024, n_q=48, n_kv=4, head_dim=64, ffn=3072, vocab=2048), dfl.synth.Q4_K)
SHAPES["heads256x5"] = (dfl.ModelConfig(n_layers=2, hidden=1280, n_q=5, n_kv=1, head_dim=256, ffn=3072, vocab=2048), dfl.synth.Q4_K)

SHAPES["heads256x1"] = (dfl.ModelConfig(n_layers=2, hidden=1024, n_q=4, n_kv=4, head_dim=256, ffn=3072, vocab=2048), dfl.synth.Q4_K)
SHAPES["held4096"] = (dfl.ModelConfig(n_layers=2, hidden=4096, n_q=16, n_kv=4, head_dim=128, ffn=3072, vocab=2048), dfl.synth.Q4_K)
# (gate|up of more tiles than one round, behind it a down projection that by its own shape the whole-K kernel would take: K of
# 27 super-blocks, and of 17, the fewest, with 9 of gate|up)
SHAPES["ffn6912"] = (dfl.ModelConfig(n_layers=2, hidden=2560, n_q=16, n_kv=4, head_dim=128, ffn=6912, vocab=2048), dfl.synth.Q4_K)
SHAPES["ffn4352"] = (dfl.ModelConfig(n_layers=2, hidden=2304, n_q=16, n_kv=4, head_dim=128, ffn=4352, vocab=2048), dfl.synth.Q4_K)
# (q|k|v of 16 super-blocks and 9216 columns: more tiles than one round of 256 CUs, the looping whole-K kernel)
SHAPES["loop4096"] = (dfl.ModelConfig(n_layers=2, hidden=4096, n_q=64, n_kv=4, head_dim=128, ffn=3072, vocab=2048), dfl.synth.Q4_K)
# (a mixture's projections in Q4_K: wo of 16 super-blocks, by sums that no kernel ahead of it has left)
SHAPES["experts_q4k"] = (dfl.ModelConfig(n_layers=3, hidden=2048, n_q=16, n_kv=2, head_dim=256, ffn=0, vocab=2048, n_expert=32, n_expert_used=4,
                                         ffn_expert=768, ffn_shared=768), dfl.synth.Q4_K)
SHAPES["heads256x64"] = (dfl.ModelConfig(n_layers=2, hidden=1024, n_q=64, n_kv=16, head_dim=256, ffn=3072, vocab=2048), dfl.synth.Q4_K)
SHAPES["heads256x12"] = (dfl.ModelConfig(n_layers=2, hidden=1024, n_q=12, n_kv=1, head_dim=256, ffn=3072, vocab=2048), dfl.synth.Q4_K)


@pytest.fixture(scope="module")
def ctx():
    c = dfl.Context(0, workspace_bytes=256 << 20)
    yield c
    c.close()


@pytest.mark.parametrize("rows", [17, 64, 80, 97, 192, 200, 273, 530, 1001])
@pytest.mark.parametrize("shape", ["experts", "narrow", "wide", "q6k4096", "q6k5120"])
def test_many_row_prefill_equals_block_by_block(ctx, shape, rows):
    cfg, attn_type = SHAPES[shape]
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type))
    one, many = dfl.Session(ctx, model, rows + 16, [0, 1]), dfl.Session(ctx, model, rows + 16, [0, 1])
    tokens = np.random.default_rng(rows).integers(0, cfg.vocab, rows).tolist()
    got = many.prefill_blocks(tokens, 0)
    want = torch.cat([one.encode_packed_verify_layer_major(tokens[i:i + 16], i, want_head=False).hidden_capture for i in range(0, rows, 16)])
    assert torch.equal(got, want)
    one.close()
    many.close()


@pytest.mark.parametrize("rows", [33, 49, 113, 129, 161, 225, 305, 369, 481])
@pytest.mark.parametrize("shape", ["experts", "narrow", "wide", "q6k4096"])
def test_last_row_tiles_of_every_fill_equal_block_by_block(ctx, shape, rows):
    """3 to 31 blocks: last row tiles of up to half their blocks (computed as half a tile), of more, and of a single row."""
    test_many_row_prefill_equals_block_by_block(ctx, shape, rows)


@pytest.mark.parametrize("rows", [17, 64, 200, 530])
@pytest.mark.parametrize("shape", ["ffn4352", "ffn6912"])
def test_down_behind_a_streamed_gate_up_equals_block_by_block(ctx, shape, rows):
    """The block path's down product streams there, although the matrix alone would be a whole-K product: K is cut elsewhere."""
    test_many_row_prefill_equals_block_by_block(ctx, shape, rows)


@pytest.mark.parametrize("head,rows", [(7, 40), (245, 33), (480, 400), (1000, 530), (1000, 1100)])
@pytest.mark.parametrize("shape", ["narrow", "experts", "heads64", "heads64x12", "heads256x5"])
def test_continued_prefill_equals_block_by_block(ctx, shape, head, rows):
    """Behind a context, where the attention takes the keys of many blocks split by split in one workgroup or leaves
    them to several (by how many workgroups there are), across buckets of context lengths, with a last split and a
    last stage that are not full, a first position off the stages' raster, and groups of 2, 5, 8 and 12 heads."""
    cfg, attn_type = SHAPES[shape]
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type))
    one, many = dfl.Session(ctx, model, head + rows + 16, [0, 1]), dfl.Session(ctx, model, head + rows + 16, [0, 1])
    tokens = np.random.default_rng(rows).integers(0, cfg.vocab, head + rows).tolist()
    for s in (one, many):
        for i in range(0, head, 16):
            s.encode_packed_verify_layer_major(tokens[i:min(i + 16, head)], i, want_head=False)
    got = many.prefill_blocks(tokens[head:], head)
    want = torch.cat([one.encode_packed_verify_layer_major(tokens[i:i + 16], i, want_head=False).hidden_capture for i in range(head, head + rows, 16)])
    assert torch.equal(got, want)
    one.close()
    many.close()


@pytest.mark.parametrize("head,rows", [(0, 2033), (64, 1500), (0, 513), (480, 70), (37, 600)])
@pytest.mark.parametrize("shape", ["experts", "heads256x1", "heads256x5", "heads256x12"])
def test_heads_of_256_equal_block_by_block(ctx, shape, head, rows):
    """Keys walked twice in one workgroup against splits and their merge: one, four, five, six and eight waves, up to eight
    splits (the total in registers) and more (in the output rows, also where the last block is short), a last split of one stage and of two."""
    test_continued_prefill_equals_block_by_block(ctx, shape, head, rows)


@pytest.mark.parametrize("shape,head,rows", [("experts", 0, 1030), ("experts", 37, 1041), ("heads256x64", 0, 272), ("heads256x64", 0, 287), ("heads256x64", 450, 318)])
def test_two_blocks_a_workgroup_equal_block_by_block(ctx, shape, head, rows):
    """Heads of 256 beyond a workgroup a CU: even and odd numbers of blocks (one in the middle without a second), a short last
    block, up to eight splits in both blocks of a workgroup, in the second alone and in neither."""
    test_continued_prefill_equals_block_by_block(ctx, shape, head, rows)


@pytest.mark.parametrize("shape,head,rows", [("heads64x12", 249, 165), ("narrow", 2980, 150), ("heads256x12", 1350, 100)])
def test_prefill_over_a_change_of_the_splits_length_equals_block_by_block(ctx, shape, head, rows):
    """Blocks of one split launch whose last has fewer splits than the ones ahead of it: the keys of a split pass a whole stage at
    384 (6 splits asked for), 3072 (32) and 1408 (22) positions, and from there on splits are longer and fewer."""
    test_continued_prefill_equals_block_by_block(ctx, shape, head, rows)


def _rescale(mat, factor):
    blocks = mat[1].view(-1, dfl.synth.BLOCK_BYTES[dfl.synth.Q4_K])
    blocks[:, :4] = (blocks[:, :4].contiguous().view(torch.float16) * factor).view(torch.uint8)


@pytest.mark.parametrize("where", ["gate_up", "down"])
@pytest.mark.parametrize("shape", ["experts", "experts128", "narrow", "wide"])
def test_prefill_equals_block_by_block_with_sums_past_f16(ctx, shape, where):
    """Activations whose sub-block sums pass the largest f16, with every activation itself inside: in the normed rows
    (gains of 4000: the sums of 32 are about +-23000) or in the SwiGLU rows (gate = up: 32 values of one sign, some 2000
    each).  A block of 16 picks some 28 of 32 experts, gate and up of a tile on two waves, or 80 of 128, both on one."""
    cfg, attn_type = SHAPES[shape]
    w = dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type)
    for L in w["layers"]:
        L["post_norm"] = L["post_norm"] * (4000.0 if where == "gate_up" else 47.0)
        for gate, up in (("gate", "up"),) + ((("gate_exps", "up_exps"),) if cfg.n_expert else ()):
            if where == "gate_up":
                _rescale(L[gate], 1 / 400)
                _rescale(L[up], 1 / 400)
            else:
                L[up] = (L[gate][0], L[gate][1].clone())
    model = dfl.TargetModel(ctx, cfg, w)
    rows = 97
    one, many = dfl.Session(ctx, model, rows + 16, [0, 1]), dfl.Session(ctx, model, rows + 16, [0, 1])
    tokens = np.random.default_rng(rows).integers(0, cfg.vocab, rows).tolist()
    got = many.prefill_blocks(tokens, 0)
    want = torch.cat([one.encode_packed_verify_layer_major(tokens[i:i + 16], i, want_head=False).hidden_capture for i in range(0, rows, 16)])
    assert torch.isfinite(got).all() and torch.isfinite(want).all()
    assert torch.equal(got, want)
    one.close()
    many.close()


@pytest.mark.parametrize("gain", [1.0, 4000.0])
@pytest.mark.parametrize("rows", [17, 64, 97, 128, 192, 200])
@pytest.mark.parametrize("shape", ["held4096", "wide", "loop4096"])
def test_projections_with_minima_by_sums_equal_block_by_block(ctx, shape, rows, gain):
    """Q4_K projections of 16 and 20 super-blocks, whose minima go by the sub-block sums on both paths (the whole-K kernel's
    own and the norm kernel's) where the block's product is one round of the chip, by twin products on both where it loops: blocks past held weights up to the last such count and the first of the split, with a
    last block that is not full, and with sums past the largest f16 (gains of 4000)."""
    cfg, attn_type = SHAPES[shape]
    w = dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type)
    for L in w["layers"]:
        L["attn_norm"] = L["attn_norm"] * gain
        for name in ("wq", "wk", "wv"):
            _rescale(L[name], min(1.0, 10 / gain))
    model = dfl.TargetModel(ctx, cfg, w)
    one, many = dfl.Session(ctx, model, rows + 16, [0, 1]), dfl.Session(ctx, model, rows + 16, [0, 1])
    tokens = np.random.default_rng(rows).integers(0, cfg.vocab, rows).tolist()
    got = many.prefill_blocks(tokens, 0)
    want = torch.cat([one.encode_packed_verify_layer_major(tokens[i:i + 16], i, want_head=False).hidden_capture for i in range(0, rows, 16)])
    assert torch.isfinite(got).all() and torch.isfinite(want).all()
    assert torch.equal(got, want)
    one.close()
    many.close()


@pytest.mark.parametrize("rows", [1344, 1361, 1777, 2033])
def test_expert_tiles_of_eight_blocks_equal_block_by_block(ctx, rows):
    """128 experts of 84 rows on average (the last count with tiles of four blocks), 85, 111 and 127 (tiles of five to eight)."""
    test_many_row_prefill_equals_block_by_block(ctx, "experts128", rows)


@pytest.mark.parametrize("hidden,n_expert,used,rows", [(512, 72, 3, 832), (512, 72, 3, 850), (2048, 200, 1, 321), (256, 129, 2, 530)])
def test_routers_of_many_rows_equal_block_by_block(ctx, hidden, n_expert, used, rows):
    """Routers whose last workgroup of 64 weight rows has eight of them or one, one to four steps of K a wave or none for some waves, row
    counts from the first that takes them, a last block of two rows and of one; slots of one, two and three picks a row."""
    SHAPES["router"] = (dfl.ModelConfig(n_layers=2, hidden=hidden, n_q=4, n_kv=2, head_dim=128, ffn=0, vocab=2048, n_expert=n_expert,
                                        n_expert_used=used, ffn_expert=256, ffn_shared=256), dfl.synth.Q6_K)
    test_many_row_prefill_equals_block_by_block(ctx, "router", rows)


@pytest.mark.parametrize("rows", [17, 192, 200, 530])
def test_a_mixture_with_q4k_projections_equals_block_by_block(ctx, rows):
    """Its output projection's minima go by sums made ahead of the product: past held weights up to their last count, and split."""
    test_many_row_prefill_equals_block_by_block(ctx, "experts_q4k", rows)


_STREAMED_PROBE = r"""
import sys
sys.path.insert(0, "tests")
import qwen_llm_amd as dfl
import test_gpu_prefill_rows as t
ctx = dfl.Context(0, workspace_bytes=256 << 20)
for rows in (40, 530):
    t.test_many_row_prefill_equals_block_by_block(ctx, "experts_q4k", rows)
print("equal")
"""


def test_a_mixture_whose_projections_stream_equals_block_by_block():
    """Without the whole-K kernels every Q4_K projection goes by sums: the first layer's q|k|v by the norm kernel's, the later
    ones', which the experts' last kernel has normalised, by sums made ahead of the product.  (The switch is read once per
    process.)"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=root + os.pathsep + os.environ.get("PYTHONPATH", ""), DFLASH_GEMM_WHOLE="0")
    r = subprocess.run([sys.executable, "-c", _STREAMED_PROBE], env=env, cwd=root, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.split()[-1] == "equal", r.stderr[-2000:]


@pytest.mark.parametrize("shape", ["narrow", "experts", "heads64"])
def test_a_prepared_session_allocates_nothing_for_its_first_prompt(ctx, shape):
    """dflash_prefill_prepare makes what the first prompt needs: a group's buffers, or the lanes of a shape (heads64: K and
    V rows of half a tile group) that the grouped pass cannot take."""
    cfg, attn_type = SHAPES[shape]
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type))
    for i in range(2):  # (the first session has the runtime load the kernels, which takes memory of its own)
        sess = dfl.Session(ctx, model, 160, [0, 1])
        sess.prepare_prefill()
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        sess.prefill_blocks(list(range(130)), 0, want_hidden=False)
        torch.cuda.synchronize()
        taken = free - torch.cuda.mem_get_info()[0]
        sess.close()
    assert taken == 0


@pytest.mark.parametrize("head", [0, 37])
@pytest.mark.parametrize("taps", [[0], [0, 1]], ids=["last layer not tapped", "tapped"])
@pytest.mark.parametrize("shape,adjacent,rows", [("experts", True, 1), ("experts", True, 16), ("experts", True, 17), ("experts", True, 300), ("experts", True, 2050),
                                                 ("experts", True, 2070), ("wide", True, 33), ("narrow", True, 130), ("narrow", False, 70), ("heads64", True, 500)])
def test_a_prompt_in_one_call_equals_its_blocks_and_their_last_one(ctx, shape, adjacent, rows, taps, head):
    """Hidden rows, the argmax behind the last token, and what a block behind the prompt computes from its K/V rows: a prompt of one block, of a few, of
    a group and a rest of a block or of more, and a target that has no groups (separate projections: its blocks go by lanes)."""
    cfg, attn_type = SHAPES[shape]
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type), adjacent=adjacent)
    two, one = dfl.Session(ctx, model, head + rows + 32, taps), dfl.Session(ctx, model, head + rows + 32, taps)
    tokens = np.random.default_rng(rows).integers(0, cfg.vocab, head + rows).tolist()
    if head:
        for s in (two, one):
            s.prefill_blocks(tokens[:head], 0, want_hidden=False)
    body = head + (rows - 1) // 16 * 16
    want = [two.prefill_blocks(tokens[head:body], head)] if body > head else []
    last = two.encode_packed_verify_layer_major(tokens[body:], body)
    got, token = one.prefill_prompt(tokens[head:], head)
    assert torch.equal(got, torch.cat(want + [last.hidden_capture])) and token == last.argmax_host[-1]
    assert one.kv_n_pos == two.kv_n_pos == head + rows
    a, b = (s.encode_packed_verify_layer_major([token, 3, 5], head + rows, want_logits=True) for s in (two, one))
    assert torch.equal(a.logits, b.logits)
    two.close()
    one.close()


@pytest.mark.parametrize("shape,rows,head", [("experts", 2303, 0), ("experts", 2304, 0), ("narrow", 3011, 0), ("narrow", 4361, 0), ("wide", 2310, 0),
                                             ("wide", 2505, 37)])
def test_prompts_of_several_passes_equal_block_by_block(ctx, shape, rows, head):
    """More rows than a pass holds (2048): a full pass and a rest, full passes and a rest, two passes of the same size (the wide shape, from position
    0 and behind a context), in both calls."""
    test_continued_prefill_equals_block_by_block(ctx, shape, head, rows)
    test_a_prompt_in_one_call_equals_its_blocks_and_their_last_one(ctx, shape, True, rows, [0], head)


def test_a_prompt_in_one_call_keeps_the_guards(ctx):
    cfg, attn_type = SHAPES["narrow"]
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type))
    sess = dfl.Session(ctx, model, 64, [0])
    for tokens, start, status in (([1, 2], 5, 10), ([1, cfg.vocab], 0, 8), ([1] * 65, 0, 10), ([], 0, 1)):
        with pytest.raises(dfl.DFlashError) as e:
            sess.prefill_prompt(tokens, start)
        assert e.value.status == status and sess.kv_n_pos == 0
    sess.close()


@pytest.mark.parametrize("first", [0, 7])
def test_context_columns_appended_at_once_equal_columns_in_blocks(ctx, first):
    """More than sixteen columns of consecutive positions: from zero (the mirror's case) and off it."""
    cfg = dfl.ModelConfig(n_layers=1, hidden=512, n_q=4, n_kv=2, head_dim=64, ffn=512, vocab=1024)
    dcfg = dfl.DraftConfig(n_layers=2, hidden=512, n_q=4, n_kv=2, head_dim=64, ffn=512, block_size=8, n_taps=2)
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda"))
    drafter = dfl.DraftHead(ctx, dcfg, dfl.synth_draft_weights_device(dcfg, 6, "cuda", vocab=cfg.vocab))
    cols = torch.randn((45, 2, 512), generator=torch.Generator(device="cuda").manual_seed(3), device="cuda")
    out = []
    for step in (16, 45):
        d = dfl.DraftSession(ctx, drafter, model, 64)
        for i in range(0, 45, step):
            d.append_target_ctx_columns(cols[i:i + step], list(range(first + i, first + min(i + step, 45))))
        out.append(d.draft_block(5, cfg.vocab - 1, first + 45, want_logits=True)[1].clone())
        d.close()
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("start", [0, 17, 31, 63, 260, 520, 569])
@pytest.mark.parametrize("shape", ["narrow", "experts", "heads64", "heads64x12", "heads256x1", "heads256x12"])
def test_a_lone_block_rotates_its_rows_as_a_group_does(ctx, shape, start):
    """A lone block's attention norms and rotates its rows itself and puts its keys and values over the cache's (groups of at most
    eight heads); a group's rows have a launch of their own: the same bits, of every number of rows, where the rows fall into one
    stage of keys, two, or the splits of two workgroups, and where the next block reads what they left in the cache.  (Starts with
    64 positions behind them whose splits are of one policy, that of their bucket of context lengths.)"""
    cfg, attn_type = SHAPES[shape]
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 5, "cuda", attn_type=attn_type))
    tokens = np.random.default_rng(start).integers(0, cfg.vocab, start + 64).tolist()
    one, many = dfl.Session(ctx, model, start + 80, [0, 1]), dfl.Session(ctx, model, start + 80, [0, 1])
    for s in (one, many) if start else ():
        s.prefill_blocks(tokens[:start], 0)
    want = many.prefill_blocks(tokens[start:], start)
    at = start
    for n in (1, 16, 5, 11, 2, 16):
        got = one.encode_packed_verify_layer_major(tokens[at:at + n], at).hidden_capture
        assert torch.equal(got, want[at - start:at - start + n]), (at, n)
        at += n
    one.close()
    many.close()
