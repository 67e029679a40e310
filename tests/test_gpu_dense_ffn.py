"""The wide gate | up product of a dense layer as one launch (csrc/gemm_dense.hip): a one-layer decoder against the oracle, and a
prompt's rows against their own blocks bit for bit.

A unit is sixteen columns; what is left over when each of 256 workgroups has as many units is cut into 16, 8, 4 or 2 parts by weight rows, or not
at all.  The shapes bring each cut, none left over, two rounds of units, K whose last chunk of four super-blocks is not full, and K of up to
32 super-blocks, the most that a norm leaves in fragment order.  Each is one that the launch takes: of the layer's products only down has a
reduction then."""
import numpy as np
import pytest
import torch

import qwen_llm_amd as dfl

pytestmark = pytest.mark.gpu

SHAPES = [(2304, 4352), (2304, 4608), (2304, 5120), (2304, 6144), (2560, 7168), (2304, 8192), (1280, 12544), (1280, 28928), (5120, 4608), (8192, 4608)]


@pytest.fixture(scope="module")
def ctx():
    c = dfl.Context(0, workspace_bytes=256 << 20)
    yield c
    c.close()


def verified(ctx, sess, tokens, at):
    """The tapped rows of a block, and how many of its products were followed by a reduction."""
    ctx.set_kernel_timing(1)
    out = sess.encode_packed_verify_layer_major(tokens, at, want_head=False)
    n = ctx.kernel_timing(ctx.T_REDUCE)[1]
    ctx.set_kernel_timing(0)
    return out.hidden_capture, n


@pytest.mark.parametrize("hidden,ffn", SHAPES)
def test_wide_ffn_matches_oracle_and_the_prompts_rows(ctx, oracle, hidden, ffn):
    cfg = dfl.ModelConfig(n_layers=1, hidden=hidden, n_q=4, n_kv=2, head_dim=128, ffn=ffn, vocab=512)
    w = dfl.synth_target_weights_blocks(cfg, 23)
    model = dfl.TargetModel(ctx, cfg, w)
    omodel, _keep = oracle.build_model(cfg.as_dict(), w)
    one, many = dfl.Session(ctx, model, 64, [0]), dfl.Session(ctx, model, 64, [0])
    ostate = oracle.TargetState(cfg.as_dict(), 64)
    tokens = np.random.default_rng(ffn).integers(0, cfg.vocab, 40).tolist()
    rows = []
    for at, n in ((0, 16), (16, 16), (32, 1), (33, 7)):
        got, reductions = verified(ctx, one, tokens[at:at + n], at)
        assert reductions == 1
        _, want = oracle.target_verify(omodel, ostate, tokens[at:at + n], at, [0])
        rows.append(got)
        # f16 operands (2^-11) in the six products that a row passes through: 5e-3 in the 2-norm, 3e-2 in an element (as for whole stacks)
        d = got.cpu().numpy().astype(np.float64) - want
        rms = np.sqrt(np.mean(np.square(want, dtype=np.float64)))
        assert np.linalg.norm(d) / np.linalg.norm(want) <= 5e-3
        assert np.max(np.abs(d) / np.maximum(np.abs(want), rms)) <= 3e-2
    got = many.prefill_blocks(tokens, 0)
    assert torch.equal(got, torch.cat(rows))
    one.close()
    many.close()


@pytest.mark.parametrize("hidden,ffn", [(2304, 4608), (2560, 9728), (5120, 4608)])
def test_one_launch_is_as_near_the_oracle_as_separate_products(ctx, oracle, hidden, ffn):
    """One f32 sum over K in place of several that are added, of the same f16 operands, and silu(gate) * up held in the f16 that down rounds it to:
    what differs is f32 rounding, 2^-24 a step, next to the operands' 2^-11 that both have: their errors agree to a percent."""
    cfg = dfl.ModelConfig(n_layers=1, hidden=hidden, n_q=4, n_kv=2, head_dim=128, ffn=ffn, vocab=512)
    w = dfl.synth_target_weights_blocks(cfg, 37)
    omodel, _keep = oracle.build_model(cfg.as_dict(), w)
    tokens = np.random.default_rng(ffn).integers(0, cfg.vocab, 16).tolist()
    _, want = oracle.target_verify(omodel, oracle.TargetState(cfg.as_dict(), 64), tokens, 0, [0])
    errors, model = [], dfl.TargetModel(ctx, cfg, w)
    up = ctx.repack_q4k_tiled(torch.from_numpy(w["layers"][0]["up"][1]).cuda(), hidden, ffn)
    for one_launch in (True, False):
        if not one_launch:  # up somewhere else than behind gate
            model.c.layers[0].up.data = up.data_ptr()
        sess = dfl.Session(ctx, model, 64, [0])
        got, reductions = verified(ctx, sess, tokens, 0)
        assert (reductions == 1) == one_launch
        errors.append(np.linalg.norm(got.cpu().numpy().astype(np.float64) - want))
        sess.close()
    assert errors[0] <= 1.01 * errors[1], errors


@pytest.mark.parametrize("adjacent", [True, False], ids=["one launch", "separate products"])
@pytest.mark.parametrize("tiled", [True, False], ids=["tiled", "row order"])
@pytest.mark.parametrize("hidden,ffn", [(2304, 4608), (1280, 8192)])
def test_down_in_q6k_behind_rows_in_row_order(ctx, oracle, hidden, ffn, tiled, adjacent):
    """A Q6_K down projection in both orders behind a gate | up that leaves its rows in row order (the one launch, as f16; separate products, as
    f32): blocks, a prompt's rows and a prompt in one call.  Only fragment-order rows go through the tiled order, so a block packs them."""
    cfg = dfl.ModelConfig(n_layers=2, hidden=hidden, n_q=4, n_kv=2, head_dim=128, ffn=ffn, vocab=512)
    w, rng = dfl.synth_target_weights_blocks(cfg, 29), np.random.default_rng(31)
    for layer in w["layers"]:
        layer["down"] = (dfl.TYPE_Q6_K, dfl.synth.random_blocks_scaled(dfl.TYPE_Q6_K, hidden, ffn, ffn ** -0.5, rng))
    model = dfl.TargetModel(ctx, cfg, w, adjacent=adjacent)
    tensors = []
    for il, layer in enumerate(w["layers"] if tiled else ()):
        assert ctx.xf_kind(dfl.TYPE_Q6_K_TILED, ffn, hidden) == dfl.XF_Q6K
        tensors.append(ctx.repack_q6k_tiled(torch.from_numpy(layer["down"][1]).cuda(), ffn, hidden))
        model.c.layers[il].down = type(model.c.layers[il].down)(dfl.TYPE_Q6_K_TILED, model.c.layers[il].down.flags, tensors[-1].data_ptr())
    omodel, _keep = oracle.build_model(cfg.as_dict(), w)
    one, many, prompt = (dfl.Session(ctx, model, 64, [0, 1]) for _ in range(3))
    ostate = oracle.TargetState(cfg.as_dict(), 64)
    tokens = np.random.default_rng(ffn).integers(0, cfg.vocab, 40).tolist()
    rows = []
    for at, n in ((0, 16), (16, 16), (32, 1), (33, 7)):
        out = one.encode_packed_verify_layer_major(tokens[at:at + n], at)
        _, want = oracle.target_verify(omodel, ostate, tokens[at:at + n], at, [0, 1])
        rows.append(out.hidden_capture)
        # (as above, two layers of it)
        d = rows[-1].cpu().numpy().astype(np.float64) - want
        rms = np.sqrt(np.mean(np.square(want, dtype=np.float64)))
        assert np.linalg.norm(d) / np.linalg.norm(want) <= 5e-3
        assert np.max(np.abs(d) / np.maximum(np.abs(want), rms)) <= 3e-2
    assert torch.equal(many.prefill_blocks(tokens, 0), torch.cat(rows))
    hidden_rows, last = prompt.prefill_prompt(tokens, 0)
    assert torch.equal(hidden_rows, torch.cat(rows)) and last == out.argmax_host[-1]
    for s in (one, many, prompt):
        s.close()


def test_misaligned_weights_are_refused(ctx):
    """Tiled Q4_K off 128 bytes is refused, as by every other kernel that reads that order, and the session goes on where it was."""
    cfg = dfl.ModelConfig(n_layers=1, hidden=1280, n_q=4, n_kv=2, head_dim=128, ffn=12544, vocab=512)
    model = dfl.TargetModel(ctx, cfg, dfl.synth_target_weights_device(cfg, 23, "cuda"))
    sess = dfl.Session(ctx, model, 64, [0])
    layer = model.c.layers[0]
    at = layer.gate.data, layer.up.data
    layer.gate.data, layer.up.data = at[0] + 64, at[1] + 64
    with pytest.raises(dfl.DFlashError) as e:
        sess.encode_packed_verify_layer_major([1, 2, 3], 0)
    assert e.value.status == 4 and sess.kv_n_pos == 0
    layer.gate.data, layer.up.data = at
    sess.encode_packed_verify_layer_major([1, 2, 3], 0)
    sess.close()
