"""The wide gate | up product of a dense layer as one launch (csrc/gemm_dense.hip): a one-layer decoder against the oracle, and a
prompt's rows against their own blocks bit for bit.

A unit is sixteen columns; what is left over when each of 256 workgroups has as many units is cut into 16, 8, 4 or 2 parts by weight rows, or not
at all.  The shapes bring each cut, none left over, two rounds of units, and K whose last chunk of four super-blocks is not full."""
import numpy as np
import pytest
import torch

import qwen_llm_amd as dfl

pytestmark = pytest.mark.gpu

SHAPES = [(2304, 4352), (2304, 4608), (2304, 5120), (2304, 6144), (2560, 7168), (2304, 8192), (1280, 12544), (1280, 28928)]


@pytest.fixture(scope="module")
def ctx():
    c = dfl.Context(0, workspace_bytes=256 << 20)
    yield c
    c.close()


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
        got = one.encode_packed_verify_layer_major(tokens[at:at + n], at).hidden_capture
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
