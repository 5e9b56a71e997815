"""Projection GEMM forms at the edges of their tiles, against the oracle.

Each case evaluates B one-token sequences in one pass: every projection and
the head multiply B rows, and every row's logits come back. A one-token
sequence attends to itself only, so the oracle evaluates each id once.
"""
import numpy as np
import pytest

from esp_amd import DecoderConfig, DecoderModel
from oracle import oracle, quant, st
from tests import synth

pytestmark = pytest.mark.gpu


def _rows_match(model, ref, vocab, rows, tol):
    ids = synth.uniform_ids(rows * 7 + 1, rows, min(vocab, 24))  # few ids: few oracle passes
    kv = model.new_cache(rows, 4)
    got = model.forward_batch(kv, list(range(rows)), [[t] for t in ids])
    want = {t: ref.forward_last(ref.new_cache(), [t]) for t in set(ids)}
    for r, t in enumerate(ids):
        scale = float(np.abs(want[t]).max())
        err = float(np.abs(got[r] - want[t]).max())
        assert err <= tol * scale, f"row {r} of {rows}: {err} vs scale {scale}"


# K of 16-key stages: one stage short of a power of two, k splits (K >= 512),
# a ragged last split (1040 = 2 x 520), and 72, which keeps the vector form
@pytest.mark.parametrize("hidden,ffn", [(48, 80), (64, 72), (512, 1040)])
@pytest.mark.parametrize("rows", [2, 31, 32, 33, 64, 65, 129, 513])
def test_f32_rows(hidden, ffn, rows):
    """f32 products and sums: the f32 contract's 1e-4 of the row's magnitude
    (K 2^-24 is 6e-5 at K 1040 if every rounding went the same way)."""
    print(f"f32 rows {rows} hidden {hidden} ffn {ffn}", flush=True)
    cfg, tensors, blob, _ = synth.tiny_llama_case(seed=5, layers=2, hidden=hidden, heads=hidden // 16,
                                                  kv_heads=hidden // 16, ffn=ffn, vocab=131, prompt_len=2)
    _rows_match(DecoderModel.from_bytes(cfg, blob, "f32"), oracle.OracleModel(cfg, tensors), 131, rows, 1e-4)


# 128-row tiles: gate/up and the head (K 64, 116 rows in the last tile), and
# down_proj in eight k splits (640 keys, one row in the last tile)
@pytest.mark.parametrize("hidden,ffn,vocab,rows", [(64, 4096, 8192, 500), (1280, 5120, 131, 257)])
def test_f32_128_row_tiles(hidden, ffn, vocab, rows):
    """The f32 tile of 128 x 128, which wide products of many rows take: 1e-4 of
    the row's magnitude, as above."""
    print(f"f32 128-row tiles hidden {hidden} ffn {ffn} rows {rows}", flush=True)
    cfg, tensors, blob, _ = synth.tiny_llama_case(seed=6, layers=1, hidden=hidden, heads=hidden // 16,
                                                  kv_heads=hidden // 16, ffn=ffn, vocab=vocab, prompt_len=2)
    _rows_match(DecoderModel.from_bytes(cfg, blob, "f32"), oracle.OracleModel(cfg, tensors), vocab, rows, 1e-4)


# q/k/v in four k splits, which the rotary pass adds up (head_dim 64 and 128)
@pytest.mark.parametrize("arch,head_dim", [("llama", 64), ("qwen2", 128), ("qwen2", 64), ("qwen3", 128)])
@pytest.mark.parametrize("lens", [(2, 5), (9, 17, 14), (60, 70)])
def test_f32_split_qkv_rows(arch, head_dim, lens):
    """f32 models whose q/k/v sums reach the rotary pass as k splits, with the
    q/k/v bias (qwen2) and the per-head q/k norm (qwen3): several sequences'
    blocks, so that every query reads other rows' keys; 1e-4 of the row's
    magnitude."""
    print(f"f32 split q/k/v {arch} hd {head_dim} blocks {lens}", flush=True)
    names = {"llama": "LlamaForCausalLM", "qwen2": "Qwen2ForCausalLM", "qwen3": "Qwen3ForCausalLM"}
    cfg = synth.llama_config(2, 1024, 1024 // head_dim, 4, 1024, 131, head_dim=head_dim,
                             extra={"architectures": [names[arch]], "model_type": arch})
    assert cfg.qkv_bias() == (arch == "qwen2") and cfg.qk_norm() == (arch == "qwen3")
    tensors = synth.make_tensors(cfg, 4, "f32", std=0.05, bias_std=0.5)
    for name in tensors:  # weights of the per-head norms, which are 1 otherwise
        if name.endswith(("q_norm.weight", "k_norm.weight")):
            tensors[name][0][:] = 1 + synth.normal(synth.tensor_seed(4, name), head_dim, 0.3)
    model, ref = DecoderModel.from_bytes(cfg, st.dump(tensors), "f32"), oracle.OracleModel(cfg, tensors)
    blocks = [synth.uniform_ids(3 + i, n, 131) for i, n in enumerate(lens)]
    got = model.forward_batch(model.new_cache(len(lens), max(lens)), list(range(len(lens))), blocks)
    for r, b in enumerate(blocks):
        want = ref.forward_last(ref.new_cache(), b)
        err = float(np.abs(got[r] - want).max())
        assert err <= 1e-4 * float(np.abs(want).max()), f"sequence {r} of {lens}: {err}"


# K 128 (one group of keys), 192 (no whole groups: tiles at any row count), 256,
# 512, 640, and 1408 in ragged k splits
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("hidden,ffn", [(128, 192), (256, 640), (512, 1408)])
@pytest.mark.parametrize("rows", [2, 31, 32, 33, 64, 65, 129, 300])
def test_packed_rows(bits, hidden, ffn, rows):
    """Packed projections and head over several rows: 1e-4 of the row's
    magnitude (activations as two bf16 halves, 2^-17 a product)."""
    print(f"q{bits} rows {rows} hidden {hidden} ffn {ffn}", flush=True)
    cfg = synth.llama_config(2, hidden, 4, 2, ffn, 131, head_dim=32 if hidden < 512 else 64)
    tensors = synth.make_tensors(cfg, 9, "f32", std=0.05)
    art = quant.convert_artifact(tensors, bits)
    shapes = {n: a.shape for n, (a, _) in tensors.items()}
    ref = oracle.OracleModel(cfg, quant.dequantized_model(art, shapes, bits))
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(art), f"q{bits}-block32"), ref, 131, rows, 1e-4)


# gate/up of 16384 columns fill two blocks per CU with two k splits, of 640 keys:
# the resident 512 (16 rows) or 256 are refilled, the last time in part
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows", [2, 16, 32, 64])
def test_packed_rows_refill_their_activations(bits, rows):
    """Packed products whose k range is longer than the resident activations:
    1e-4 of the row's magnitude."""
    print(f"q{bits} refill rows {rows}", flush=True)
    cfg = synth.llama_config(1, 1280, 10, 2, 16384, 131, head_dim=128)
    tensors = synth.make_tensors(cfg, 9, "f32", std=0.02, fast=True)
    art = quant.convert_artifact(tensors, bits)
    ref = oracle.OracleModel(cfg, quant.dequantized_model(art, {n: a.shape for n, (a, _) in tensors.items()}, bits))
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(art), f"q{bits}-block32"), ref, 131, rows, 1e-4)


# every form of the packed head: 16, 32 and 64 resident rows, tiles above; a K
# without whole 128-key groups (tiles only); 65500 columns fill the chip without
# k splits, so that the 256 (9 rows) or 128 resident keys are refilled
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("hidden,rows,vocab", [(2048, 2, 515), (2048, 17, 515), (2048, 64, 515), (2048, 131, 515),
                                               (1088, 5, 515), (640, 9, 65500), (640, 20, 65500)])
def test_packed_head_keeps_f32_activations(bits, hidden, rows, vocab):
    """The packed head of several sequences against 64 bits, on hidden states
    that are the embeddings (zero output projections): 6e-7 of the logits,
    which f32 operands and sums over K / 32 blocks keep (about 2e-7) and
    activations of two bf16 halves do not (2.3e-6 at any K)."""
    print(f"packed head q{bits} K {hidden} rows {rows}", flush=True)
    cfg = synth.llama_config(1, hidden, 2, 2, 64, vocab, head_dim=32)
    tensors = synth.make_tensors(cfg, 9, "f32", std=0.05, fast=vocab > 60000)
    for name in ("self_attn.o_proj", "mlp.down_proj"):
        tensors[f"model.layers.0.{name}.weight"][0][:] = 0
    art = quant.convert_artifact(tensors, bits)
    deq = quant.dequantized_model(art, {n: a.shape for n, (a, _) in tensors.items()}, bits)
    model = DecoderModel.from_bytes(cfg, st.dump(art), f"q{bits}-block32")
    ids = synth.uniform_ids(rows, rows, vocab)
    x = np.asarray(deq["model.embed_tokens.weight"][0], np.float64)[ids]
    x = x / np.sqrt((x * x).mean(1, keepdims=True) + 1e-5) * np.asarray(deq["model.norm.weight"][0], np.float64)
    want = x @ np.asarray(deq["lm_head.weight"][0], np.float64).T
    got = model.forward_batch(model.new_cache(rows, 4), list(range(rows)), [[t] for t in ids])
    one = model.try_forward_cached_last([ids[0]], model.new_cache(1, 4))
    rel = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert rel <= 6e-7, rel
    assert np.linalg.norm(one - want[0]) <= 6e-7 * np.linalg.norm(want[0])


# 16, 32 and 64 resident rows and tiles, with k splits (hidden 512, ffn 1408)
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("rows", [2, 17, 40, 70])
def test_packed_products_keep_the_f32_range(bits, rows):
    """Values and gated units around 5e36 (up to 6e37) into o_proj and down_proj
    weights around 5e-37: 32 integers times them leave the range of f32, times
    the block's scale they do not. The outputs are the dequantized weights' own
    (1e-4 of the row's magnitude, as in range)."""
    print(f"packed range q{bits} rows {rows}", flush=True)
    cfg = synth.llama_config(1, 512, 8, 4, 1408, 131, head_dim=64)
    tensors = synth.make_tensors(cfg, 9, "f32", std=0.05)
    for name, s in (("self_attn.v_proj", 4e36), ("self_attn.o_proj", 1e-35), ("mlp.up_proj", 4e36),
                    ("mlp.down_proj", 1e-35)):
        tensors[f"model.layers.0.{name}.weight"][0][:] *= np.float32(s)
    art = quant.convert_artifact(tensors, bits)
    ref = oracle.OracleModel(cfg, quant.dequantized_model(art, {n: a.shape for n, (a, _) in tensors.items()}, bits))
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(art), f"q{bits}-block32"), ref, 131, rows, 1e-4)


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("lens", [(16, 128, 129), (257, 16, 31, 400), (1100, 20), (2050, 2049, 40)])
def test_prompt_blocks_in_one_launch(kv, lens):
    """Several sequences' prompt blocks of 16 rows or more attend in one launch
    (edges of 128-row query blocks and their pairs; the last case crosses a
    4096-row chunk): each sequence's logits are those of its prompt alone,
    whose projections split K elsewhere, within the bf16 path's rounding."""
    print(f"prompt blocks {lens} {kv}", flush=True)
    cfg = synth.llama_config(2, 256, 4, 2, 512, 300, head_dim=64, max_pos=4096)
    model = DecoderModel.synthetic(cfg, seed=3, std=0.05, fmt="bf16")
    blocks = [synth.uniform_ids(11 + i, n, 300) for i, n in enumerate(lens)]
    cache = model.new_cache(len(lens), max(lens) + 1, kv)
    got = model.forward_batch(cache, list(range(len(lens))), blocks)
    one = model.new_cache(1, max(lens) + 1, kv)
    tol = 1e-4 if kv == "f32" else 2e-3  # a half-precision cache rounds other last bits
    for r, b in enumerate(blocks):
        one.reset(0)
        want = model.try_forward_cached_last(b, one)
        err = float(np.abs(got[r] - want).max())
        assert err <= tol * float(np.abs(want).max()), f"sequence {r} of {lens}: {err}"


# The narrow shapes take the few-row form for gate/up only (K 128, 256 and 512:
# its k ranges are a group or two); hidden 4224 takes it everywhere (33, 55 and
# more column blocks with k splits, more than one round of 256 CUs).
@pytest.mark.parametrize("hidden,ffn,heads,kv_heads", [(128, 256, 4, 2), (256, 640, 8, 2), (512, 1152, 8, 2),
                                                       (4224, 2048, 33, 11)])
@pytest.mark.parametrize("rows", [2, 4, 5, 8, 9, 15, 16])
def test_bf16_few_rows(hidden, ffn, heads, kv_heads, rows):
    """bf16 weights over few rows, on both sides of the few-row form's ends
    (15 rows, one round of blocks): 1e-4 of the row's magnitude (activations
    as two bf16 halves)."""
    print(f"bf16 rows {rows} hidden {hidden} ffn {ffn}", flush=True)
    wide = hidden > 4000
    cfg = synth.llama_config(1 if wide else 2, hidden, heads, kv_heads, ffn, 131, head_dim=hidden // heads)
    tensors = synth.make_tensors(cfg, 9, "bf16", std=0.02 if wide else 0.05, fast=wide)
    ref = oracle.OracleModel(cfg, tensors)
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(tensors), "bf16"), ref, 131, rows, 1e-4)


# a head of 65500 columns fills two blocks per CU without k splits, so each row
# form's resident keys (4 rows: 2048, 8: 1024, 16: 512) are refilled, with 128
@pytest.mark.parametrize("hidden,rows", [(2176, 2), (2176, 4), (1152, 5), (1152, 8), (640, 9), (640, 15)])
def test_bf16_few_rows_refill_their_activations(hidden, rows):
    """The few-row form over a k range longer than its resident activations:
    1e-4 of the row's magnitude."""
    print(f"bf16 refill rows {rows} K {hidden}", flush=True)
    cfg = synth.llama_config(1, hidden, hidden // 64, hidden // 64, 256, 65500, head_dim=64,
                             extra={"tie_word_embeddings": True})
    tensors = synth.make_tensors(cfg, 9, "bf16", std=0.05, fast=True)
    ref = oracle.OracleModel(cfg, tensors)
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(tensors), "bf16"), ref, 65500, rows, 1e-4)


# rows per expert on average: 1, 3, 8, 20, 48 and past each
@pytest.mark.parametrize("rows", [2, 6, 7, 16, 17, 40, 42, 96, 100])
def test_bf16_moe_rows(rows):
    """Routed experts over few rows: grouped few-row products whose tiles end
    inside and between the experts' rows, read through the router's grouping."""
    print(f"moe rows {rows}", flush=True)
    cfg = DecoderConfig.mixtral_style(vocab_size=131, hidden_size=256, intermediate_size=384,
                                      num_hidden_layers=2, num_attention_heads=4, num_key_value_heads=2,
                                      max_position_embeddings=64, num_experts=4, num_experts_per_tok=2,
                                      moe_intermediate_size=384)
    tensors = synth.make_tensors(cfg, 9, "bf16", std=0.05)
    ref = oracle.OracleModel(cfg, tensors)
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(tensors), "bf16"), ref, 131, rows, 1e-4)


@pytest.mark.parametrize("fmt", ["bf16", "f32"])
@pytest.mark.parametrize("rows", [2, 7, 40])
def test_moe_combine_norm_rows(fmt, rows):
    """The combine joined with the next layer's norm: an odd number of experts
    per token, outputs that come as split sums (K 1024 in up to four)."""
    print(f"moe combine {fmt} rows {rows}", flush=True)
    cfg = DecoderConfig.mixtral_style(vocab_size=131, hidden_size=256, intermediate_size=1024,
                                      num_hidden_layers=3, num_attention_heads=4, num_key_value_heads=2,
                                      max_position_embeddings=64, num_experts=5, num_experts_per_tok=3,
                                      moe_intermediate_size=1024)
    tensors = synth.make_tensors(cfg, 11, fmt, std=0.05)
    ref = oracle.OracleModel(cfg, tensors)
    _rows_match(DecoderModel.from_bytes(cfg, st.dump(tensors), fmt), ref, 131, rows, 1e-4)
