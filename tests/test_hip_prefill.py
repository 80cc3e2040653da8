"""Batched MFMA prefill (kernels/prefill.h) == the same prompt fed as single-position passes (the decode kernels,
which are parity-green against the oracle), and == the oracle directly on the fixtures.  Size-independent property at
real layer shapes: prefill(S) then decode == step-by-step, KV cache contents equal up to bf16 rounding flips."""
import copy

import numpy as np
import pytest

from conftest import GPU_FAMILIES, load_golden, rel_err
from tinygpt_amd import known_desc, synth
from tinygpt_amd.desc import desc_from_hf_config
from tinygpt_amd.ffi import GREEDY, Model, product_backend

pytestmark = pytest.mark.gpu


def run(model, prompt, mfma, n_decode=4):
    model.reset_cache()
    model.set_option("prefill.mfma", int(mfma))
    model.forward(prompt)
    logits = model.logits(rounded=False).copy()
    first = model.sample(GREEDY).copy()
    rest = model.decode(n_decode, GREEDY).copy()
    kv = [model.read_kv(0, l) for l in range(model.desc.layers)]
    return logits, first, rest, kv


@pytest.mark.parametrize("fam", GPU_FAMILIES)
@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp32"])
def test_fixture_prefill_matches_steps_and_oracle(fam, dtype, oracle_lib):
    """Every family incl. GPT-2 (LayerNorm-split prologue, bias + gelu_new epilogue, learned positions) and every storage dtype: 16-bit
    storage runs the split-term bf16 / f16 MFMA GEMMs, fp32 storage the f32-input MFMA GEMMs (kernels/gemm_f32.h) with the decode
    attention kernel over the prompt rows."""
    from oracle.oracle_ffi import OracleModel
    cfg, g = load_golden(fam)
    d = desc_from_hf_config(cfg, dtype)
    gpu = Model(d, product_backend()).load_synthetic(int(g["seed"]), float(g["std"])).finalize()
    ref = OracleModel(d).load_synthetic(int(g["seed"]), float(g["std"])).finalize()
    # a longer prompt than the golden one so that M is not a tile multiple and causal masking crosses a key tile
    prompt = synth.synth_prompt(d.vocab, min(d.max_ctx - 8, 97), 5)[None, :]
    l1, f1, r1, kv1 = run(gpu, prompt, mfma=True)
    l0, f0, r0, kv0 = run(gpu, prompt, mfma=False)
    ref.forward(prompt)
    lr = ref.logits(rounded=False)
    assert rel_err(l1, lr) < 1e-3 and rel_err(l0, lr) < 1e-3
    assert rel_err(l1, l0) < 1e-3          # same contract bound; the two schedules differ by bf16 KV rounding flips
    np.testing.assert_array_equal(f1, f0)
    np.testing.assert_array_equal(f1, ref.sample(GREEDY))
    np.testing.assert_array_equal(r1, r0)
    ulp = {"bf16": 8e-3, "fp16": 1e-3, "fp32": 1e-5}[dtype]
    for (k1, v1), (k0, v0) in zip(kv1, kv0):
        # cache entries of the two schedules: equal to within one storage ulp of the tensor's magnitude (the split
        # MFMA products are exact to ~2^-17 (bf16 x2) / 2^-22 (fp16 x2) of |x||w|, so near-zero elements may round differently)
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp
    if dtype == "fp32":                      # fp32 storage: both schedules sit on the oracle (and on HF fp32) to fp32 summation order
        assert rel_err(l1, lr) < 1e-4 and rel_err(l1, l0) < 1e-4


@pytest.mark.parametrize("name,S,dtype", [("llama-3.2-1b", 300, "bf16"), ("mistral-7b-v0.3", 130, "bf16"), ("qwen2.5-0.5b", 257, "bf16"),
                                          ("llama-3.2-1b", 300, "fp16"), ("mistral-7b-v0.3", 130, "fp16"),
                                          ("qwen2.5-3b", 200, "bf16"), ("qwen3-1.7b", 150, "bf16"),   # the README's other checkpoints: 8 query heads per kv head; q/k norm
                                          ("gpt2", 300, "bf16"), ("gpt2", 300, "fp16"), ("gpt2", 300, "fp32"),           # BASELINE configs[0]'s model
                                          ("llama-3.2-1b", 300, "fp32"), ("mistral-7b-v0.3", 130, "fp32"), ("qwen2.5-0.5b", 257, "fp32"), ("qwen3-1.7b", 90, "fp32"),
                                          # the long-prompt forms of round 5 at the shapes their A / B tests used (those compared new against old bit for bit through option
                                          # switches that are gone): gate_up on whole 128-byte lines, the QKV product on shared activation lines with RoPE /
                                          # cache append / q split in its epilogue (also with a QKV bias, ADVICE r5, and a ragged last row block), `down` as one slab
                                          ("llama-3.2-1b", 1024, "bf16"), ("llama-3.2-1b", 1900, "bf16"), ("llama-3.2-1b", 2048, "fp16"), ("mistral-7b-v0.3", 1100, "bf16"),
                                          ("llama-3.2-1b+qkv_bias", 1000, "bf16"), ("llama-3.2-1b", 2048, "bf16")])
def test_real_layer_shapes_prefill_equals_steps(name, S, dtype):
    """Real hidden/intermediate/head geometry (2 layers, 4096-entry vocabulary to keep the upload small): the batched matrix-core prefill against the same
    prompt through the decode kernels (other kernels, the same math)."""
    d = copy.deepcopy(known_desc(name.split("+")[0], dtype))
    d.layers, d.vocab, d.max_ctx = 2, 4096, max(512, S + 16)
    if name.endswith("+qkv_bias"):
        d.qkv_bias = True
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 77)[None, :]
    l1, f1, r1, kv1 = run(m, prompt, mfma=True, n_decode=3)
    l0, f0, r0, kv0 = run(m, prompt, mfma=False, n_decode=3)
    assert rel_err(l1, l0) < 1e-3, rel_err(l1, l0)
    np.testing.assert_array_equal(f1, f0)
    np.testing.assert_array_equal(r1, r0)
    ulp = {"bf16": 8e-3, "fp16": 1e-3, "fp32": 1e-5}[dtype]
    for (k1, v1), (k0, v0) in zip(kv1, kv0):
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp
    if dtype == "fp32":
        assert rel_err(l1, l0) < 1e-4


@pytest.mark.parametrize("fam,dtype", [("llama_tiny", "bf16"), ("qwen2_tiny", "bf16"), ("qwen3_tiny", "bf16"), ("mistral_tiny", "fp16")])
@pytest.mark.parametrize("nb,S", [(1, 33), (1, 48), (1, 64), (2, 29), (3, 21), (1, 65), (1, 100), (1, 128), (3, 40)])
def test_prompts_of_33_to_64_rows_on_the_skinny_kernels(fam, dtype, nb, S, oracle_lib):
    """Prompts whose rows (batch x length) number 33..64 run every product as a skinny MFMA GEMM with FOUR 16-row activation blocks, 65..128 rows with
    EIGHT (round 3, kernels/skinny.h MB = 4, kernels/skinny_dma.h MB = 4 / 8; option prefill.skinny_rows = 32 sends them back to the tiled split-K GEMMs;
    the fixtures' hidden sizes are below the 2048 limit of the eight-block form): against the oracle (<= 1e-3, first id where
    the gap is clear) and against the tiled path (<= 1e-3; K tails at hidden 192, QKV bias, q / k norm, head_dim 128, three-term QKV product in bf16)."""
    from oracle.oracle_ffi import OracleModel
    cfg, g = load_golden(fam)
    d = desc_from_hf_config(cfg, dtype, max_batch=nb)
    d.max_ctx = 136
    gpu = Model(d, product_backend()).load_synthetic(int(g["seed"]), float(g["std"])).finalize()
    ref = OracleModel(d).load_synthetic(int(g["seed"]), float(g["std"])).finalize()
    ids = np.stack([synth.synth_prompt(d.vocab, S, 9 + b) for b in range(nb)])
    ref.forward(ids)
    lr = ref.logits(rounded=False)
    out = {}
    for rows in (128, 32):
        gpu.set_option("prefill.skinny_rows", rows)
        gpu.reset_cache(); gpu.forward(ids)
        lg = gpu.logits(rounded=False).copy()
        assert rel_err(lg, lr) < 1e-3, (rows, rel_err(lg, lr))
        first = gpu.sample(GREEDY).copy()
        out[rows] = (lg, first, gpu.decode(4, GREEDY).copy(), [gpu.read_kv(nb - 1, l) for l in range(d.layers)])
    top2 = np.sort(lr, axis=1)[:, -2:]
    clear = (top2[:, 1] - top2[:, 0]) > 2e-3 * np.abs(lr).max()
    np.testing.assert_array_equal(out[128][1][clear], ref.sample(GREEDY)[clear])
    assert rel_err(out[128][0], out[32][0]) < 1e-3
    ulp = {"bf16": 8e-3, "fp16": 1e-3}[dtype]
    for (k1, v1), (k0, v0) in zip(out[128][3], out[32][3]):
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp


@pytest.mark.parametrize("name,S,dtype", [("llama-3.2-1b", 48, "bf16"), ("mistral-7b-v0.3", 40, "bf16"), ("qwen2.5-0.5b", 64, "bf16"), ("qwen3-1.7b", 57, "fp16")])
def test_real_layer_shapes_33_to_64_row_prompts_skinny_equals_tiled(name, S, dtype):
    """the same at real hidden / intermediate / head geometry (2 layers, 4096-entry vocabulary): the four-block skinny path against the tiled split-K path"""
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 2, 4096, 128
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 77)[None, :]
    res = {}
    m.set_option("prefill.skinny_hidden_max", 1 << 20)       # by default hidden > 2048 keeps 33-64-row prompts on the tiled path (faster there)
    for rows in (64, 32):
        m.set_option("prefill.skinny_rows", rows)
        res[rows] = run(m, prompt, mfma=True, n_decode=3)
    assert rel_err(res[64][0], res[32][0]) < 1e-3, rel_err(res[64][0], res[32][0])
    np.testing.assert_array_equal(res[64][1], res[32][1])
    np.testing.assert_array_equal(res[64][2], res[32][2])
    ulp = {"bf16": 8e-3, "fp16": 1e-3}[dtype]
    for (k1, v1), (k0, v0) in zip(res[64][3], res[32][3]):
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp


@pytest.mark.parametrize("name,S,dtype", [("llama-3.2-1b", 300, "bf16"), ("llama-3.2-1b", 1024, "bf16"), ("llama-3.2-1b", 700, "fp16"), ("mistral-7b-v0.3", 400, "bf16"), ("qwen2.5-0.5b", 600, "bf16")])
def test_n_hidden_products_as_k_slabs_on_the_eight_wave_kernel(name, S, dtype):
    """Round 4 (option prefill.splitk_8k, on by default): the o_proj / down products of a 129-1500-row prompt, whose 128 x 128 tiles number less than a chip, run as
    2-8 K slabs on the eight-wave LDS-DMA kernel (gemm_dma8k_kernel<.., GEMM_PARTIAL>; slabs summed in z order by the next row-wise kernel or the reducer).
    Against the same prompt without it (64-row register-staged slabs below 256 tiles, a half-empty chip above): the same products in another summation
    order — ONE layer (no cache row has a schedule-dependent input): logits within 2e-5, the same first token; and bit-identical on a second run."""
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 1, 4096, S + 16
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 78)[None, :]
    outs = []
    for on in (0, 1, 1):
        m.set_option("prefill.splitk_8k", on)
        m.reset_cache(); m.forward(prompt)
        outs.append((m.logits(rounded=False).copy(), m.sample(GREEDY).copy()))
    assert rel_err(outs[1][0], outs[0][0]) < 2e-5, rel_err(outs[1][0], outs[0][0])
    np.testing.assert_array_equal(outs[1][1], outs[0][1])
    np.testing.assert_array_equal(outs[1][0], outs[2][0])


@pytest.mark.parametrize("name,S", [("llama-3.2-1b", 1200), ("llama-3.2-1b", 1500), ("mistral-7b-v0.3", 600)])
def test_gate_up_on_128_tiles_where_the_256_tiling_is_ragged(name, S):
    """Round 4 (option prefill.wide_8k_eff, 76): a prompt whose 256 x 256 gate_up tiles would fill their last round of workgroups to less than 76 % (1152-1536 rows at
    intermediate 8192) takes the eight-wave 128 x 128 kernel instead — the kernel of the 129-384-row prompts on a larger grid.  Against the 256 x 256 tiling of the
    same prompt (option 0): the same products, the same siluMul epilogue, another tile shape: ONE layer, logits within 2e-5, same first token; the balanced QKV launch
    against K slabs (option prefill.qkv_nosplit) within 2e-4 (its results are rounded into this layer's cache)."""
    d = copy.deepcopy(known_desc(name, "bf16"))
    d.layers, d.vocab, d.max_ctx = 1, 4096, S + 16
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 79)[None, :]
    outs = []
    for eff, nosplit in ((0, 1), (76, 1), (76, 1), (76, 0)):
        m.set_option("prefill.wide_8k_eff", eff); m.set_option("prefill.qkv_nosplit", nosplit)
        m.reset_cache(); m.forward(prompt)
        outs.append((m.logits(rounded=False).copy(), m.sample(GREEDY).copy()))
    assert rel_err(outs[1][0], outs[0][0]) < 2e-5, rel_err(outs[1][0], outs[0][0])        # tile shape of gate_up only: no cache row changes
    np.testing.assert_array_equal(outs[1][1], outs[0][1])
    np.testing.assert_array_equal(outs[1][0], outs[2][0])
    # another schedule of the QKV product moves K / V entries across 16-bit rounding boundaries in THIS layer's cache: the two-layer bound of the form tests
    assert rel_err(outs[3][0], outs[1][0]) < 2e-4, rel_err(outs[3][0], outs[1][0])
    np.testing.assert_array_equal(outs[3][1], outs[1][1])


@pytest.mark.parametrize("name,S,dtype", [("llama-3.2-1b", 300, "bf16"), ("llama-3.2-1b", 777, "fp16"), ("qwen2.5-0.5b", 257, "bf16"),
                                          ("mistral-7b-v0.3", 300, "bf16"), ("llama-3.2-3b", 200, "fp16"), ("qwen3-1.7b", 333, "bf16"),
                                          ("llama-3.2-1b", 1100, "bf16"), ("mistral-7b-v0.3", 1061, "fp16")])
def test_prefill_attention_forms_agree(name, S, dtype):
    """Round 5: the two other schedules of the prompt attention — K / V tiles by LDS-DMA with the next tile's scores under the current softmax (head_dim 64,
    kernels/attn_prefill_dma.h: the same matrix instructions on the same operands in the same order -> BIT-identical) and the key split inside the workgroup
    (attn_prefill_kernel KP = 2: the odd tiles' online-softmax stream merged once at the end -> another fp32 summation order, 2e-5 on one layer) — forced on prompts
    that are ragged in the 128-query blocks and in the 64-key tiles.  The defaults take these forms only for long prompts / head_dim 128.  The key split runs in blocks of 64 queries
    while those of 128 do not outnumber the compute units (up to 1024 rows of 32 heads), in blocks of 128 beyond: the two longest prompts."""
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 1, 4096, S + 16
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 80)[None, :]
    outs = {}
    for form, (dma, ks) in {"plain": (0, 0), "dma": (2, 0), "ksplit": (0, 2), "plain2": (0, 0)}.items():
        m.set_option("prefill.attn_dma", dma); m.set_option("prefill.attn_ksplit", ks)
        m.reset_cache(); m.forward(prompt)
        outs[form] = (m.logits(rounded=False).copy(), m.sample(GREEDY).copy())
    np.testing.assert_array_equal(outs["plain"][0], outs["plain2"][0])
    if d.head_dim == 64:
        np.testing.assert_array_equal(outs["dma"][0], outs["plain"][0])
    assert rel_err(outs["ksplit"][0], outs["plain"][0]) < 2e-5, rel_err(outs["ksplit"][0], outs["plain"][0])
    np.testing.assert_array_equal(outs["ksplit"][1], outs["plain"][1])


@pytest.mark.parametrize("name,S,dtype", [("llama-3.2-1b", 1024, "bf16"), ("llama-3.2-1b", 1900, "bf16"), ("llama-3.2-1b", 2048, "fp16"), ("mistral-7b-v0.3", 1100, "bf16")])
def test_down_on_wide_tiles_matches_the_square_tiles(name, S, dtype):
    """Round 5: the K >> N product (`down`) of a prompt worth two chips of its workgroups (regime knob prefill.wide_n_min) runs on 128 x 256 tiles x 2 K slabs (kernels/gemm_dma.h
    gemm_dma8n_kernel: a third fewer operand lines per output; the slabs are summed in z order by the next norm launch) instead of one slab of 128 x 128 tiles — the same
    products in another fp32 summation order: TWO layers (the second layer's norm consumes the slabs), logits within 2e-5, the same first token; bit-identical on a rerun."""
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 2, 4096, S + 16
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 84)[None, :]
    outs = []
    for chips in (1 << 20, 1, 1):                     # never / from one chip's worth of workgroups on (the default: two)
        m.set_option("prefill.wide_n_min", chips)
        m.reset_cache(); m.forward(prompt)
        outs.append((m.logits(rounded=False).copy(), m.sample(GREEDY).copy()))
    assert rel_err(outs[1][0], outs[0][0]) < 2e-5, rel_err(outs[1][0], outs[0][0])
    np.testing.assert_array_equal(outs[1][1], outs[0][1])
    np.testing.assert_array_equal(outs[1][0], outs[2][0])




# query blocks of 64 (workgroups below a chip): the last block of one, 63 and 64 rows, keys that end at and beside a pair of tiles; gate_up whole below a chip of tiles; more than
# four slabs for the N = hidden products.  Bound: the two schedules differ by roundings of the cached keys and values, as above
@pytest.mark.parametrize("name", ["qwen3-0.6b", "qwen2.5-0.5b"])
@pytest.mark.parametrize("S,dtype", [(129, "bf16"), (191, "bf16"), (192, "fp16"), (193, "bf16"), (255, "fp16"), (385, "bf16"), (511, "fp16")])
def test_short_prompt_blocks_equal_steps(name, S, dtype):
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 2, 4096, 640
    gpu = Model(d, product_backend()).load_synthetic(17, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 3)[None, :]
    l1, _, _, kv1 = run(gpu, prompt, mfma=True)
    l0, _, _, kv0 = run(gpu, prompt, mfma=False)
    assert rel_err(l1, l0) < 1e-3
    ulp = {"bf16": 8e-3, "fp16": 1e-3}[dtype]
    for (k1, v1), (k0, v0) in zip(kv1, kv0):
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp


# blocks of 32 queries whose keys four waves divide (up to a chip of them; head_dim 128 from seven tiles of keys on): the last block of one, 31 and 32 rows, streams without a tile, keys
# that end at and beside four tiles.  Against the undivided form on one layer: another order of fp32 sums, 2e-5 as for two streams
@pytest.mark.parametrize("name,S", [("qwen2.5-0.5b", 129), ("qwen2.5-0.5b", 160), ("qwen2.5-0.5b", 191), ("qwen2.5-0.5b", 257), ("llama-3.2-1b", 256), ("qwen3-0.6b", 385), ("qwen3-0.6b", 449), ("qwen3-0.6b", 512)])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_four_streams_of_keys(name, S, dtype):
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 1, 4096, S + 16
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 80)[None, :]
    outs = []
    for ksplit in (0, 1, 1):
        m.set_option("prefill.attn_ksplit", ksplit)
        m.reset_cache(); m.forward(prompt)
        outs.append(m.logits(rounded=False).copy())
    np.testing.assert_array_equal(outs[1], outs[2])
    assert not (outs[0] == outs[1]).all()
    assert rel_err(outs[1], outs[0]) < 2e-5, rel_err(outs[1], outs[0])


# the eight-wave 128 x 128 tiles with a stage's k16 steps in halves (chains of up to 32 stages; 33 and 34 take quarters): the last row tile of one row, 32 and 127, column tiles that end
# inside, gate_up whole, N = hidden products in slabs and (700 rows) whole.  Against the steps as above
@pytest.mark.parametrize("S", [129, 160, 255, 257, 700])
@pytest.mark.parametrize("heads,inter,dtype", [(7, 1472, "bf16"), (32, 2048, "fp16"), (33, 2176, "bf16")])
def test_eight_wave_tiles_in_halves(heads, inter, dtype, S):
    d = copy.deepcopy(known_desc("llama-3.2-1b", dtype))
    d.hidden, d.heads, d.kv_heads, d.inter, d.layers, d.vocab, d.max_ctx = 64 * heads, heads, 1 if heads < 32 else heads // 8 if heads % 8 == 0 else 3, inter, 1, 1024, 704
    gpu = Model(d, product_backend()).load_synthetic(23, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 5)[None, :]
    l1, _, _, kv1 = run(gpu, prompt, mfma=True)
    l0, _, _, kv0 = run(gpu, prompt, mfma=False)
    assert rel_err(l1, l0) < 1e-3
    ulp = {"bf16": 8e-3, "fp16": 1e-3}[dtype]
    for (k1, v1), (k0, v0) in zip(kv1, kv0):
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp


# A stage's four k16 steps keep sums of their own, (0 + 2) + (1 + 3) at the end, whichever waves have them.  Weights of one large number in step 0 of every stage, its negative in step 2 and
# small multiples of 1/8 in steps 1 and 3, on an activation row of one value: sums of 0 and 2 cancel to nothing, those of 1 and 3 are exact to 2^-20; where 0 and 1 shared a sum, the large
# numbers (2^15 a stage) took the small ones' last bits, 1e-3 of the result and more.  What remains is a hidden value stored as two 16-bit terms (2^-17) through one product.
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("S", [129, 300])
@pytest.mark.parametrize("which", ["up", "down"])
def test_steps_of_a_stage_keep_their_own_sums(which, S, dtype):
    d = copy.deepcopy(known_desc("llama-3.2-1b", dtype))
    d.hidden, d.heads, d.kv_heads, d.inter, d.layers, d.vocab, d.max_ctx, d.tied = 1024, 16, 4, 2048, 1, 1024, 320, False
    rng = np.random.default_rng(3)
    w = {n: np.zeros(s, np.float32) for n, s in d.tensor_shapes().items()}
    for n in w:
        if "norm" in n:
            w[n][:] = 1
    w["model.embed_tokens.weight"][:] = 1
    w["lm_head.weight"][:] = np.eye(1024)
    gate, up, down = (w["model.layers.0.mlp.%s_proj.weight" % n] for n in ("gate", "up", "down"))
    gate[:, 0] = up[:, 0] = 1
    down[:, :1024] = np.eye(1024)
    m = up if which == "up" else down
    m[:] = rng.integers(-8, 9, m.shape) / 8
    k = np.arange(m.shape[1]) % 64
    m[:, (k < 16) | ((k >= 32) & (k < 48))] = 0
    m[:, k == 0], m[:, k == 32] = 2.0 ** 15, -2.0 ** 15
    gpu = Model(d, product_backend())
    for n, v in w.items():
        gpu.upload(n, v)
    gpu.finalize()
    gpu.set_option("prefill.mfma", 1)
    gpu.forward(rng.integers(0, 1024, S)[None, :])
    x = 1 / np.sqrt(1 + np.float64(d.norm_eps))
    g, u = gate.astype(np.float64).sum(1) * x, up.astype(np.float64).sum(1) * x
    y = 1 + down.astype(np.float64) @ (g / (1 + np.exp(-g)) * u)
    want = y / np.sqrt((y * y).mean() + d.norm_eps)
    assert rel_err(gpu.logits(rounded=False)[0], want) < 5e-5


# N = hidden products whose steps of 64 do not fill six or seven slabs (25 and 29 steps; tests/test_prefill_plan.py has the rule): the counts that do are taken.  Bound as above
@pytest.mark.parametrize("heads,S,dtype", [(25, 129, "bf16"), (25, 245, "fp16"), (29, 200, "bf16"), (29, 131, "fp16")])
def test_products_that_fill_no_six_slabs(heads, S, dtype):
    d = copy.deepcopy(known_desc("llama-3.2-1b", dtype))
    d.hidden, d.heads, d.kv_heads, d.inter, d.layers, d.vocab, d.max_ctx = 64 * heads, heads, 5 if heads == 25 else heads, 64 * heads, 2, 2048, 264
    gpu = Model(d, product_backend()).load_synthetic(19, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 5)[None, :]
    l1, _, _, kv1 = run(gpu, prompt, mfma=True)
    l0, _, _, kv0 = run(gpu, prompt, mfma=False)
    assert rel_err(l1, l0) < 1e-3
    ulp = {"bf16": 8e-3, "fp16": 1e-3}[dtype]
    for (k1, v1), (k0, v0) in zip(kv1, kv0):
        assert rel_err(k1, k0) < ulp and rel_err(v1, v0) < ulp


# gate_up on both sides of the rule that keeps it whole (tests/test_prefill_plan.py): 65 to 128 rows and half a chip of tiles (slabs), 65 rows and more tiles (whole), and the slabs that
# a low prefill.wide_8k_max asks for.  One layer: the same products and epilogue in another summation order
@pytest.mark.parametrize("name,S,dtype", [("llama-3.2-3b", 100, "bf16"), ("llama-3.2-3b", 128, "fp16"), ("mistral-7b-v0.3", 65, "bf16"), ("mistral-7b-v0.3", 128, "fp16"), ("qwen3-1.7b", 129, "bf16"), ("qwen3-0.6b", 257, "fp16")])
def test_gate_up_whole_equals_slabs(name, S, dtype):
    d = copy.deepcopy(known_desc(name, dtype))
    d.layers, d.vocab, d.max_ctx = 1, 4096, S + 16
    m = Model(d, product_backend()).load_synthetic(1234, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 81)[None, :]
    outs = []
    for most in (8, 0, 8):
        m.set_option("prefill.wide_8k_max", most)
        m.reset_cache(); m.forward(prompt)
        outs.append((m.logits(rounded=False).copy(), m.sample(GREEDY).copy()))
    assert rel_err(outs[1][0], outs[0][0]) < 2e-5, rel_err(outs[1][0], outs[0][0])
    np.testing.assert_array_equal(outs[1][1], outs[0][1])
    np.testing.assert_array_equal(outs[2][0], outs[0][0])


# the QKV product of a bf16 prompt in slabs of the eight-wave tiles, columns from the keys on with a third term: chains of one, four and more stages, a tile that holds queries and keys, the
# last tile of one row.  What the cache holds are sums rounded to bf16 (2^-9): with three terms (2^-25) and fp32 sums of at most 3072 terms (2^-24 each, some 2^-20 of the result) one entry
# in a thousand rounds to the other neighbour, with two (2^-17) one in a hundred and more
@pytest.mark.parametrize("name,S", [("qwen3-0.6b", 129), ("qwen3-0.6b", 384), ("qwen3-0.6b", 509), ("llama-3.2-1b", 133), ("llama-3.2-1b", 257), ("qwen2.5-0.5b", 640), ("wide", 129), ("wide", 255)])
def test_third_term_in_slabs(name, S):
    d = copy.deepcopy(known_desc("llama-3.2-1b" if name == "wide" else name, "bf16"))
    if name == "wide":      # 33 heads: keys begin inside a tile
        d.hidden, d.heads, d.kv_heads, d.inter = 2112, 33, 3, 2048
    d.layers, d.vocab, d.max_ctx = 1, 1024, 704
    m = Model(d, product_backend()).load_synthetic(29, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 6)[None, :]
    (k1, v1), = run(m, prompt, mfma=True, n_decode=1)[3]
    (k0, v0), = run(m, prompt, mfma=False, n_decode=1)[3]
    assert np.mean(k1 != k0) < 3e-3 and np.mean(v1 != v0) < 3e-3, (np.mean(k1 != k0), np.mean(v1 != v0))
    assert rel_err(k1, k0) < 8e-3 and rel_err(v1, v0) < 8e-3


@pytest.mark.parametrize("name,S", [("llama-3.2-1b", 257), ("qwen3-0.6b", 384)])
def test_qkv_slabs_by_option(name, S):
    """option prefill.qkv_8k 0: the QKV product on the register-staged tiles, as where the eight-wave kernels are off (prefill.gemm_dma without 8); prefill.splitk_8k leaves it alone"""
    d = copy.deepcopy(known_desc(name, "bf16"))
    d.layers, d.vocab, d.max_ctx = 1, 1024, S + 16
    m = Model(d, product_backend()).load_synthetic(31, 0.02).finalize()
    prompt = synth.synth_prompt(d.vocab, S, 7)[None, :]
    kv = {}
    for key, options in (("default", {}), ("slabs", {"splitk_8k": 0}), ("staged", {"qkv_8k": 0}), ("off", {"gemm_dma": 543 - 8})):
        for o, v in {"splitk_8k": 1, "qkv_8k": 1, "gemm_dma": 543, **options}.items():
            m.set_option("prefill." + o, v)
        kv[key] = np.concatenate([x.ravel() for x in run(m, prompt, mfma=True, n_decode=1)[3][0]])
    np.testing.assert_array_equal(kv["staged"], kv["off"])
    np.testing.assert_array_equal(kv["slabs"], kv["default"])
    assert (kv["staged"] != kv["default"]).any()
