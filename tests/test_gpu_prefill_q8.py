"""Q8_0 stacks with f32 activations over many rows (prefill chunks, the
lm.pas:391-408 forward over a block of embeddings): the products run on the
bf16 matrix cores (quants exact in bf16, activations split exactly into three
bf16 parts), in 16-row tiles up to 64 rows and in 64-row tiles staged through
LDS above. Every layer's output of every row against the oracle's (the
reference's Q8_0 bar, 1e-3 of max |ref|; QwenDiff of tests/test.tts.qwen.ref.pas),
for chunk sizes that take each tile shape, ragged last tiles and the K-sliced
o_proj / down products, with the context growing across chunks."""
import numpy as np
import pytest

import q3h
import q3o
import synth
from models import rel

pytestmark = pytest.mark.gpu


# chunks of one context: 16-row tiles (TM 1, 2, 4) and 64-row tiles staged in
# LDS (65 = one full tile and one row, 130 = two and two rows, 200)
@pytest.mark.parametrize("chunks", [(5, 17, 48), (33, 65, 130), (64, 200, 1)],
                         ids=["tiles16", "tiles64", "big_then_decode"])
def test_q8_prefill_layers_match_the_oracle(device, chunks):
    print(f"case chunks={chunks}", flush=True)
    dims = dict(synth.TALKER, layers=3)
    layers, final = synth.stack_weights(43, "talker.model.", dims, norm_std=0.1,
                                        quantize=q3o.quantize_q8_0)
    st = q3h.Stack(device, dict(dims, dtype=q3h.Q8_0, kv_f16=0, act_q8=0, max_positions=512),
                   layers, final, q3h.Q8_0)
    ost = q3o.Stack(dims, layers, final, q3o.Q8_0, act_q8=0)
    ctx, oc = q3h.Context(st, 512), q3o.Ctx(ost, 512)
    worst = 0.0
    try:
        for i, rows in enumerate(chunks):
            x = synth.prompt(700 + i, rows)
            _, normed, lo, _ = ctx.forward_probe(x)
            onormed, olo = oc.forward(x, layer_out=True)
            for l in range(dims["layers"]):
                r = rel(lo[l], olo[l])
                worst = max(worst, r)
                assert r < 1e-3, (rows, l, r)
            assert rel(normed, onormed) < 1e-3
        assert ctx.length == sum(chunks)
        print(f"worst relative error {worst:.2e}", flush=True)
    finally:
        ctx.destroy()
        oc.destroy()
        st.destroy()
        ost.destroy()


# other shapes: 4 query / 2 kv heads (o_proj K = 512: 2 slices) and an
# intermediate size of 1536 (down: 6 slices); 24 and 40 rows take the
# 256-column slices, 8 rows the whole-K tiles
def test_q8_prefill_other_slice_counts(device):
    dims = dict(synth.TALKER, layers=2, heads=4, kv_heads=2, intermediate=1536)
    layers, final = synth.stack_weights(44, "talker.model.", dims, norm_std=0.1,
                                        quantize=q3o.quantize_q8_0)
    st = q3h.Stack(device, dict(dims, dtype=q3h.Q8_0, kv_f16=0, act_q8=0, max_positions=128),
                   layers, final, q3h.Q8_0)
    ost = q3o.Stack(dims, layers, final, q3o.Q8_0, act_q8=0)
    ctx, oc = q3h.Context(st, 128), q3o.Ctx(ost, 128)
    try:
        for i, rows in enumerate((24, 40, 8)):
            x = synth.prompt(710 + i, rows)
            _, normed, lo, _ = ctx.forward_probe(x)
            onormed, olo = oc.forward(x, layer_out=True)
            for l in range(dims["layers"]):
                assert rel(lo[l], olo[l]) < 1e-3, (rows, l, rel(lo[l], olo[l]))
            assert rel(normed, onormed) < 1e-3
    finally:
        ctx.destroy()
        oc.destroy()
        st.destroy()
        ost.destroy()


# Relative bar of the many-row products against the oracle's fp32 forward. Both
# round each residual add of the layer once (2^-24 of the largest value, 6e-8, two
# adds on each side: 2.4e-7 where they fall together); the products' own sums are
# closer than that (weights of 0.02 beside residuals of order one). 2.1e-7 to
# 3.8e-7 measured; a lost lowest part of the activations is 8.8e-6, of both
# operands 1.6e-5.
MANY_ROWS_BAR = 1e-6


def _one_layer(device, dtype, positions, kv16=0):
    dims = dict(synth.TALKER, layers=1)
    quant = q3o.quantize_q8_0 if dtype == q3h.Q8_0 else None
    layers, final = synth.stack_weights(47, "talker.model.", dims, norm_std=0.1, quantize=quant)
    st = q3h.Stack(device, dict(dims, dtype=dtype, kv_f16=kv16, act_q8=0,
                                max_positions=positions), layers, final, dtype)
    odt = q3o.Q8_0 if dtype == q3h.Q8_0 else q3o.F32
    return st, q3o.Stack(dims, layers, final, odt, kv_f16=kv16, act_q8=0)


@pytest.mark.parametrize("f32", [0, 1], ids=["q8", "f32"])
@pytest.mark.parametrize("rows", [65, 97, 203, 321, 1030])
def test_many_row_tiles(device, f32, rows):
    """The products over split activations (more than 64 rows) at row counts
    that take each tile (32 x 64, 64 x 64, 64 x 128 by rounds of the chip),
    last tiles of 1, 11 and 6 rows, and the 32-query attention tiles (1030):
    the layer output of every row."""
    print(f"case f32={f32} rows={rows}", flush=True)
    st, ost = _one_layer(device, q3h.F32 if f32 else q3h.Q8_0, rows)
    ctx, oc = q3h.Context(st, rows), q3o.Ctx(ost, rows)
    try:
        x = synth.prompt(720, rows)
        _, normed, lo, _ = ctx.forward_probe(x)
        onormed, olo = oc.forward(x, layer_out=True)
        worst = max(rel(lo[0], olo[0]), rel(normed, onormed))
        print(f"relative error {worst:.2e}", flush=True)
        assert worst < MANY_ROWS_BAR, worst
    finally:
        ctx.destroy()
        oc.destroy()
        st.destroy()
        ost.destroy()


@pytest.mark.parametrize("f32", [0, 1], ids=["q8", "f32"])
def test_wide_attention_tiles_onto_a_context(device, f32):
    """32-query attention tiles (1024 rows and more at 16 heads) onto positions
    that are there already: 37 rows, then 1030, whose first tile starts at 37, in
    the middle of a 32-key block, and whose last has 6 rows."""
    st, ost = _one_layer(device, q3h.F32 if f32 else q3h.Q8_0, 1067)
    ctx, oc = q3h.Context(st, 1067), q3o.Ctx(ost, 1067)
    try:
        for rows in (37, 1030):
            x = synth.prompt(740, rows)
            _, normed, lo, _ = ctx.forward_probe(x)
            onormed, olo = oc.forward(x, layer_out=True)
            worst = max(rel(lo[0], olo[0]), rel(normed, onormed))
            print(f"rows {rows}: relative error {worst:.2e}", flush=True)
            assert worst < MANY_ROWS_BAR, (rows, worst)
    finally:
        ctx.destroy()
        oc.destroy()
        st.destroy()
        ost.destroy()


@pytest.mark.parametrize("f32", [0, 1], ids=["q8", "f32"])
def test_many_contexts_one_row_each(device, f32):
    """70 contexts of 1 to 5 positions, one row each in one call: the many-row
    products behind the decode attention."""
    n = 70
    st, ost = _one_layer(device, q3h.F32 if f32 else q3h.Q8_0, 72)
    ctxs = [q3h.Context(st, 8) for _ in range(n)]
    octxs = [q3o.Ctx(ost, 8) for _ in range(n)]
    try:
        for i in range(n):
            p = synth.prompt(730 + i, 1 + i % 5)
            ctxs[i].forward(p, want_logits=False, want_normed=False)
            octxs[i].forward(p)
        x = synth.prompt(729, n)
        _, normed = q3h.forward_batch(ctxs, x)
        worst = max(rel(normed[i], octxs[i].forward(x[i:i + 1])) for i in range(n))
        print(f"relative error {worst:.2e}", flush=True)
        assert worst < MANY_ROWS_BAR, worst
    finally:
        for c in ctxs + octxs:
            c.destroy()
        st.destroy()
        ost.destroy()
