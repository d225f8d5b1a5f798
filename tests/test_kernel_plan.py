"""This backend's launch and buffer plans checked against the reference's own Kernel IR goldens
(crates/modelspec-cli/tests/golden/{linear_regression,mnist_mlp}.kernel.ir, copied under
tests/golden/): every fusion group of the reference's step and forward plans is one launch here,
completing the same value, with the same fused operation chain or epilogue, in an order that keeps
every buffer dependency of the reference plan; operands the reference reads transposed are read in
place here too (no Transpose launch); every value a reference dispatch writes has storage here
(the arena, or the gradient arena for a gradient the optimizer reads). Planned without a device
(msx_plan), so this runs on the CPU.

Where this backend plans differently, by design: the reference's one sgd_update kernel a parameter
is one optimizer launch over the flat parameter arena; a RecordLoss launch appends the step's loss
to the device loss log (the reference's loss slots, kernel.rs:1515; where a cross-entropy loss
launch forms the loss, that launch appends it); weight-gradient GEMMs that only the optimizer reads
run on the side stream."""
import os

import pytest

from modelspec_amd import api

import kernel_ir
from ops_lib import Prog

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")


def plans(config):
    ref = kernel_ir.parse_reference(open(os.path.join(GOLDEN, f"{config}.kernel.ir")).read())
    step_ir, forward_ir = api.compile_config(config)
    ours = kernel_ir.parse_plan(api.plan(step_ir, forward_ir))
    return ref, ours, step_ir


def label(kernel):
    """The fused chain as this backend names it: Sub>Mul for the reference's Sub>Mul@0."""
    return ">".join(op.split("@")[0] for op in kernel["ops"])


@pytest.mark.parametrize("config", ["linear_regression", "mnist_mlp"])
@pytest.mark.parametrize("which", ["step", "forward"])
def test_every_reference_fusion_group_is_one_launch(config, which):
    ref, ours, step_ir = plans(config)
    launches = ours[which]["launches"]
    assert not any(l["what"].startswith("Transpose") for l in launches)
    placed = {}
    for d in ref["plans"][which]:
        k = ref["kernels"][d["kernel"]]
        if k["kind"] == "sgd_update":
            hits = [i for i, l in enumerate(launches) if l["what"] in ("SGD", "AdamW")]
        else:
            hits = [i for i, l in enumerate(launches) if d["value"] in l["values"]]
        assert len(hits) == 1, (config, which, d, [l["what"] for l in launches])
        what = launches[hits[0]]["what"]
        if k["kind"] == "matmul":
            assert what.startswith("MatMul"), what
            if k["epilogue"]:
                assert f"+{k['epilogue']} %" in what, (k, what)
        elif k["kind"] == "elementwise":
            assert what.startswith(label(k)), (k, what)
        elif k["kind"] == "loss_sum":
            assert what.startswith(k["ops"][0]), (k, what)
        placed[(d["kernel"], d["value"])] = hits[0]
    # Buffer dependencies of the reference plan keep their order here.
    ds = ref["plans"][which]
    for i, a in enumerate(ds):
        for b in ds[i + 1:]:
            if set(a["writes"]) & set(b["reads"]):
                pa, pb = placed[(a["kernel"], a["value"])], placed[(b["kernel"], b["value"])]
                assert pa < pb or ref["kernels"][b["kernel"]]["kind"] == "sgd_update", (a, b)
    # Every launch here is a reference group, or the loss log (step), or the loss (forward: the
    # reference's forward plan is the prediction's; this backend's forward program also gives the
    # final and held-out loss).
    groups = set(placed.values())
    extra = [l["what"].split()[0] for i, l in enumerate(launches) if i not in groups]
    assert extra == (["RecordLoss"] if which == "step" else ["Mse"]), extra


@pytest.mark.parametrize("config", ["linear_regression", "mnist_mlp"])
def test_every_value_a_reference_dispatch_writes_has_storage(config):
    ref, ours, step_ir = plans(config)
    gradients = {int(l.split("%")[1].split()[0]) for l in step_ir.splitlines()
                 if l.startswith("output %") and " gradient @" in l}
    for which in ("step", "forward"):
        slices = ours[which]["slices"]
        launches = ours[which]["launches"]
        for d in ref["plans"][which]:
            k = ref["kernels"][d["kernel"]]
            if k["kind"] == "sgd_update":
                continue  # the parameter arena, updated in place
            stored = lambda v: v in slices or (which == "step" and v in gradients)
            if k["epilogue"]:
                # A group with an epilogue stores its epilogue's value (the reference's buffer of the
                # dispatch holds it too): the other value of the launch completing d.
                owner = next(l for l in launches if d["value"] in l["values"])
                assert any(stored(v) for v in owner["values"] if v != d["value"]), (config, which, d, owner)
            else:
                assert stored(d["value"]), (config, which, d)


def test_the_forward_program_is_the_reference_tensor_ir_with_the_prediction():
    """golden/linear_regression.tensor.ir is the reference's lowered forward program; this
    backend's forward program is it with the prediction appended as a second output (held-out
    evaluation and synthetic teacher targets read it)."""
    _, forward_ir = api.compile_config("linear_regression")
    want = open(os.path.join(GOLDEN, "linear_regression.tensor.ir")).read()
    assert forward_ir == want + "output %3\n"


def test_bert_tiny_step_plan_takes_the_fused_paths():
    """The BERT-tiny step (the benchmark and the 1,000-step parity run) plans the fusions the GPU
    op tests check one by one: the Embedding gathers inside the LayerNorm pass, the masked-row
    scatter with its DropoutGrad, the Q/K/V input-gradient chains as K-segment GEMMs (one ending in
    a DropoutGrad epilogue), the loss summed and logged by a block of the optimizer launch (with the
    deferred column finalize), the EmbeddingGrad plans made on the host, and no Dropout,
    DropoutGrad, Embedding, RecordLoss, loss, finalize or EmbeddingPlan launch of its own."""
    step_ir, forward_ir = api.compile_config("bert_tiny")
    launches = kernel_ir.parse_plan(api.plan(step_ir, forward_ir))["step"]["launches"]
    whats = [l["what"] for l in launches]
    assert any(w.startswith("LayerNorm+fused") and w.count(" embedding %") == 2 for w in whats), whats
    assert any(w.startswith("EmbeddingGrad") and "+DropoutGrad %" in w for w in whats), whats
    chains = [w for w in whats if w.startswith("MatMul") and w.count(" (+) ") == 2]
    assert len(chains) == 2 and sum("+DropoutGrad %" in w for w in chains) == 1, chains
    assert any(w.startswith("ColumnFinalize") and "+ AdamW + CrossEntropyRows" in w and "+RecordLoss" in w
               for w in whats), whats
    assert not any(w.split()[0] in ("Dropout", "DropoutGrad", "Embedding", "RecordLoss", "AdamW") for w in whats), whats
    assert sum(w.startswith("CrossEntropyRows") for w in whats) == 1, whats
    # The EmbeddingGrad plans of the host-staged ids are made by the host with the step's inputs.
    assert not any(w.startswith("EmbeddingPlan") for w in whats), whats


def forward_plan(p, mixed):
    """The launch plan of a program of its own, beside any step."""
    step_ir, _ = api.compile_config("linear_regression")
    return kernel_ir.parse_plan(api.plan(step_ir, p.text(), 0, mixed))["forward"]


@pytest.mark.parametrize("m,k,n,ta,tb,chained", [
    (64, 64, 2 ** 25, False, False, True), (64, 64, 2 ** 25 + 64, False, False, False),
    (2 ** 25, 64, 64, True, False, True), (2 ** 25 + 64, 64, 64, True, False, False),
    (4096, 2 ** 23, 4096, False, True, True), (4096, 2 ** 23 + 64, 4096, False, True, False),
])
def test_mixed_products_past_32_bit_offsets_stay_off_the_f16_kernels(m, k, n, ta, tb, chained):
    """The f16 GEMM addresses an operand's tile by 32-bit byte offsets: 63 rows of a pitch up to 2^25
    halves where the rows run along K's columns, 255 of one up to 2^23 where they are contiguous along
    K, so 63 (2^25 + 256) 2 and 255 2^23 2 + 128 bytes both stay below 2^32. Two products added into
    one value join over their K only where that kernel takes them, which shows where the plan draws
    the line; a wider pitch goes to the kernel with 64-bit addresses."""
    p = Prog()
    total = p.input("x", (m, n))
    for q in (1, 2):
        a = p.input(f"a{q}", (k, m) if ta else (m, k))
        w = p.input(f"w{q}", (n, k) if tb else (k, n))
        lhs = p.op("Transpose", [a], (m, k)) if ta else a
        rhs = p.op("Transpose", [w], (k, n)) if tb else w
        total = p.op("Add", [total, p.op("MatMul", [lhs, rhs], (m, n))], (m, n))
    products = [l["what"] for l in forward_plan(p.out(total), True)["launches"] if l["what"].startswith("MatMul")]
    assert len(products) == (1 if chained else 2) and (" (+) " in products[0]) == chained, products


@pytest.mark.parametrize("L,S,H,heads,taken", [
    (96, 512, 64, 1, "all"), (512, 512, 64, 1, "all"), (157, 157, 64, 1, "all"), (158, 158, 64, 1, "none"),
    (100, 112, 64, 1, "all"), (100, 240, 64, 1, "forward"),  # 2 S d + S floats fit one LDS, with 2 L d + 3 L not
    (100, 512, 64, 1, "none"), (1, 336, 64, 1, "none"), (300, 304, 16, 1, "all"), (80, 80, 24, 1, "none"),
])
def test_attention_row_counts_are_refused_by_the_plan(L, S, H, heads, taken):
    """What no launch takes is refused when the program is planned, as unsupported, and not by the
    launch (inside a step's capture): row counts that are no multiple of 16 past the size limit, also
    where only the query rows are none."""
    for op in ("Attention", "AttentionGradQ", "AttentionGradK", "AttentionGradV"):
        p = Prog()
        q, k, v = p.input("q", (L, H)), p.input("k", (S, H)), p.input("v", (S, H))
        operands = [q, k, v, p.input("mask", (1, S))] + ([p.input("G", (L, H))] if op != "Attention" else [])
        p.out(p.op(op, operands, (L if op in ("Attention", "AttentionGradQ") else S, H), f"[heads = {heads}]"))
        if taken == "all" or (taken == "forward" and op == "Attention"):
            assert any(l["what"].startswith("Attention") for l in forward_plan(p, False)["launches"]), op
        else:
            with pytest.raises(api.MsxError, match="no HIP kernel") as e:
                forward_plan(p, False)
            assert e.value.code == -5, (op, e.value.code)


@pytest.mark.parametrize("m,k,n,mixed,split", [
    (4096, 5003, 256, True, 16),  # an untied head's input gradient over 5003 classes: 64 tiles of 128 x 128
    (2016, 580, 192, True, 1),    # K under 1024: unsplit
    (1000, 2052, 260, True, 22),  # rows of 4 mod 8 halves: 24 tiles, 22 slices of 96 K
    (4096, 5008, 256, True, 1),   # whole 16-byte groups: gemm16, which has smaller tiles instead
    (1000, 9000, 264, True, 4),   # the same with a deep K: 8 of its 256 x 192 tiles, slices of 2048 K or more
])
def test_a_product_is_split_for_the_kernel_that_runs_it(m, k, n, mixed, split):
    """Split-K slices fill the chip with the tiles of the kernel that takes the product: 128 x 128 ones,
    about 1024 blocks, for a mixed product whose pitches are no multiple of 8. The slices show in the
    arena: m n floats each beside the operands, their f16 copies and the outputs."""
    p = Prog()
    a, b, bias = p.input("a", (m, k)), p.input("b", (k, n)), p.input("bias", (n,))
    p.out(p.op("AddRows", [p.op("MatMul", [a, b], (m, n)), bias], (m, n)))
    plan = forward_plan(p, mixed)
    assert sum(l["what"].startswith("MatMul") for l in plan["launches"]) == 1
    slices = (plan["arena"] - 6 * (m * k + k * n) - 4 * n) / (4 * m * n) - 1  # less the output itself
    assert abs(slices - (split if split > 1 else 0)) <= 0.01, slices
