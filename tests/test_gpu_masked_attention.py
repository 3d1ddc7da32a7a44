"""GPU parity of the masked prefill attention kernel against the dense CPU oracle.

Covers the reference's mask language (attention_lab/masks.py) and both
implementations of attention_lab/triton_attention.py (interval, csr), the
global-prefix extension, document masks, LSE, strided inputs and the BASELINE
config-5 shape. Tolerances: bf16 2e-2, fp16 4e-3 on outputs; LSE 1e-2 / 2e-3.
"""

import itertools

import pytest
import torch

from oracle.attention import masked_attention, spec_mask
from systems_for_llms_amd.attention import attention
from systems_for_llms_amd.masks import MaskSpec, compile_mask

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: (2e-2, 1e-2), torch.float16: (4e-3, 2e-3)}

SPECS = [
    MaskSpec(causal=True),
    MaskSpec(),
    MaskSpec(causal=True, window_left=31),
    MaskSpec(window_left=7, window_right=3),
    MaskSpec(causal=True, window_left=40, global_prefix=64),
    MaskSpec(window_left=5, window_right=0, global_prefix=17),
]


def inputs(b, h, n, d, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    return [torch.randn((b, h, n, d), generator=g).to(dtype) for _ in range(3)]


def check(q, k, v, spec, docs, impl, use_full, block=64, return_lse=True):
    n = q.shape[2]
    doc_list = docs.tolist() if isinstance(docs, torch.Tensor) else docs
    schedule = compile_mask(n, spec, block, block, doc_list)
    gq, gk, gv = (t.cuda() for t in (q, k, v))
    out, lse = attention(gq, gk, gv, schedule, spec, document_ids=docs, implementation=impl,
                         use_full_blocks=use_full, return_lse=True)
    torch.cuda.synchronize()
    mask = spec_mask(n, spec, doc_list)
    ref_out, ref_lse = masked_attention(q, k, v, mask)
    atol, ltol = TOL[q.dtype]
    torch.testing.assert_close(out.float().cpu(), ref_out.float(), atol=atol, rtol=atol)
    torch.testing.assert_close(lse.cpu(), ref_lse.float(), atol=ltol, rtol=ltol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_specs_both_implementations(dtype, d):
    for n, spec in itertools.product((1, 17, 64, 65, 200), SPECS):
        q, k, v = inputs(2, 3, n, d, dtype, n + d)
        for impl in ("interval", "csr"):
            check(q, k, v, spec, None, impl, True)
    q, k, v = inputs(1, 2, 129, d, dtype, 5)
    check(q, k, v, MaskSpec(causal=True, window_left=20), None, "csr", False)
    check(q, k, v, MaskSpec(causal=True, window_left=20), None, "interval", False)


def test_document_masks_csr():
    docs = [(i // 23) % 4 for i in range(150)]
    q, k, v = inputs(2, 2, 150, 64, torch.bfloat16, 11)
    for spec in (MaskSpec(same_document=True), MaskSpec(causal=True, same_document=True),
                 MaskSpec(causal=True, window_left=30, same_document=True, global_prefix=10)):
        check(q, k, v, spec, docs, "csr", True)
    check(q, k, v, MaskSpec(causal=True, same_document=True), torch.tensor(docs), "csr", True)


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("n", [1, 63, 65, 128, 515])
def test_document_labels_at_tile_edges(n, d):
    """Scattered labels that differ in their upper 32 bits only, at the edges of the key tiles."""
    g = torch.Generator().manual_seed(n)
    docs = (torch.randint(0, 3, (n,), generator=g) << 32).sort().values
    docs[n // 2:] = docs[n // 2:][torch.randperm(n - n // 2, generator=g)]
    q, k, v = inputs(1, 3, n, d, torch.bfloat16, n + d)
    for spec in (MaskSpec(same_document=True), MaskSpec(causal=True, same_document=True),
                 MaskSpec(causal=True, window_left=70, same_document=True, global_prefix=5)):
        check(q, k, v, spec, docs.tolist(), "csr", True)


@pytest.mark.parametrize("b,h,n,d", [(5, 12, 1000, 64), (3, 11, 600, 32), (9, 15, 300, 128)])
def test_every_query_tile_is_dealt_once(b, h, n, d):
    """Grids of one to four workgroups per CU, the last round of an XCD partial."""
    q, k, v = inputs(b, h, n, d, torch.float16, n)
    check(q, k, v, MaskSpec(causal=True), None, "interval", True)


def test_schedule_compiled_for_other_tiles_is_recompiled():
    q, k, v = inputs(1, 2, 300, 64, torch.bfloat16, 3)
    for block in (16, 32, 128):
        check(q, k, v, MaskSpec(causal=True, window_left=50), None, "csr", True, block=block)


def test_strided_inputs_and_output_buffer():
    g = torch.Generator().manual_seed(9)
    b, n, h, d = 2, 130, 4, 64
    qkv = torch.randn((b, n, 3, h, d), generator=g).to(torch.bfloat16).cuda()
    q, k, v = (qkv[:, :, i].transpose(1, 2) for i in range(3))  # [B, H, N, D] views
    out = torch.empty((b, n, h, d), dtype=torch.bfloat16, device="cuda").transpose(1, 2)
    spec = MaskSpec(causal=True)
    res = attention(q, k, v, compile_mask(n, spec), spec, implementation="interval", out=out)
    assert res.data_ptr() == out.data_ptr()
    ref, _ = masked_attention(q.cpu(), k.cpu(), v.cpu(), spec_mask(n, spec))
    torch.testing.assert_close(out.float().cpu(), ref.float(), atol=2e-2, rtol=2e-2)


def test_config5_shape_sampled_heads():
    """B=4, H=16, N=4096, D=64, causal window 1024 + 4 global 64-key blocks."""
    spec = MaskSpec(causal=True, window_left=1023, global_prefix=256)
    b, h, n, d = 4, 16, 4096, 64
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((b, h, n, d), device="cuda", generator=g, dtype=torch.bfloat16) for _ in range(3))
    schedule = compile_mask(n, spec, 64, 64)
    outs = {impl: attention(q, k, v, schedule, spec, implementation=impl, return_lse=True)
            for impl in ("interval", "csr")}
    torch.cuda.synchronize()
    mask = spec_mask(n, spec)
    for bi, hi in ((0, 0), (3, 11)):
        ref_out, ref_lse = masked_attention(q[bi, hi].cpu(), k[bi, hi].cpu(), v[bi, hi].cpu(), mask,
                                            dtype=torch.float32)
        for impl, (out, lse) in outs.items():
            torch.testing.assert_close(out[bi, hi].float().cpu(), ref_out, atol=2e-2, rtol=2e-2)
            torch.testing.assert_close(lse[bi, hi].cpu(), ref_lse, atol=1e-2, rtol=1e-2)
    torch.testing.assert_close(outs["interval"][0], outs["csr"][0], atol=0, rtol=0)


@pytest.mark.parametrize("use_full", [True, False])
def test_kernel_follows_a_hand_edited_schedule(use_full):
    """The kernel walks the CSR it is given (validate.py:31-55 semantics), not the mask behind it:
    a dropped tile is skipped, a partial tile flagged full is taken whole (unless use_full_blocks
    is off, when every tile goes through the token mask)."""
    from oracle.attention import scheduled_attention

    n = 300
    spec = MaskSpec(causal=True, window_left=70)
    schedule = compile_mask(n, spec, 64, 64)
    # Row 3: drop its first tile. Row 2: flag its diagonal (partial) tile as full.
    first = schedule.row_ptr[3]
    assert schedule.row_ptr[4] - first >= 2
    schedule.col_idx.pop(first)
    schedule.full_blocks.pop(first)
    schedule.row_ptr[4:] = [p - 1 for p in schedule.row_ptr[4:]]
    diag = schedule.row_ptr[3] - 1
    assert schedule.col_idx[diag] == 2 and not schedule.full_blocks[diag]
    schedule.full_blocks[diag] = True
    q, k, v = inputs(2, 3, n, 64, torch.bfloat16, 41)
    out = attention(q.cuda(), k.cuda(), v.cuda(), schedule, spec, implementation="csr",
                    use_full_blocks=use_full)
    ref = scheduled_attention(q, k, v, schedule, spec, use_full_blocks=use_full)
    torch.testing.assert_close(out.float().cpu(), ref.float(), atol=2e-2, rtol=2e-2)
    unedited = masked_attention(q, k, v, spec_mask(n, spec))[0]
    assert (ref - unedited).abs().max() > 0.1  # the edits matter


@pytest.mark.parametrize("d", [32, 64, 128])
def test_launch_metadata_records_the_launched_kernels_resources(d):
    """launch_metadata gets the compiler's resource data for the kernel the call ran
    (triton_attention.py:39-57 records the same fields from Triton): rows of at most 512
    visible keys run one 64-query row per workgroup at head dim 64."""
    for n, spec, kind in ((130, MaskSpec(causal=True), "short"), (1000, MaskSpec(causal=True), "long"),
                          (1000, MaskSpec(causal=True, window_left=127), "short")):
        q, k, v = (t.cuda() for t in inputs(1, 2, n, d, torch.bfloat16, 3))
        meta = {}
        attention(q, k, v, compile_mask(n, spec), spec, launch_metadata=meta)
        expected = {32: "masked_attention_kernel<D=32>",
                    64: "masked_attention32_kernel<D=64, 2 waves>" if kind == "short"
                    else "masked_attention32_kernel<D=64>",
                    128: "masked_attention32_kernel<D=128>"}[d]
        print(meta)
        assert meta["kernel_name"] == expected + " bf16"
        assert meta["queries_per_workgroup"] == (64 if d == 32 or "2 waves" in expected else 128)
        assert 0 < meta["n_regs"] <= 512 and meta["n_spills"] == (0 if meta["private_segment_bytes"] == 0 else None)
        assert meta["shared_memory_bytes"] > 0 and meta["threads"] in (128, 256)
        assert meta["asm_sha256"] == {} and len(meta["library_sha256"]) == 64
        assert "not rocprof" in meta["source"]


@pytest.mark.parametrize("d,n,name", [(32, 300, "masked_attention_kernel<D=32>"),
                                      (64, 130, "masked_attention32_kernel<D=64, 2 waves, documents>"),
                                      (64, 1000, "masked_attention32_kernel<D=64, documents>"),
                                      (128, 300, "masked_attention32_kernel<D=128, documents>")])
def test_launch_metadata_of_document_masks(d, n, name):
    """Masks with documents run kernels of their own at head dims 64 and 128, which keep a tile's labels in LDS."""
    q, k, v = (t.cuda() for t in inputs(1, 2, n, d, torch.bfloat16, 3))
    plain, with_documents, docs = {}, {}, [i // 70 for i in range(n)]
    spec = MaskSpec(causal=True)
    attention(q, k, v, compile_mask(n, spec), spec, launch_metadata=plain)
    spec = MaskSpec(causal=True, same_document=True)
    attention(q, k, v, compile_mask(n, spec, document_ids=docs), spec, docs, launch_metadata=with_documents)
    assert with_documents["kernel_name"] == name + " bf16"
    labels = 0 if d == 32 else 8 * 64 * with_documents["threads"] // 64
    assert with_documents["shared_memory_bytes"] >= plain["shared_memory_bytes"] + labels
    assert (with_documents["kernel_name"] == plain["kernel_name"]) == (d == 32)
