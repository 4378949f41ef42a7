"""Host-side decisions about kernel launches (CPU): key splits of the decode attention, pieces of
a sampled row, and which matrix-product kernel a tuned table sends a product to."""

import pytest
import torch

from torchllms_amd.kernels import attention_ops, ops, products, sequence_ops


def test_decode_splits_cover_the_range_and_stay_under_a_cu_s_share_of_blocks():
    for head_dim, per_cu in ((32, 3), (64, 3), (128, 2), (256, 1)):
        for n_tokens in (1, 2, 3, 8, 17, 64, 200):
            for n_kv_heads in (1, 2, 8):
                for longest in (1, 15, 256, 1000, 8192, 70000, 131072):
                    for uneven in (False, True):
                        split, n_splits = ops.plan_decode_splits(n_tokens, n_kv_heads, longest, head_dim, uneven=uneven)
                        assert split % 64 == 0 and split >= 128
                        assert n_splits >= 1 and (n_splits - 1) * split < max(longest, 1) <= n_splits * split
                        if uneven:
                            assert split <= attention_ops.DECODE_UNEVEN_SPLIT == 512
                        elif longest >= 4096 and split == 1024:
                            pass  # long contexts: no split beyond 1,024 keys, however many blocks that makes
                        elif n_splits > 1:
                            # (few long rows at head size 128 aim at one block a CU)
                            at_a_time = 256 * (1 if head_dim == 128 and n_tokens * n_kv_heads <= 32 else per_cu)
                            # never more blocks than the CUs take at a time, unless the shortest split allowed is reached
                            assert split == 128 or n_tokens * n_kv_heads * n_splits <= at_a_time
                            # and no fewer splits than that allows: one split more would be too many
                            shorter = split - 64
                            assert shorter < 128 or n_tokens * n_kv_heads * -(-longest // shorter) > at_a_time or -(-longest // shorter) == n_splits
    # head sizes with fewer bytes a key take more blocks a CU
    assert ops.plan_decode_splits(8, 8, 2176, 128) == (320, 7)
    assert ops.plan_decode_splits(8, 8, 2176, 64) == (192, 12)
    assert ops.plan_decode_splits(8, 4, 8192, 256) == (1024, 8)


def test_short_uneven_requests_in_numbers_are_left_whole():
    assert ops.decode_splits(64, 8, 1024, 128, uneven=True) == (1024, 1) and ops.decode_splits(64, 8, 768, 64, uneven=True) == (768, 1)
    for args in ((64, 8, 1025, 128), (63, 8, 1024, 128), (64, 4, 1000, 64), (8, 8, 300, 128)):  # longer, or fewer pairs: as planned
        assert ops.decode_splits(*args, uneven=True) == ops.plan_decode_splits(*args, uneven=True)
        assert ops.decode_splits(*args) == ops.plan_decode_splits(*args)


def test_requests_of_512_keys_and_fewer_are_left_whole_from_five_pairs_for_eight_cus_on():
    for head_dim in (32, 64, 128):
        assert ops.decode_splits(20, 8, 512, head_dim) == ops.decode_splits(160, 1, 100, head_dim, uneven=True) == (512, 1)
    # longer, fewer (16 requests of 512 keys take 10% more time whole at head size 64), or wider heads: as planned
    for args in ((20, 8, 513, 64), (19, 8, 512, 128), (16, 8, 512, 64), (20, 8, 512, 256)):
        assert ops.decode_splits(*args) == ops.plan_decode_splits(*args)


def test_32_bit_prompts_take_the_matrix_cores_where_few_requests_meet_in_a_block():
    one, eights, ragged = [0, 562], [8 * i for i in range(33)], [3, 25, 30, 400, 700]
    for heads, kv, dim, bounds, longest, want in (
            (32, 8, 64, one, 562, True), (32, 8, 128, one, 562, True), (6, 2, 128, one, 562, True), (4, 4, 32, [0, 33], 33, True),
            (8, 8, 128, eights, 8, False), (6, 2, 64, eights, 508, False), (8, 1, 128, eights, 508, False),  # 8, 8 and 2 meet
            (64, 8, 64, eights, 508, True), (32, 8, 64, [0, 32], 32, False), (32, 8, 128, [0, 64], 64, False),  # blocks for every CU; few keys
            (32, 8, 64, ragged, 700, True), (8, 8, 64, ragged, 700, False)):
        assert ops.runs_on_end(bounds, heads, kv, dim, longest) is want, (heads, kv, dim, bounds[-1], longest)


def test_recurrences_are_walked_where_the_workspace_of_the_chunks_is_too_large_or_not_to_be_had(monkeypatch):
    sizes = []

    class Library:
        @staticmethod
        def tl_chunk_floats(n, rows, heads, dim, memory):
            sizes.append((n, rows, heads, dim, memory))
            return 1000 if rows < 50 else sequence_ops.CHUNK_FLOATS_MOST + 1

    monkeypatch.setattr(sequence_ops, "core", lambda: Library)
    args = dict(n_heads=2, head_dim=64, device="cpu")
    ws, floats = sequence_ops._chunk_workspace(torch.bfloat16, 16, 3, 40, 5, **args)
    assert ws.numel() == floats == 1000 and ws.dtype == torch.float32 and sizes == [(37, 2, 2, 64, 0)]
    assert sequence_ops._chunk_workspace(torch.bfloat16, 16, 0, 2000, 50, **args) == (None, 0)

    def full(*_, **__):
        raise torch.OutOfMemoryError("full")

    monkeypatch.setattr(torch, "empty", full)
    assert sequence_ops._chunk_workspace(torch.bfloat16, 16, 3, 40, 5, **args) == (None, 0)


def test_a_sampled_row_is_cut_only_when_rows_are_few_and_long():
    assert ops.sample_chunks(1, 128256) == 15 and ops.sample_chunks(8, 128256) == 15
    assert ops.sample_chunks(64, 128256) == 4 and ops.sample_chunks(256, 128256) == 1
    assert ops.sample_chunks(1, 8191) == 1 and ops.sample_chunks(1, 32000) == 3 and ops.sample_chunks(0, 128256) == 15


def test_the_tuned_table_decides_per_shape_rows_and_use():
    w = torch.zeros(96, 256, dtype=torch.bfloat16)
    x = torch.zeros(40, 256, dtype=torch.bfloat16)
    keys = [(96, 256, b, use) for b in (8, 64, 128) for use in ops.LINEAR_USES]
    saved = {k: products.LINEAR_CHOICE[k] for k in keys if k in products.LINEAR_CHOICE}
    try:
        for k in keys:
            products.LINEAR_CHOICE.pop(k, None)
        assert ops.linear_choice(x, w) is None  # 40 rows, never measured: the library
        assert ops.linear_choice(x[:8], w) == ("stream", 0)  # 8 rows, never measured: the size rule
        products.LINEAR_CHOICE[(96, 256, 64, "plain")] = ("wide", 1, 2, 3)
        products.LINEAR_CHOICE[(96, 256, 64, "glu")] = ("wide", 2, 1, 3)
        products.LINEAR_CHOICE[(96, 256, 8, "plain")] = None
        assert ops.linear_choice(x, w) == ("wide", 1, 2, 3) and ops.linear_choice(x, w, "glu") == ("wide", 2, 1, 3)
        assert ops.linear_choice(x, w, "qkv") is None and ops.linear_choice(x[:8], w) is None
        assert ops.linear_choice(x[:33], w) == ("wide", 1, 2, 3)  # 33 to 64 rows share a bucket
        assert ops.linear_choice(torch.zeros(65, 256, dtype=torch.bfloat16), w) is None  # the next bucket, never measured
        assert ops.linear_choice(torch.zeros(129, 256, dtype=torch.bfloat16), w) is None  # too many rows
        assert ops.linear_choice(torch.zeros(40, 192, dtype=torch.bfloat16), torch.zeros(96, 192, dtype=torch.bfloat16)) is None  # K % 128
        assert ops.linear_choice(x.float(), w.float()) is None
    finally:
        for k in keys:
            products.LINEAR_CHOICE.pop(k, None)
        products.LINEAR_CHOICE.update(saved)


def test_which_candidates_are_charged_a_kernel_of_their_own_for_the_second_half():
    stream, whole, split, narrow = ("stream", 4), ("wide", 2, 1, 3), ("wide", 1, 4, 3), ("narrow",)
    for choice in (None, stream, whole, split, narrow):
        assert products.fuses_tail(choice, "plain")
    # the streaming product adds itself to the residual rows and leaves the norm's statistics; the library cannot
    assert [products.fuses_tail(c, "sum") for c in (None, stream, whole, split)] == [False, True, True, True]
    assert [products.fuses_tail(c, "glu") for c in (None, stream, whole, split)] == [False, True, True, False]
    assert [products.fuses_tail(c, "qkv") for c in (None, stream, whole, split)] == [False, True, False, True]
    assert [products.fuses_tail(narrow, use) for use in ("plain", "glu", "qkv", "sum")] == [True, False, True, True]


@pytest.mark.parametrize("n, k, narrow", [(3072, 2048, True), (4096, 2048, True), (96, 128, True), (4112, 1024, True), (2048, 8192, False),
                                          (4112, 2048, False), (8200, 512, False), (4096, 2176, False), (48, 192, False)])
def test_which_products_of_17_to_32_rows_run_by_the_kernel_for_few_columns(n, k, narrow):
    w, x = torch.empty((n, k), dtype=torch.bfloat16), torch.empty((33, k), dtype=torch.bfloat16)
    for m in (17, 32):
        for use in ops.LINEAR_USES:
            assert (ops.linear_choice(x[:m], w, use) == ("narrow",)) == (narrow and use in ("plain", "qkv"))
    assert ops.linear_choice(x[:16], w) != ("narrow",) and ops.linear_choice(x, w) != ("narrow",)


def test_what_the_kernels_for_17_rows_and_more_do_not_take_stays_with_the_library():
    """Columns that lie apart, more than two dimensions, matrices without rows or columns: no rule of sizes and no table sends
    them to a kernel that would refuse them."""
    bf = torch.bfloat16
    x, w = torch.empty((24, 256), dtype=bf), torch.empty((96, 256), dtype=bf)
    refused = [(torch.empty((24, 512), dtype=bf)[:, ::2], w), (x, torch.empty((96, 512), dtype=bf)[:, ::2]),
               (torch.empty((24, 256, 256), dtype=bf), w), (x, torch.empty((0, 256), dtype=bf)),
               (torch.empty((24, 0), dtype=bf), torch.empty((96, 0), dtype=bf))]
    saved = dict(products.LINEAR_CHOICE)
    try:
        for table in ({}, {(96, 256, 32, "plain"): ("wide", 1, 2, 3)}):
            products.LINEAR_CHOICE.clear()
            products.LINEAR_CHOICE.update(table)
            assert ops.linear_choice(x, w) is not None
            for a, b in refused:
                for use in ops.LINEAR_USES:
                    assert ops.linear_choice(a, b, use) is None, (a.shape, a.stride(), b.shape, b.stride(), use)
    finally:
        products.LINEAR_CHOICE.clear()
        products.LINEAR_CHOICE.update(saved)


def test_float32_products_of_what_is_no_matrix_are_refused_as_kernel_errors():
    for x in (torch.zeros(4), torch.zeros((2, 3, 4))):
        with pytest.raises(ops.KernelError):
            ops.linear_glu(x, torch.zeros((6, 4)))
        with pytest.raises(ops.KernelError):
            ops.qkv_rope_store(x, torch.zeros((12, 4)), None, 1, 1, 4, torch.zeros(2, dtype=torch.int32), None, 0, 0, None, None, None, None, 0)


def test_the_table_decides_before_the_rule_of_sizes():
    """Also for 17 to 32 rows of a shape that the rule gives to the kernel for few columns; and where the table has a use
    of the same shape only as a sum, a model that asks for the plain product gets that launch, at every row count."""
    w, x = torch.empty((3072, 2048), dtype=torch.bfloat16), torch.empty((24, 2048), dtype=torch.bfloat16)
    saved = dict(products.LINEAR_CHOICE)
    try:
        products.LINEAR_CHOICE.clear()
        ops.load_kernel_table({"3072,2048,32,plain": None, "3072,2048,32,qkv": ["wide", 1, 4, 3]})
        assert ops.linear_choice(x, w) is None and ops.linear_choice(x, w, "qkv") == ("wide", 1, 4, 3)
        ops.load_kernel_table({"3072,2048,32,plain": ["narrow"], "4096,4096,32,qkv": ["narrow"]})
        assert ops.linear_choice(x, w) == ("narrow",) and ops.kernel_table()["4096,4096,32,qkv"] == ["narrow"]
        for bad in ({"256,256,64,plain": ["narrow"]}, {"256,256,16,plain": ["narrow"]}, {"256,200,32,plain": ["narrow"]},
                    {"256,256,32,glu": ["narrow"]}, {"256,256,32,sum": ["narrow"]}, {"256,256,32,plain": ["narrow", 4]}):
            with pytest.raises(ValueError, match="kernel table"):
                ops.load_kernel_table(bad)
        ops.clear_kernel_table()
        old = {"3072,2048,8,sum": ["stream", 4], "3072,2048,32,sum": ["wide", 1, 8, 3], "3072,2048,64,sum": None}
        ops.load_kernel_table(old, [((3072, 2048), "sum")])
        assert len(ops.kernel_table()) == 3
        ops.load_kernel_table(old, [((3072, 2048), "plain")])
        assert ops.linear_choice(x, w) == ("wide", 1, 8, 3) and ops.linear_choice(x[:8], w) == ("stream", 4)
        ops.load_kernel_table(dict(old, **{"3072,2048,32,plain": None}), [((3072, 2048), "plain")])
        assert ops.linear_choice(x, w) is None
    finally:
        products.LINEAR_CHOICE.clear()
        products.LINEAR_CHOICE.update(saved)


def test_which_launches_of_the_wide_kernel_fit_lds():
    assert ops.wide_fits(64, 2, 3) and ops.wide_fits(128, 1, 3) and ops.wide_fits(128, 2, 2) and not ops.wide_fits(128, 2, 3)
    assert ops.wide_fits(20, 2, 3) and ops.wide_fits(65, 1, 2)


def test_the_table_survives_a_file(tmp_path):
    saved = dict(products.LINEAR_CHOICE)
    try:
        products.LINEAR_CHOICE.clear()
        products.LINEAR_CHOICE.update({(96, 256, 64, "plain"): ("wide", 2, 1, 3), (96, 256, 8, "glu"): ("stream", 4, 8),
                                       (96, 256, 8, "plain"): None, (512, 128, 1, "qkv"): ("stream", 0)})
        table = ops.kernel_table()
        assert table == {"96,256,8,glu": ["stream", 4, 8], "96,256,8,plain": None, "96,256,64,plain": ["wide", 2, 1, 3],
                         "512,128,1,qkv": ["stream", 0]}
        assert ops.kernel_table([((96, 256), "plain")]) == {"96,256,8,plain": None, "96,256,64,plain": ["wide", 2, 1, 3]}
        ops.save_kernel_table(tmp_path / "t.json")
        before = dict(products.LINEAR_CHOICE)
        ops.clear_kernel_table()
        assert products.LINEAR_CHOICE == {}
        ops.load_kernel_table(tmp_path / "t.json")
        assert products.LINEAR_CHOICE == before
    finally:
        products.LINEAR_CHOICE.clear()
        products.LINEAR_CHOICE.update(saved)


def test_libraries_built_in_the_tree_match_their_sources():
    """A library built before its source was last edited is compiled again at its next use, on the GPU
    box, where the time counts: build again after every change (``__graft_entry__.build()``).  A
    tree without built libraries (a fresh checkout) has nothing to compare."""
    from torchllms_amd.kernels import build

    assert build.stale_libraries() == []


def test_launch_plans_take_the_device_s_own_figures(monkeypatch):
    """Compute units and LDS size come from the device (the target's published figures where there is
    no GPU, as here): a GPU with half the CUs gets half the splits, one with less LDS fewer buffers."""
    from torchllms_amd.kernels import lib

    assert lib.device_facts() == (256, 160 * 1024)
    assert ops.plan_decode_splits(1, 8, 8192) == (256, 32) and ops.plan_decode_splits(8, 8, 2176) == (320, 7)
    assert ops.wide_fits(64, 2, 3) and ops.rmsnorm_max_hidden() == 40704
    monkeypatch.setattr(lib, "_facts", (128, 64 * 1024))
    assert ops.plan_decode_splits(1, 8, 8192) == (512, 16) and ops.plan_decode_splits(8, 8, 2176) == (576, 4)  # half the blocks at a time
    assert not ops.wide_fits(64, 2, 3) and ops.wide_fits(32, 1, 2) and ops.rmsnorm_max_hidden() == 16128


def test_a_head_size_without_matrix_core_kernels_is_reported_once(caplog):
    """A bfloat16 model whose head size only the plain attention kernel takes runs, right and slowly:
    the attention part says so, once per shape, when the engine asks it about its sizes."""
    import logging

    from torchllms_amd.config.spec import PartSpec
    from torchllms_amd.parts import MIXERS

    def part(head_dim, heads=6, kv=3):
        return MIXERS.build(PartSpec("attention", dict(
            hidden_size=96, num_heads=heads, num_kv_heads=kv, head_dim=head_dim, qkv_bias=False, softmax_scale=head_dim ** -0.5, window=0,
            position=PartSpec("rope", dict(head_dim=head_dim, rotary_dim=head_dim, theta=100.0, scaling=None)))))

    with caplog.at_level(logging.WARNING, logger="torchllms_amd"):
        part(64).check_sizes(torch.bfloat16)
        part(96).check_sizes(torch.float32)
        assert not caplog.records
        part(96).check_sizes(torch.bfloat16)
        part(96).check_sizes(torch.bfloat16)
        assert len(caplog.records) == 1 and "head size 96" in caplog.text and "decode steps and prompts run the plain kernel" in caplog.text
        part(256, heads=16, kv=1).check_sizes(torch.bfloat16)  # 16 query heads per kv head: prompts only
        assert len(caplog.records) == 2 and "; decode steps run the plain kernel" in caplog.records[1].getMessage()


def test_near_ties_of_the_measurement_are_decided_by_rule_not_by_the_stopwatch():
    """Candidates within 4% of the fastest count as equal; among them one that does the whole use in its own
    kernels wins over one that needs a kernel behind it, a kernel of the package over the library, and the
    candidates' fixed order decides the rest: the table, and with it the bfloat16 bits, does not flip from
    run to run on a tie."""
    lib, split, whole = None, ("wide", 1, 2, 3), ("wide", 2, 1, 3)
    assert products.pick([(lib, 17.9), (split, 18.4), (whole, 22.0)], "qkv") == split  # rotates in its second kernel
    assert products.pick([(lib, 18.4), (split, 17.9)], "qkv") == split
    assert products.pick([(lib, 17.0), (split, 18.4)], "qkv") is lib  # 8% apart: no tie
    assert products.pick([(lib, 50.0), (whole, 50.5), (split, 50.2)], "glu") == whole  # the gate ends a whole product
    assert products.pick([(lib, 10.0), (split, 10.3), (whole, 10.2)], "sum") == split  # first of the package's in the list
    assert products.pick([(lib, 10.0)], "plain") is lib


def test_layers_that_make_a_tensor_of_a_branch_at_once_have_its_last_product_run_whole():
    from torchllms_amd.parts import blocks
    from torchllms_amd.parts.base import Part

    for block, whole in ((blocks.PreNormMixerBlock, False), (blocks.PreNormBlock, False), (blocks.SandwichBlock, True),
                         (blocks.SandwichNormedPairBlock, True), (blocks.BranchNormBlock, True)):
        built = block({slot: Part() for slot in block.SLOTS})
        for slot, kind in block.SLOTS.items():
            if kind != "norm":
                assert built.parts[slot].closing_use == ("plain" if whole else "sum"), (block, slot)
