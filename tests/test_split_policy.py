"""The policy that splits the K range of residual-writing products (no GPU needed)."""

from burn_transformers_amd.parts.base import split_count


def slices(k, splits):
    chunks = (k + 31) // 32
    per = (chunks + splits - 1) // splits
    return [min(per, max(0, chunks - i * per)) for i in range(splits)]


def test_many_rows_never_split():
    assert split_count(65, 1600, 6400) == 1
    assert split_count(2048, 1600, 1600) == 1


def test_every_slice_has_work_and_is_not_thin():
    for rows in (1, 8, 16, 17, 64):
        for columns in (16, 64, 96, 517, 1600, 50257):
            for k in (8, 64, 96, 320, 1600, 1608, 6400, 20480):
                for units in (64, 256, 304):
                    splits = split_count(rows, columns, k, units)
                    assert 1 <= splits <= 8
                    parts = slices(k, splits)
                    assert all(p > 0 for p in parts), (rows, columns, k, units, parts)
                    if splits > 1:
                        assert parts[0] >= 4


def test_choices_at_measured_sizes():
    # 100 tiles of 16 columns on 256 compute units: measured best are 2 splits for K 1600, 5 for K 6400
    assert split_count(8, 1600, 1600) == 2
    assert split_count(8, 1600, 6400) == 5
    # wide outputs fill the compute units on their own
    assert split_count(8, 50257, 1600) == 1
    # beyond 16 rows a work-group owns 32 columns, so there are half as many tiles to spread
    assert split_count(64, 1600, 6400) >= split_count(8, 1600, 6400)
    # every slice is read again by the norm behind the product: K = 1,024 is not cut into eight slices of
    # four chunks where four of eight do nearly as well (a step of 17 rows at width 1,024 was 2 % slower)
    assert split_count(17, 1024, 1024) == 4


def test_a_folded_norm_is_worth_it_by_rows_and_width():
    """Up to eight rows at every width the kernel takes; nine to sixteen rows only where a wave's two
    rows are short (measured at widths 768, 1,024 and 1,600)."""
    from burn_transformers_amd.kernels.library import Normalized
    assert all(Normalized.worth_it(8, width) for width in (768, 1024, 1600, 2048))
    assert Normalized.worth_it(16, 768) and Normalized.worth_it(9, 1024) and Normalized.worth_it(16, 1024)
    assert not Normalized.worth_it(9, 1600) and not Normalized.worth_it(16, 1280)
    assert not Normalized.worth_it(17, 768) and not Normalized.worth_it(4, 4096) and not Normalized.worth_it(4, 772)


# --- the runs a decode step's keys are cut into, and the classes of context ---------------------

def _runs(monkeypatch, n_seqs, context_limit, kv_heads=25, head_dim=64, bf16=True, window=0, decode=True, units=256, chunk=0, keep=0):
    from types import SimpleNamespace
    from burn_transformers_amd.parts import attention
    monkeypatch.setattr(attention, "compute_units", lambda device: units)
    mixer = SimpleNamespace(kv_heads=kv_heads, head_dim=head_dim, window=window, chunk=chunk, keep=keep)
    step = SimpleNamespace(decode=decode, context_limit=context_limit, dtype_is_bf16=bf16, n_seqs=n_seqs)
    return attention.CausalSelfAttention.decode_runs(mixer, step, "cuda:0")


def _prompt_runs(monkeypatch, capacity, n_seqs, context_limit, heads=25, head_dim=64, bf16=True, window=0, units=256, chunk=0):
    from types import SimpleNamespace
    from burn_transformers_amd.parts import attention
    monkeypatch.setattr(attention, "compute_units", lambda device: units)
    mixer = SimpleNamespace(heads=heads, head_dim=head_dim, window=window, chunk=chunk, plain_only=False)
    step = SimpleNamespace(decode=False, context_limit=context_limit, dtype_is_bf16=bf16, n_seqs=n_seqs,
                           token_capacity=capacity)
    return attention.CausalSelfAttention.prompt_runs(mixer, step, "cuda:0")


def test_prompt_runs_for_chunks_behind_long_contexts(monkeypatch):
    """A chunk of a prompt has few tiles of 128 queries: their keys are cut into runs until the
    work-groups fill the chip, each run at least 8 blocks of keys per 256 tokens of the step, none
    while the class of context is 1,024 tokens or less, and only where the kernel that takes runs
    is the one that runs (bfloat16, heads of 64 to 128, no window)."""
    assert _prompt_runs(monkeypatch, 256, 1, 1024) == 1
    assert _prompt_runs(monkeypatch, 256, 1, 2048) == 4            # 32 blocks in runs of 8
    assert _prompt_runs(monkeypatch, 256, 1, 4096) == 5            # 2 tiles x 25 heads x 5 = 250 work-groups
    assert _prompt_runs(monkeypatch, 256, 1, 8192) == 5
    assert _prompt_runs(monkeypatch, 128, 1, 8192) == 8            # never more than eight
    assert _prompt_runs(monkeypatch, 512, 2, 2048) == 2            # 5 tiles x 25 heads: two runs fit the chip, 16 blocks each
    assert _prompt_runs(monkeypatch, 512, 2, 4096) == 2
    assert _prompt_runs(monkeypatch, 1024, 1, 2048) == 1           # 8 blocks per 256 tokens: 32 a run here
    assert _prompt_runs(monkeypatch, 2048, 1, 8192) == 1           # 16 tiles x 25 heads fill the chip already
    assert _prompt_runs(monkeypatch, 256, 1, 8192, bf16=False) == 1
    assert _prompt_runs(monkeypatch, 256, 1, 8192, head_dim=32) == 1
    assert _prompt_runs(monkeypatch, 256, 1, 8192, head_dim=128) == 5
    assert _prompt_runs(monkeypatch, 256, 1, 8192, head_dim=144) == 1
    assert _prompt_runs(monkeypatch, 256, 1, 8192, window=512) == 1
    assert _prompt_runs(monkeypatch, 256, 1, 8192, chunk=512) == 1
    assert _prompt_runs(monkeypatch, 256, 1, 8192, heads=4) == 8   # few heads: the runs are what fills the chip


def test_decode_runs_at_measured_sizes(monkeypatch):
    # 25 heads of 64: bfloat16 is not cut at 1,024 keys, and best with 4 / 8 runs at 2,048 / 4,096
    assert _runs(monkeypatch, 1, 1024) == 1
    assert _runs(monkeypatch, 1, 2048) == 4
    assert _runs(monkeypatch, 1, 4096) == 8
    assert _runs(monkeypatch, 1, 8192) == 10           # no more work-groups than compute units
    assert _runs(monkeypatch, 4, 8192) == 2
    assert _runs(monkeypatch, 8, 8192) == 1            # 200 pairs of sequence and head fill the chip
    assert _runs(monkeypatch, 64, 8192) == 1
    # float32 holds twice the bytes per key
    assert _runs(monkeypatch, 1, 1024, bf16=False) == 4
    assert _runs(monkeypatch, 8, 1024, bf16=False) == 1
    # a window bounds the keys a query reads; steps with prompt tokens are never cut
    assert _runs(monkeypatch, 1, 8192, window=512) == 1
    assert _runs(monkeypatch, 1, 8192, chunk=512) == 1          # so do chunks
    assert _runs(monkeypatch, 1, 8192, decode=False) == 1


def test_decode_runs_of_wide_heads(monkeypatch):
    """Heads of 128 in bfloat16: eight runs at least, as far as there are compute units."""
    assert _runs(monkeypatch, 8, 1024, kv_heads=2, head_dim=128) == 8
    assert _runs(monkeypatch, 8, 8192, kv_heads=2, head_dim=128) == 16
    assert _runs(monkeypatch, 32, 1024, kv_heads=2, head_dim=128) == 4
    assert _runs(monkeypatch, 200, 1024, kv_heads=2, head_dim=128) == 1
    assert _runs(monkeypatch, 8, 1024, kv_heads=2, head_dim=128, window=512) == 1
    assert _runs(monkeypatch, 8, 1024, kv_heads=2, head_dim=128, bf16=False) == 8      # (by the bytes of a run)


def test_context_classes():
    from burn_transformers_amd.engine.step import StepPlan, context_limit
    assert [context_limit(n) for n in (1, 1024, 1025, 2048, 2049, 5000)] == [1024, 1024, 2048, 2048, 4096, 8192]
    plan = StepPlan([0, 1], [10, 3000], [1, 1], [5, 6], [0, 1], [[[0], list(range(47))]], 128)
    assert plan.context_limit == 4096 and plan.decode
    # never more than a sequence can hold (3 blocks of 64 tokens here)
    assert StepPlan([0], [100], [1], [5], [0], [[[0, 1]]], 3).context_limit == 192


def test_whether_a_graph_pays_is_decided_by_the_median_of_the_measured_steps():
    """``engine.launch_bound``: the GPU is the limit (no graph) when its time for a step stands
    clearly above the host's time for walking the step's launch list; one odd sample of three
    changes nothing."""
    from burn_transformers_amd.engine.engine import launch_bound
    host_bound = (1.00e-3, 0.98e-3)       # the GPU waited for every launch: both times about equal
    gpu_bound = (1.70e-3, 1.30e-3)        # the kernels outlast their launches
    assert launch_bound([gpu_bound] * 3) is True
    assert launch_bound([host_bound] * 3) is False
    assert launch_bound([gpu_bound, host_bound, gpu_bound]) is True
    assert launch_bound([host_bound, (9e-3, 1e-3), host_bound]) is False      # a first use, a clock still rising
    assert launch_bound([gpu_bound, (1e-3, 9e-3), gpu_bound]) is True         # the host was interrupted once
    assert launch_bound([(1.05e-3, 1e-3)]) is False and launch_bound([(1.2e-3, 1e-3)]) is True
    assert launch_bound([(1e-3, 0.0)]) is True                                # never a division by zero


def test_products_of_short_prompts_and_how_they_cut_k():
    """``deep_form_rows`` / ``deep_split_count``: 65 to 256 rows with K a multiple of 64 go to the
    tile kernel, up to 512 where slices of K may stay pending and up to 384 where keys and
    values are scattered into the cache (the vendor's library would need a copy behind it); a residual-writing one
    cuts K so that every work-group has a compute unit, or at most two share one, into at most four
    slices of at least four tiles of K."""
    from burn_transformers_amd.kernels.library import deep_form_rows, deep_split_count
    assert not deep_form_rows(64, 1600, 1600, 4800) and deep_form_rows(65, 1600, 1600, 4800)
    assert deep_form_rows(256, 1600, 1600, 4800) and not deep_form_rows(257, 1600, 1600, 4800)
    assert deep_form_rows(512, 1600, 1600, 1600, sliced=True) and not deep_form_rows(513, 1600, 1600, 1600, sliced=True)
    assert deep_form_rows(384, 1600, 1600, 4800, scatters=True) and not deep_form_rows(385, 1600, 1600, 4800, scatters=True)
    assert not deep_form_rows(128, 1608, 1608, 4800)            # K in tiles of 64
    assert not deep_form_rows(128, 64, 1 << 25, 64)             # operands addressed with 32 bits
    assert deep_split_count(128, 1600, 1600) == 4 and deep_split_count(128, 1600, 6400) == 4
    assert deep_split_count(192, 1600, 1600) == 3 and deep_split_count(192, 1600, 6400) == 3
    assert deep_split_count(256, 1600, 1600) == 2 and deep_split_count(256, 1600, 6400) == 2
    assert deep_split_count(384, 1600, 6400) == 3 and deep_split_count(512, 1600, 6400) == 2     # two work-groups a unit
    assert deep_split_count(128, 768, 768) == 3                 # 12 tiles of K: three slices of four
    assert deep_split_count(100, 64, 64) == 1 and deep_split_count(100, 64, 256) == 1   # K too short to cut
    assert deep_split_count(512, 6400, 1600) == 1               # tiles enough without a cut
    assert deep_split_count(64, 1600, 1600) == 1 and deep_split_count(513, 1600, 1600) == 1
    for rows in (65, 100, 128, 200, 256, 300, 512):
        for columns in (64, 768, 1024, 1600, 50257):
            for k in (64, 128, 768, 1024, 1600, 6400):
                splits = deep_split_count(rows, columns, k)
                assert 1 <= splits <= 4 and (splits == 1 or (k // 64) // splits >= 4)


def test_which_products_leave_the_library_whatever_their_k():
    """A fused projection that scatters keys and values keeps its line where K is long, what adds to the stream does not."""
    from burn_transformers_amd.kernels.library import own_tiles
    for k in (1024, 1984, 2048, 4096):
        assert own_tiles(640, 6144, k, k, scatters=True) and not own_tiles(768, 6144, k, k, scatters=True)     # 480 and 576 tiles of 64 x 128
    assert own_tiles(2048, 2048, 1984, 1984, residual=True) and not own_tiles(2048, 2048, 2048, 2048, residual=True)
    assert own_tiles(512, 2048, 2048, 2048) and not own_tiles(513, 2048, 2048, 2048)
    # the activation that the library has too: while tiles of 64 x 64 have a unit each, or by the rows alone
    assert own_tiles(300, 3072, 768, 768, gelu=True) and own_tiles(400, 3072, 768, 768) and not own_tiles(400, 3072, 768, 768, gelu=True)
    assert own_tiles(256, 6400, 1600, 1600, gelu=True) and not own_tiles(257, 6400, 1600, 1600, gelu=True)


def test_which_products_the_tile_kernel_takes():
    """``tile_kernel_takes``: ``own_tiles``' products and those whose form is the faster way, as measured beside the library; inside what was measured only."""
    from burn_transformers_amd.kernels.library import own_tiles, tile_kernel_takes as takes
    # faster on tiles by a tenth and more, left to the library by own_tiles
    for m, n, k, options in ((400, 3072, 768, {"gelu": True}), (448, 1024, 1024, {"residual": True}), (600, 512, 1024, {}), (1536, 256, 1856, {"residual": True}),
                             (768, 6144, 2048, {"scatters": True}), (2048, 4800, 1600, {"scatters": True}), (632, 3072, 576, {"gelu": True}), (3497, 128, 1536, {"gelu": True}), (6118, 1600, 6400, {})):
        assert takes(m, n, k, k, **options) and not own_tiles(m, n, k, k, **options), (m, n, k)
    # long K in steps of 128 on tiles of 64 x 64, and products that large tiles do not fill well
    for m, n, k, options in ((448, 1024, 2048, {}), (440, 832, 1280, {}), (1318, 192, 1152, {"gelu": True}), (752, 512, 1792, {"residual": True}),
                             (555, 768, 2560, {}), (2048, 128, 2048, {}), (2048, 6400, 1600, {"gelu": True}), (1959, 4096, 1024, {"gelu": True}), (2048, 4096, 1024, {}), (4096, 4096, 1024, {})):
        assert not takes(m, n, k, k, **options), (m, n, k)
    # beyond what the model was held against
    for m in (65, 300, 513, 1024, 2048, 4096):
        for n, k in ((2048, 6464), (2048, 8192), (1024, 16384), (12352, 1024), (50304, 1600), (32000, 1024)):
            for options in ({}, {"scatters": True}, {"residual": True}, {"gelu": True}):
                assert takes(m, n, k, k, **options) == own_tiles(m, n, k, k, **options), (m, n, k, options)
    assert not takes(64, 1024, 1024, 1024) and not takes(566, 1024, 1000, 1000) and not takes(1300, 1604, 1600, 1600)


def test_products_leave_the_library_alike_in_all_steps_of_a_class():
    """One launch list serves all steps of a class: whose product it is, and on which form, may not depend on which of them came first."""
    from burn_transformers_amd.engine.step import token_capacity
    from burn_transformers_amd.kernels.library import own_tiles, tile_form, tile_kernel_takes
    for n, k in ((768, 768), (1600, 1600), (3072, 1024), (4800, 1600), (6144, 2048), (1024, 4096)):
        for options in ({}, {"sliced": True}, {"scatters": True}, {"residual": True}, {"gelu": True}):
            for rows in range(65, 1700):
                capacity = token_capacity(rows)
                assert own_tiles(rows, n, k, k, **options) == own_tiles(capacity, n, k, k, **options)
                assert tile_kernel_takes(rows, n, k, k, **options) == tile_kernel_takes(capacity, n, k, k, **options)
                assert tile_form(-(-rows // 64), n, k) == tile_form(-(-capacity // 64), n, k)


def test_forms_of_the_tile_kernel():
    """Every form chosen is one that the kernel has; of products with few tiles of K the measured ones take the fastest form or one within a twentieth of it."""
    import re
    from burn_transformers_amd.kernels import library as K
    from burn_transformers_amd.kernels.build import CSRC_DIR
    with open(f"{CSRC_DIR}/gemm_mfma.hip") as source:
        forms = source.read().split("static int launch_form(hipStream_t s, int variant, const bf16_t* a", 1)[1].split("unknown form", 1)[0]
    known = {int(number) for number in re.findall(r"case (\d+):", forms)}
    assert set(K.TILE_FORMS) | {4, 5} <= known
    for rows64 in (2, 5, 9, 17, 32, 64):
        for n in (64, 768, 1600, 4800, 8192, 50304):
            for k in (64, 320, 768, 1600, 6400):
                for splits in (1, 2, 4):
                    assert K.tile_form(rows64, n, k, splits)[1] in set(K.TILE_FORMS) | {4, 5}
    for rows, n, k, fast in ((125, 2176, 64, (4, 5)), (1584, 128, 64, (4, 5)), (910, 192, 64, (4, 5)), (66, 384, 192, (4, 5)), (112, 1344, 64, (4, 5)),
                             (2172, 5568, 576, (7, 12, 14)), (2926, 7424, 704, (7, 14)), (1982, 7168, 576, (7, 14)), (3945, 832, 576, (2,)), (1148, 3584, 704, (2,))):
        assert K.tile_form(-(-rows // 64), n, k)[1] in fast, (rows, n, k)


def test_float_products_are_cut_alike_in_all_steps_of_a_class(monkeypatch):
    """One launch list serves all steps of a class, so the slices of a float32 product may not depend on which of them came first."""
    from types import SimpleNamespace
    import torch
    from burn_transformers_amd.engine.step import token_capacity
    from burn_transformers_amd.kernels.library import float_split_count
    from burn_transformers_amd.parts import base
    monkeypatch.setattr(base, "compute_units", lambda device: 256)

    def cuts(rows, columns, k):
        step = SimpleNamespace(dtype_is_bf16=False, n_tokens=rows, token_capacity=token_capacity(rows))
        return base.stream_product_splits(step, torch.empty(rows, k, device="meta"), torch.empty(columns, k, device="meta"))

    asked_exactly = 0
    for columns, k in ((768, 768), (768, 3072), (1024, 1024), (1024, 2048), (1024, 4096), (1600, 1600), (1600, 6400), (2048, 2048)):
        for most in range(128, 2305, 64):
            found = {cuts(rows, columns, k) for rows in range(most - 63, most + 1)}
            assert len(found) == 1, (columns, k, most, found)
            asked_exactly += len({float_split_count(rows, columns, k) for rows in range(most - 63, most + 1)}) > 1
    assert asked_exactly > 0                                            # the rule itself turns within classes


def test_which_experts_run_on_their_rows():
    """Few operations less are no reason to; whatever is decided holds for all steps of a class, whose launch list is one."""
    import torch
    from types import SimpleNamespace
    from burn_transformers_amd.engine.step import token_capacity
    from burn_transformers_amd.kernels import library as K
    from burn_transformers_amd.parts.experts import RoutedExperts

    def way(tokens, experts, top, ff, shared_ff, width, dtype=torch.bfloat16, unit="gated"):
        """True: on their rows, by the calls that the part makes."""
        made = []
        part = RoutedExperts.__new__(RoutedExperts)
        part.__dict__.update(rides=False, experts=experts, identity=0, outputs=experts, top=top, ff=ff, shared_ff=shared_ff, width=width, gated=unit == "gated", unit=unit,
                             shared_mix=None, router=None, correction=None, groups=1, keep=1, score="softmax", group_rank=1, normalize=True, router_bias=None,
                             in_weight=None, down_weight=None, limit=None, alpha=1.0, in_packed=None, down_packed=None, fused_cols=8, hidden_cols=8)
        buffer = lambda key, *sizes: torch.empty(1, device="meta")
        step = SimpleNamespace(n_tokens=tokens, token_capacity=token_capacity(tokens), dtype=dtype, dtype_is_bf16=dtype == torch.bfloat16, buffer=buffer, partial_sums=buffer)
        taken = {}

        class Chosen(Exception):
            pass

        def route(*args, used=None, **more):
            taken["way"] = used is not None
            raise Chosen
        held, K.route = K.route, route
        try:
            part.forward(torch.empty(tokens, width, dtype=dtype, device="meta"), step, None)
        except Chosen:
            pass
        finally:
            K.route = held
        return taken["way"]

    assert not way(64, 8, 2, 1024, 0, 1024) and way(65, 8, 2, 1024, 0, 1024) and way(65, 8, 2, 512, 0, 1024)
    assert not way(200, 4, 1, 512, 0, 512) and way(300, 4, 1, 512, 0, 512)
    assert not way(200, 4, 2, 512, 512, 1024) and way(773, 4, 2, 512, 512, 1024)
    assert not way(400, 8, 2, 128, 0, 256) and way(1100, 8, 2, 128, 0, 256)
    assert not way(100, 16, 4, 256, 256, 1024) and way(200, 16, 4, 256, 256, 1024)
    assert way(65, 64, 4, 64, 0, 256) and way(65, 8, 2, 64, 0, 64, torch.float32) and not way(64, 8, 2, 64, 0, 64, torch.float32)
    for sizes in ((4, 1, 512, 0, 512), (4, 2, 512, 512, 1024), (8, 2, 128, 0, 256), (16, 4, 256, 256, 1024), (8, 2, 512, 0, 1024)):
        for unit in ("gated", "silu"):
            for most in range(128, 1217, 64):
                assert len({way(rows, *sizes, unit=unit) for rows in range(most - 63, most + 1)}) == 1
