"""The host-side choices of kernels and launch shapes (tensorline_amd/ops/kernels.py): pure functions of
the step's facts and the matrices' shapes, checked here without a GPU.  They decide speed, never a
result beyond rounding; what they must keep is stated per test."""
import pytest
import torch

from tensorline_amd.engine.batch import StepFacts
from tensorline_amd.ops import kernels as K


@pytest.fixture
def launches(monkeypatch):
    """Every launch as (entry point, arguments) instead of on a GPU: operands may be CPU or meta tensors."""
    calls = []
    monkeypatch.setattr(K, "_on_gpu", lambda *t: None)
    monkeypatch.setattr(K, "_stream", lambda: None)
    monkeypatch.setattr(K, "_call", lambda name, *args: calls.append((name, args)))
    return calls


def _expert_launches(launches, T, E, top, Kd, F, N):
    """The rows of a tile that each product of an experts' call is launched with; operands without memory."""
    at = lambda *shape, dtype=torch.bfloat16: torch.empty(*shape, dtype=dtype, device="meta")
    launches.clear()
    K.moe_experts(at(T, Kd), at(E, 2 * F, Kd), at(E, N, F), at(T, top, dtype=torch.int32), at(T, top, dtype=torch.float32), 7.0, 1.0)
    return [args[12] for name, args in launches if name == "tl_moe_gemm"]


def test_key_splits_follow_the_batch_and_the_context_and_never_exceed_what_the_merge_takes():
    for seqs in (1, 2, 8, 9, 64, 65, 300):
        for kv in (1, 4, 8):
            last = None
            for ctx in (1, 63, 64, 65, 4096, 4097, 8192, 8193, 32768, 70001, 1 << 20):
                length, n = K._key_splits(seqs, kv, ctx)
                if length == 0:
                    assert n == 1                                   # a large batch fills the GPU unsplit
                    continue
                assert length % 32 == 0 and n == max(1, -(-ctx // length)) and n <= K.MAX_KEY_SPLITS
                assert last is None or length >= last               # longer contexts never get shorter runs
                last = length
    # the runs double where the graphs' context buckets do, and stop at LONG_SPLIT_KEYS until the merge's limit is reached
    assert [K._key_splits(8, 4, c)[0] for c in (4096, 4097, 8193, 16385, 32768, 65536)] == [128, 256, 512, 1024, 1024, 1024]
    assert K._key_splits(1, 4, 4096)[0] == 64 and K._key_splits(64, 4, 4096)[0] == 512
    # fitted to the engine's longest context, a short step cuts as the graph captured for the longest one does
    assert K._fit_key_splits(64, 100, fit_context=1 << 20)[0] == K._fit_key_splits(64, 1 << 20)[0]


def test_splits_of_one_wave_never_touch_more_pages_than_lanes():
    """The decode kernel has a split's page ids one a lane: it takes the splits that touch at most 64 pages wherever they begin."""
    takes = K.library().tl_attention_decode_takes
    for page in (16, 32, 64, 128, 256, 1024):
        for blocks in [*range(1, 40), *range(2 * page - 40, 2 * page + 40)]:
            if blocks < 1:
                continue
            length = 32 * blocks
            touched = max(((i + 1) * length - 1) // page - i * length // page + 1 for i in range(page))
            assert bool(takes(page, blocks)) == (touched <= 64), (page, blocks, touched)
    assert not takes(128, 255) and not takes(256, 511) and takes(128, 256) and takes(128, 254) and takes(64, 127) and takes(16, 32)
    assert not any(takes(page, 4) for page in (8, 24, 48, 0)) and not takes(16, 0)


def test_one_token_sequences_of_a_step():
    mixed = StepFacts(max_context=900, max_query_len=300, decode_only=False, num_seqs=5, q_lens=[300, 1, 1, 7], starts=[600, 40, 0, 3])
    assert K.one_token_sequences(mixed) == [1, 2, 4]                # the padding sequence too
    decode = StepFacts(max_context=900, max_query_len=1, decode_only=True, num_seqs=3, q_lens=[1, 1, 1], starts=[5, 6, 7])
    assert K.one_token_sequences(decode) == []


def test_one_token_sequences_get_a_launch_of_their_own_only_behind_long_contexts():
    def facts(portion, single_ctx, n_single=8):
        return StepFacts(max_context=max(portion, single_ctx), max_query_len=portion, decode_only=False, num_seqs=1 + n_single,
                         q_lens=[portion] + [1] * n_single, starts=[0] + [single_ctx - 1] * n_single)
    singles = list(range(1, 9))
    assert K._singles_get_own_launch(facts(64, 32768), singles, 28, 4, 128, 0)
    assert K._singles_get_own_launch(facts(2040, 32768), singles, 28, 4, 128, 0)
    assert not K._singles_get_own_launch(facts(64, 1000), singles, 28, 4, 128, 0)
    assert not K._singles_get_own_launch(facts(64, 32768), singles, 28, 4, 128, 512)      # a window bounds their walk


def test_prompt_kernels_by_the_shape_of_the_step():
    # 32 columns per wave: thousands of keys per column and columns enough for 128 work-groups of 256
    assert K._tile32_waves([2048], [30720], 28) == 8
    assert K._tile32_waves([2048], [4096], 28) == 8
    assert K._tile32_waves([2048], [0], 28) == 0                    # a fresh prompt: too few keys per column
    assert K._tile32_waves([300], [30720], 28) == 0                 # too few columns
    assert K._tile32_waves([1, 1, 2048], [9, 9, 30720], 28) == 8    # one-token sequences do not count
    assert K._tile32_waves([1, 1], [5, 6], 28) == 0
    # two chains of tiles: at most one work-group per CU and a walk of 16 tiles or more
    assert K._tile16_chains(56, 4, None, 5120) == 2                 # 1,024 tokens behind 4,096 at 28 / 4 heads
    assert K._tile16_chains(112, 4, None, 2048) == 1                # a fresh prompt of 2,048: 448 work-groups
    assert K._tile16_chains(4, 4, None, 300) == 1                   # short walks
    assert K._tile16_chains(112, 4, "mfma-tile16x2") == 2 and K._tile16_chains(1, 1, "mfma-tile16", 1 << 20) == 1


def test_few_row_products_of_long_k_and_an_unfull_last_round_go_to_the_kernel_that_shares_k():
    assert K._few_rows_go_to_rows64(5120, 13824) and K._few_rows_go_to_rows64(5120, 27648)   # the 14B and 32B down projections
    assert not K._few_rows_go_to_rows64(5120, 5120)                 # K too short to pay for a second kernel
    assert not K._few_rows_go_to_rows64(3584, 18944)                # 224 tiles: one round
    assert not K._few_rows_go_to_rows64(152064, 3584)               # many rounds: the last one hardly matters


def test_head_sizes_the_kernels_take():
    assert [d for d in range(1, 300) if K.attention_takes_head_dim(d)] == list(range(16, 257, 16))


def test_launches_worked_out_for_a_step_follow_its_facts():
    """A step's layers share one choice; facts that a caller writes the next step's numbers into get another."""
    key = (2, 28, 4, 128, 0, 0, 0, None, None, None, False)
    facts = StepFacts(max_context=900, max_query_len=300, num_seqs=2, q_lens=[300, 20], starts=[600, 40])
    first = K._worked_out_launch(facts, *key)
    assert K._worked_out_launch(facts, *key) is first and first == K._attention_launch(facts, *key)
    for change in (lambda: facts.q_lens.__setitem__(1, 280), lambda: facts.starts.__setitem__(0, 0),
                   lambda: setattr(facts, "q_lens", [1, 299]), lambda: setattr(facts, "max_query_len", 299),
                   lambda: setattr(facts, "max_context", 8000), lambda: setattr(facts, "num_seqs", 3)):
        change()
        assert K._worked_out_launch(facts, *key) == K._attention_launch(facts, *key)


def test_short_prompts_at_a_head_size_of_256_walk_on_their_own():
    def chains(q_lens, starts=None, heads=(32, 1), path=None, **mask):
        starts = starts or [0] * len(q_lens)
        facts = StepFacts(max_context=max(a + b for a, b in zip(q_lens, starts)), max_query_len=max(q_lens), num_seqs=len(q_lens),
                          q_lens=q_lens, starts=starts)
        m = dict(window=0, keep_first=0, chunk=0) | mask
        return K._attention_launch(facts, len(q_lens), *heads, 256, m["window"], m["keep_first"], m["chunk"], path, None, None, False).chains
    assert chains([17]) == chains([40]) == chains([64]) == chains([17] * 8) == chains([3] * 64) == chains([17], [120]) == 0
    assert chains([130]) and chains([400]) and chains([2048]) and chains([100] * 8) and chains([17], [200])       # long walks, or many columns
    assert chains([17], [200], window=64) == 0                                                  # a window bounds the walk
    assert chains([17], path="mfma-tile16") == 1 and chains([400], path="mfma-direct") == 0
    assert chains([2], [3000]) > 0                                                              # in runs of keys


def test_experts_in_wide_tiles_by_tiles_rows_and_size(launches):
    """The tiles that the products are launched with, by rows an expert, experts, width and the experts' width."""
    def wide(rows, experts, width, ff):
        tiles = set(_expert_launches(launches, rows * experts // 4, experts, 4, width, ff, width))
        assert tiles in ({64}, {256})
        return tiles == {256}
    # large stacks, with tiles for every CU or not
    assert wide(20, 64, 4096, 2048) and wide(20, 64, 2048, 1408) and wide(20, 128, 2048, 768) and wide(20, 128, 2048, 512)
    assert wide(188, 32, 1024, 512) and wide(100, 8, 4096, 2048) and wide(20, 256, 1024, 256) and wide(32, 256, 512, 512) and wide(48, 512, 512, 256)
    # small ones, with twice as many tiles as CUs and many rows, with fewer tiles, with few rows
    assert wide(64, 512, 128, 128) and wide(1100, 16, 512, 1024) and wide(600, 64, 512, 384)
    assert not wide(20, 16, 1024, 512) and not wide(100, 16, 1024, 512) and not wide(200, 8, 1024, 512) and not wide(48, 32, 512, 128)
    assert not wide(60, 512, 128, 128)


def test_many_row_products_are_cut_within_the_tiles_limits():
    plan = K.library().tl_gemm_tiles_plan
    for M, N, Kd in ((65, 64, 64), (512, 37888, 3584), (801, 1536, 8960), (100000, 896, 896), (70, 512, 1 << 16), (2048, 2048, 6144)):
        for gated, takes in ((0, 0), (0, 1), (1, 0)):
            p = plan(M, N, Kd, gated, takes)
            tile, shares = p & 255, p >> 8
            assert 0 <= tile < 8 and 1 <= shares <= 12 and shares <= max(1, Kd // 256) and not (gated and (shares > 1 or tile == 1))
            assert gated or tile != 7
    for M, N, Kd, gated in ((70, 64, 96, 0), (70, 66, 64, 0), (70, 48, 64, 1), (70, 1 << 17, 1 << 15, 0), (0, 64, 64, 0), (513, 3584, 3584, 0)):
        assert plan(M, N, Kd, gated, 0) == -1
    # what is launched is what the plan says: gated products of more such tiles than CUs with their matrix in registers where that is ahead
    for M, N, Kd, tile in ((801, 17920, 1536, 7), (2048, 17920, 1536, 7), (380, 37888, 3584, 7), (1521, 9728, 896, 0), (1300, 17920, 1536, 6),
                           (513, 17920, 1536, 6), (300, 17920, 1536, 2), (65280, 32, 64, 3)):
        assert plan(M, N, Kd, 1, 0) == 256 + tile, (M, N, Kd)


def test_a_many_row_product_with_an_activation_refuses_a_wrong_bias(launches):
    """The product with relu squared in its epilogue takes the biases that the one without takes: float32, contiguous, N entries."""
    a, w = torch.zeros(100, 256, dtype=torch.bfloat16), torch.zeros(512, 256, dtype=torch.bfloat16)
    sh = K.shuffle_weight(w)
    for bias in (torch.zeros(3), torch.zeros(512, dtype=torch.bfloat16), torch.zeros(1024)[::2], torch.zeros(513)):
        for act in ("relu2", None):
            with pytest.raises(K.KernelError, match="bias must be float32 of 512"):
                K.linear(a, w, bias, shuffled=sh, act=act)
    assert not launches
    K.linear(a, w, torch.zeros(512), shuffled=sh, act="relu2")
    assert [name for name, _ in launches] == ["tl_gemm_tiles"]


def test_many_row_products_take_and_refuse_the_matrices_that_the_other_ways_do(launches, monkeypatch):
    """More than 64 rows: a weight of another type, shape or layout is no business of the tiles whatever its copy says, and a copy
    of another matrix, or a result in another type, goes the way that does not look at the copy."""
    monkeypatch.setattr(K, "_library_linear", lambda a, weight, bias, out_dtype, keep_shares=False: launches.append(("library", ()))
                        or torch.empty(a.shape[0], weight.shape[0], dtype=out_dtype))
    a, w = torch.zeros(100, 256, dtype=torch.bfloat16), torch.zeros(512, 256, dtype=torch.bfloat16)
    sh, other = K.shuffle_weight(w), K.shuffle_weight(w[:256])
    names = lambda: [name for name, _ in launches]

    def run(weight, copy):
        for call in (lambda: K.linear(a, weight, None, shuffled=copy), lambda: K.linear(a, weight, None, shuffled=copy, act="relu2"),
                     lambda: K.swiglu_gate_up(a, weight, copy), lambda: K.swiglu_gate_up(a, weight, copy, activation="gelu_tanh")):
            launches.clear()
            try:
                call()
            except K.KernelError:
                yield "refused"
                continue
            yield names()[0]
    assert list(run(w, sh)) == ["tl_gemm_tiles"] * 4
    assert list(run(w, other)) == ["library", "library", "refused", "library"]
    assert list(run(w.float(), sh)) == ["tl_gemm_generic"] * 4                       # (which refuses the pair of types)
    assert list(run(torch.zeros(512, 512, dtype=torch.bfloat16)[:, ::2], sh)) == ["refused"] * 4
    assert list(run(torch.zeros(512, 1, 256, dtype=torch.bfloat16), sh)) == ["refused"] * 4
    launches.clear()
    assert K.linear(a, w, None, out_dtype=torch.float16, shuffled=sh).dtype == torch.float16 and names() == ["library"]


def test_experts_whose_result_is_no_whole_quads_stay_in_tiles_of_64_rows(launches):
    assert _expert_launches(launches, 600, 16, 2, 1024, 1024, 1024) == _expert_launches(launches, 600, 16, 2, 1024, 1024, 68) == [256, 256]
    assert all(_expert_launches(launches, 600, 16, 2, 1024, 1024, n) == [64, 64] for n in (66, 1023, 1, 1025))


def test_rows_beyond_the_wide_tiles_reach_go_in_passes(launches):
    """Wide tiles whatever the number of pairs: in passes over the tokens whose rows 32-bit offsets reach, and whose tiles one launch
    takes (tiles of 64 rows would be too many of them)."""
    E, top, Kd, F = 64, 8, 1024, 512
    for T in (240_000, 600_000):
        assert set(_expert_launches(launches, T, E, top, Kd, F, 1024)) == {256}
        sorts, products = [a for n, a in launches if n == "tl_moe_sort"], [a for n, a in launches if n == "tl_moe_gemm"]
        assert sum(a[3] for a in sorts) == T * top and len(products) == 2 * len(sorts) and len(sorts) == (1 if T < 250_000 else 3)
        assert all((a[10] * 256 + 256) * a[2] * 2 < 4e9 and a[10] <= 65535 for a in products)       # what tl_moe_gemm asks for
        assert sum(a[6] for n, a in launches if n == "tl_moe_combine") == T


def test_the_library_is_searched_for_its_own_products_only(launches, monkeypatch):
    """What runs on the many-row tiles is not searched: with the copy that the program calls it with, in the form it has."""
    class Tunable:
        def __getattr__(self, name):
            return lambda *a: None
    searched = []
    monkeypatch.setattr(torch.cuda, "tunable", Tunable())
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(K, "_keep_tuning_records_out_of_the_way", lambda tn: None)
    monkeypatch.setattr(K, "_library_linear", lambda a, weight, bias, out_dtype: searched.append((a.shape[0], *weight.shape)))
    matrix = lambda N, Kd: torch.zeros(N, Kd, dtype=torch.bfloat16)
    w, odd, narrow = matrix(512, 256), matrix(512, 120), matrix(80, 256)
    for rows, weight, copy, form, is_searched in ((100, w, True, "plain", False), (100, w, True, "gated", False), (100, w, True, "relu2", False),
                                                  (100, w, False, "plain", True), (100, odd, True, "plain", True), (64, w, True, "plain", False),
                                                  (100, narrow, True, "plain", False), (100, narrow, True, "gated", True)):      # 40 pairs: no whole blocks
        searched.clear()
        got = K.tune_library_linear(rows, weight, torch.float32, 2.0, K.shuffle_weight(weight) if copy else None, form)
        assert got is is_searched and searched == ([(rows, *weight.shape)] if is_searched else []), (rows, tuple(weight.shape), copy, form)
    assert K.tune_library_linear(100, w, torch.float32) and not launches            # without a copy, as ever


def test_products_bound_by_their_weights_take_the_tiles_that_keep_the_cus_least_busy():
    """A head's matrix is read from memory once whatever the tile: no more rows in a tile than there are."""
    plan = K.library().tl_gemm_tiles_plan
    for N, Kd in ((152064, 3584), (151936, 1536), (131072, 5120)):
        assert all(plan(M, N, Kd, 0, 0) == 256 + 2 for M in (65, 96, 128)) and plan(192, N, Kd, 0, 0) == 256 + 6      # of 128 and 192 rows


def test_heads_have_the_lanes_that_are_faster():
    """Rows of heads past 128, a few heads and small steps: 64 lanes a head; many heads of up to 128: sixteen."""
    lanes = K.library().tl_head_lanes
    for T, units, D in ((128, 12, 256), (2048, 12, 256), (2048, 40, 256), (2048, 32, 192), (2048, 5, 64), (512, 5, 128), (128, 16, 64), (200, 12, 128),
                        (100, 64, 128), (1, 40, 128)):
        assert lanes(T, units, D) == 64, (T, units, D)
    for T, units, D in ((512, 16, 64), (512, 12, 128), (160, 36, 128), (200, 24, 128), (2048, 7, 64), (2048, 48, 96)):
        assert lanes(T, units, D) == 16, (T, units, D)


def test_recurrences_have_helping_waves_where_that_is_faster():
    """One to a CU (a decay per channel, keys past 64): a second round of work-groups only beside one long sequence."""
    helps = lambda lens, H, dk, dv, form: K.library().tl_linear_recurrence_helps(len(lens), sum(lens), max(lens), H, dk, dv, form)
    for lens, H, dk, dv in (([40] * 4, 16, 128, 128), ([17] * 8, 8, 96, 96), ([64] * 16, 8, 128, 64), ([1] * 15 + [20], 8, 128, 64), ([19, 19, 13, 2], 16, 128, 128),
                            ([1, 4, 17], 16, 80, 128), ([500] * 4, 16, 128, 128), ([600, 600, 600, 120], 16, 128, 128)):
        assert not helps(lens, H, dk, dv, 1), (lens, H, dk, dv)
        assert helps(lens, H, dk, dv, 0) and helps(lens, H, dk, dv, 2) and helps(lens, H, 64, dv, 1)
    for lens, H, dk, dv in (([17], 16, 128, 128), ([803, 211, 507], 16, 128, 128), ([75, 218, 686, 311], 16, 128, 128), ([40] * 4, 8, 96, 96)):
        assert helps(lens, H, dk, dv, 1), (lens, H, dk, dv)
    for form in (0, 1, 2):
        assert not helps([16] * 4, 4, 64, 64, form) and not helps([300], 4, 144, 64, form) and not helps([40] * 40, 16, 64, 128, form)
        assert not K.library().tl_linear_recurrence_helps(1, 100, 0, 4, 64, 64, form)


def test_products_per_head_have_tall_waves_where_rows_fill_them():
    """64 rows a wave: not for few rows, whatever the batch, nor for three work-groups' rows, nor where waves are few."""
    tall = K.library().tl_gemm_batched_tall
    for M, N, Kd, batch in ((1, 1024, 1024, 16), (17, 1024, 1024, 16), (64, 256, 1024, 64), (96, 512, 512, 32), (300, 1024, 1024, 16), (384, 256, 1024, 64), (600, 192, 128, 32),
                            (128, 128, 512, 32), (2048, 96, 64, 4)):
        assert not tall(M, N, Kd, batch), (M, N, Kd, batch)
    for M, N, Kd, batch in ((128, 1024, 1024, 16), (256, 512, 512, 32), (300, 2048, 1024, 4), (400, 1024, 768, 16), (600, 1024, 1024, 16), (2048, 192, 128, 32), (2049, 128, 192, 32)):
        assert tall(M, N, Kd, batch), (M, N, Kd, batch)
