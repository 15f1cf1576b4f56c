"""Kernel-selection rules of the op layer that are plain functions of the shape (no GPU needed)."""
from llm_consensus_amd import ops
from llm_consensus_amd.models.config import get_preset


def gate_up_cols(name):
    return 2 * get_preset(name).intermediate_size


def test_wide_panel_workgroups_only_where_they_save_a_round():
    """160-column workgroups are for matrices of 257-320 column tiles of 128 whose K is not split:
    among the served models that is Qwen2.5-7B's gate/up projection (296 tiles -> 237 workgroups).
    Narrower matrices fit one round anyway, much wider ones need several rounds either way, and
    the rule stops at the panel kernel's 256 rows."""
    q, l = get_preset("qwen2.5-7b"), get_preset("llama-3-8b")
    assert gate_up_cols("qwen2.5-7b") // 128 == 296
    for rows in (1, 32, 64, 128, 256):
        assert ops.use_wide_panel(rows, gate_up_cols("qwen2.5-7b"), q.hidden_size)
        assert not ops.use_wide_panel(rows, gate_up_cols("llama-3-8b"), l.hidden_size)       # 224 tiles
        assert not ops.use_wide_panel(rows, l.vocab_size, l.hidden_size)                     # 1002 tiles
        assert not ops.use_wide_panel(rows, q.vocab_size, q.hidden_size)                     # 1188 tiles
        assert not ops.use_wide_panel(rows, 6144, 4096)                                      # QKV: K is split
    assert not ops.use_wide_panel(300, gate_up_cols("qwen2.5-7b"), q.hidden_size)
    assert ops.use_wide_panel(64, 320 * 128, 4096) and not ops.use_wide_panel(64, 321 * 128, 4096)


def test_four_wave_prefill_gemm_for_long_reductions_only():
    """The four-wave 256 x 256 kernel wins where its longer prologue is spread over many K-tiles
    (measured: K = 14336 +3 %, K = 4096 -1..-4 %): the down projections take it, the projections
    whose reduction runs over d_model do not, and fp32 outputs (split-K slabs) never do."""
    for name in ("llama-3-8b", "qwen2.5-7b", "mistral-7b", "llama-3-70b"):
        c = get_preset(name)
        assert ops.use_four_wave_gemm(c.intermediate_size)          # down: K = intermediate size
        assert not ops.use_four_wave_gemm(c.hidden_size) or c.hidden_size >= 8192   # QKV / O / gate-up
        assert not ops.use_four_wave_gemm(c.intermediate_size, out_f32=True)
    assert not ops.use_four_wave_gemm(4096) and ops.use_four_wave_gemm(8192)


def test_the_kernel_of_a_few_rows_is_never_handed_more_than_it_holds(monkeypatch):
    """Whatever the most rows it may take is set to (wide outputs over a short depth go to twice that), and where a split is forced."""
    for most, force in ((8, -1), (33, -1), (64, -1), (200, -1), (8, 2)):
        monkeypatch.setattr(ops, "KGEMM_MAX_M", most)
        monkeypatch.setattr(ops, "KGEMM_SHORT_K_MAX_M", 2 * most)
        monkeypatch.setattr(ops, "KGEMM_FORCE_NTW", force)
        for swiglu in (False, True):
            for n_pad, k in ((4096, 4096), (8320, 2048), (28672, 4096), (128256, 2048)):
                assert all(ops._kgemm_ntw(n_pad, rows, swiglu, k) == 0 for rows in (65, 100, 128, 256))


def test_wide_outputs_of_few_rows_go_by_their_depth():
    """Outputs of more than 8192 columns split their depth over the waves of a workgroup unless it is too short for eight waves, or
    long with more than four rows; narrower outputs do at any depth up to the long ones."""
    assert [ops._kgemm_ntw(28672, 1, False, k) > 0 for k in (64, 192, 256, 2048, 4096, 8192)] == [False, False, True, True, True, True]
    assert [ops._kgemm_ntw(28672, 1, True, k) > 0 for k in (64, 256, 512, 4096)] == [False, False, True, True]
    assert [ops._kgemm_ntw(9216, rows, False, 8192) > 0 for rows in (1, 4, 5, 8)] == [True, True, False, False]
    assert all(ops._kgemm_ntw(8192, 8, False, k) > 0 for k in (64, 2048, 8192))


def test_gemm256_plan_stays_within_its_kernels():
    """Every height is one that the kernel has, splits are whole numbers of at least eight K-tiles within one round, and the four-wave
    kernel comes up only where its depth allows it."""
    for M in (1, 129, 257, 300, 513, 1500, 2048, 2361, 3001, 7072, 8192, 40000):
        for n_pad in (256, 512, 2048, 2304, 8448, 28672, 152064):
            for K in (64, 192, 512, 2048, 3584, 8192, 14336):
                for four in (False, True):
                    f, s, us = ops._gemm256_plan(M, n_pad, K, 2, False, 8, four, False)
                    tiles = (n_pad // 256) * -(-M // (32 * f or 256))
                    assert f in (4, 5, 6, 7, 8) or (f == 0 and four and s == 1)
                    assert s == 1 or (tiles * s <= 256 and (K // 64) % s == 0 and K // 64 // s >= 8)
                    assert us > 0
    assert ops._gemm256_plan(3001, 2048, 8192, 4, True, 8, False, True)[0] == 8
    # 320 tiles of 256 rows are a round and a quarter; lower tiles fill two rounds that are shorter
    assert ops._gemm256_plan(2361, 8192, 2048, 2, False, 8, False, False)[0] < 8


def test_strip_splits_stay_within_a_round():
    for n_pad in (128, 1024, 2048, 3584, 4096, 4608, 6144, 8192, 12288, 16384, 28672):
        for K in (64, 512, 896, 2048, 3584, 8192, 14336, 18944):
            tiles, s = ops._strip_splits(n_pad, K)
            assert tiles in (2, 4) and n_pad % (16 * tiles) == 0
            assert s == 1 or ((n_pad // (16 * tiles)) * s <= 256 and (K // 64) % s == 0 and K // 64 // s >= 4)
