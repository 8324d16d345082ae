"""Which calls take a kernel in a library call's place."""
import pytest
import torch
import torch.autograd.forward_ad as fwd
from torch.fx.experimental.proxy_tensor import make_fx
from torch.overrides import TorchFunctionMode
from torch.utils.flop_counter import FlopCounterMode

from nanorlhf_amd import ops
from nanorlhf_amd.ops.linear import plain_call


def test_plain_calls_are_those_that_nobody_sees():
    x, seen = torch.randn(2, 2), []

    class Listens(TorchFunctionMode):
        def __torch_function__(self, fn, types, args=(), kwargs=None):
            return fn(*args, **(kwargs or {}))

    def call(a):
        seen.append(plain_call(a))
        return a + 1

    assert not plain_call(x)                        # gradients are on
    with torch.no_grad():
        for pre_dispatch in (False, True):
            make_fx(call, pre_dispatch=pre_dispatch)(x)
        torch.jit.trace(call, x, check_trace=False)
        torch.func.vmap(call)(x)
        for mode in (FlopCounterMode(display=False), Listens()):
            with mode:
                call(x)
        with fwd.dual_level():
            call(x)
        assert seen and not any(seen)
        assert not plain_call(x.as_subclass(type("Sub", (torch.Tensor,), {})))
        assert plain_call(x, torch.nn.Parameter(x))
        with torch.device("cpu"):                   # only says where new tensors go
            assert plain_call(x)


def test_big_tiles_of_the_adapter_product_stop_where_offsets_end():
    if not ops.ext_available():
        pytest.skip("extensions are not built")
    big = ops.ext().lora_gemm_big
    assert big(4096, 1536, 1536) and not big(4096, 1280, 1536)
    assert big(24576, 256, (1 << 22) - 64) and not big(24576, 256, 1 << 22)
    tiles = ops.ext().lora_gemm_tiles                   # of the kernel that runs
    for rows in (129, 24576):
        assert tiles(rows, 64) == tiles(rows, (1 << 22) - 64) == 256
        assert tiles(rows, 1 << 22) == tiles(128, 64) == 128


def test_adapter_products_of_one_round_by_one_rule():
    """What is called "fused" without a timing is what the kernel's own choice makes of it."""
    if not ops.ext_available():
        pytest.skip("extensions are not built")
    from nanorlhf_amd.ops.lora import one_round
    seen = set()
    for M in (1, 64, 65, 128, 129, 896, 897, 999, 1000, 1152, 1153, 2048, 2049, 4000, 16384, 16385, 32769):
        for N in (8, 64, 65, 128, 129, 896, 1024, 1025, 1536, 2048, 8192, 16384, 16385, 32768, 32769):
            for K in (64, 2048, 2112, 4864, 9728, 10176, 10240, 16384, 16448, 17920, (1 << 22) - 64,
                      1 << 22, (1 << 24) - 64, 1 << 24):
                assert one_round(M, N, K) == ops.ext().lora_gemm_round(M, N, K), (M, N, K)
                seen.add(one_round(M, N, K))
    assert seen == {0, 64, 128} and one_round(4000, 64, 1536) == 64


def test_activations_behind_an_adapter_s_product_by_rows_and_depth():
    from nanorlhf_amd.ops.lora import glu_keeps
    for M, N, K in [(129, 17920, 1536), (46673, 17920, 1536), (13000, 9728, 896), (700, 22016, 2048)]:
        assert glu_keeps(M, N, K)
    # another kernel's rows, blocks, tiles of 128, odd columns, and depths where a pass is as fast
    for M, N, K in [(128, 37888, 1536), (212, 4096, 896), (300, 9728, 896), (13000, 17924, 1536),
                    (13000, 37888, 3584), (2667, 17920, 2112)]:
        assert not glu_keeps(M, N, K)


def test_adapter_strategies_are_kept_by_what_the_kernels_depend_on(monkeypatch):
    from types import SimpleNamespace
    from nanorlhf_amd.ops import lora
    monkeypatch.setattr(lora, "_TUNE", {})
    monkeypatch.setattr(lora, "ext", lambda: SimpleNamespace(
        lora_gemm_tiles=lambda M, K: 256 if M > 128 else 128,
        lora_gemm_big=lambda M, N, K: M > 1000, lora_gemm=None, lora_add_=None))
    # fused, epilogue of each new key
    times = iter([1.0, 3.0, 3.0, 1.0, 1.0, 3.0, 3.0, 1.0, 3.0, 1.0])
    monkeypatch.setattr(lora, "_time_cuda", lambda fn: next(times))
    w, bias = torch.zeros(64, 64), torch.zeros(64)

    def choose(rows, b=None):
        return lora._choose_strategy(torch.zeros(rows, 64), w, None, None, b)

    assert [choose(240), choose(4000), choose(240, bias)] == ["fused", "epilogue", "fused"]
    assert [choose(129), choose(9000), choose(500, bias)] == ["fused", "epilogue", "fused"]
    assert len(lora._TUNE[64, 64]) == 3
    # up to 128 rows are another kernel's, whose time is its own
    assert [choose(60), choose(60, bias)] == ["epilogue", "epilogue"]
    assert [choose(17), choose(128, bias), choose(240)] == ["epilogue", "epilogue", "fused"]
    assert next(times, None) is None and len(lora._TUNE[64, 64]) == 5


@pytest.mark.parametrize("K,rule", [(64, "fused"), (4096, "fused"), (4160, "epilogue"),
                                    (8960, "epilogue")])
def test_near_ties_of_the_adapter_strategies_do_not_hang_on_the_timer(monkeypatch, K, rule):
    from types import SimpleNamespace
    from nanorlhf_amd.ops import lora
    monkeypatch.setattr(lora, "ext", lambda: SimpleNamespace(
        lora_gemm_tiles=lambda M, K: 256, lora_gemm_big=lambda M, N, K: True, lora_gemm=None,
        lora_add_=None))
    w, x = torch.zeros(64, K), torch.zeros(300, K)
    # fused against epilogue
    for ratio, want in [(0.95, rule), (1.0, rule), (1.05, rule), (0.5, "fused"), (2.0, "epilogue")]:
        monkeypatch.setattr(lora, "_TUNE", {})
        times = iter([ratio, 1.0])
        monkeypatch.setattr(lora, "_time_cuda", lambda fn: next(times))
        assert lora._choose_strategy(x, w, None, None, None) == want


def test_a_capture_takes_the_strategy_that_is_known_of_its_weight(monkeypatch):
    from types import SimpleNamespace
    from nanorlhf_amd.ops import lora
    monkeypatch.setattr(lora, "_TUNE", {})
    monkeypatch.setattr(lora, "ext", lambda: SimpleNamespace(
        lora_gemm_tiles=lambda M, K: 256 if M > 128 else 128,
        lora_gemm_big=lambda M, N, K: M > 1000, lora_gemm=None, lora_add_=None))
    times = iter([3.0, 1.0])
    monkeypatch.setattr(lora, "_time_cuda", lambda fn: next(times))
    w = torch.zeros(64, 64)
    assert lora._choose_strategy(torch.zeros(240, 64), w, None, None, None) == "epilogue"
    monkeypatch.setattr(lora, "_capturing", lambda x: True)
    assert lora._choose_strategy(torch.zeros(4000, 64), w, None, None, None) == "epilogue"
    assert len(lora._TUNE[64, 64]) == 1         # and leaves the timing for later


def test_a_rule_s_strategy_is_not_taken_for_a_measured_one(monkeypatch):
    from types import SimpleNamespace
    from nanorlhf_amd.ops import lora
    monkeypatch.setattr(lora, "_TUNE", {})
    monkeypatch.setattr(lora, "ext", lambda: SimpleNamespace(
        lora_gemm_tiles=lambda M, K: 256 if M > 128 else 128,
        lora_gemm_big=lambda M, N, K: M > 1000, lora_gemm=None, lora_add_=None))
    w = torch.empty(1, dtype=torch.bfloat16)

    def known(rows, N, K):
        return lora._known_strategy(w.expand(rows, K), w.expand(N, K), None)

    # blocks, tiles of 128, and more rows of the weight whose 100 rows are timed
    for rows, N, K in [(64, 3000, 8960), (1024, 1536, 17920), (300, 9216, 2048)]:
        assert known(rows, N, K) == "fused"
    assert known(100, 9216, 12288) is None
    known(200, 9216, 12288)
    assert known(100, 9216, 12288) is None and not any(lora._TUNE.values())
    # nor does a capture that has nothing measured try to time: it takes the rule of the depth
    monkeypatch.setattr(lora, "_capturing", lambda x: True)
    for K, want in [(2048, "fused"), (8960, "epilogue")]:
        x = w.expand(4000, K)
        assert known(64, 3000, K) == "fused"
        assert lora._choose_strategy(x, w.expand(3000, K), None, None, None) == want


def test_linears_of_few_rows_leave_what_the_library_does_faster():
    from nanorlhf_amd.ops.linear import rows_pay
    for M, N, K in [(1, 1536, 1536), (64, 16384, 2048), (32, 32768, 1536), (16, 18944, 1536),
                    (64, 151936, 1536), (64, 3584, 18944), (16, 14336, 4096)]:
        assert rows_pay(M, N, K)
    for M, N, K in [(33, 32768, 1536), (17, 18944, 1536), (17, 14336, 4096), (1, 6144, 8192)]:
        assert not rows_pay(M, N, K)


def test_operands_of_a_product_are_looked_at_once(monkeypatch):
    import sys
    linear = sys.modules["nanorlhf_amd.ops.linear"]
    asked = []
    monkeypatch.setattr(linear, "_plain_operands", lambda x, w: asked.append(x.shape[0]))
    table, w = ops.build_rope_cache(64, 10), torch.zeros(192, 896)
    # few rows, blocks of 64, tiles of 128 and of 256, and sizes that the library takes anyway
    rows = [4, 130, 8192, 60000]
    with torch.no_grad():
        for M in (*rows, 1500):
            x = torch.zeros(M, 896)
            ops.linear(x, w), ops.linear_parts(x, w)
            ops.linear_qkv_rope(x, w, None, table, torch.zeros(M, dtype=torch.int64), 1, 1)
    assert asked == [M for M in rows for _ in range(3)]
    with torch.no_grad():
        for M in rows[1:]:
            ops.linear(torch.zeros(M, 896), w, None, routed=True)      # the library's anyway
    assert len(asked) == 12


def test_what_an_autograd_function_has_to_see():
    from nanorlhf_amd.ops.linear import differentiated
    x, y = torch.zeros(2), torch.zeros(2, requires_grad=True)
    assert not differentiated(x) and differentiated(x, y)
    with torch.no_grad():
        assert not differentiated(x, y)
        with torch.autograd.forward_ad.dual_level():
            assert differentiated(x)
    seen = []
    torch.func.vmap(lambda t: seen.append(differentiated(t)) or t)(torch.zeros(3, 2))
    assert seen == [True]
    with torch.no_grad():                            # a trace keeps functions, not kernels' calls
        torch.jit.trace(lambda t: seen.append(differentiated(t)) or t + 1, x, check_trace=False)
    assert seen == [True] * 2


def test_products_in_blocks_are_one_round_and_deep_ones_full():
    from nanorlhf_amd.ops.linear import blocks_fill, blocks_pay
    for M, N, K in [(65, 64, 64), (512, 2048, 1536), (896, 1152, 896), (1152, 896, 4864),
                    (212, 1536, 8960), (66, 3584, 18944), (130, 1024, 4096)]:
        assert blocks_fill(M, N) and blocks_pay(M, N, K)
    for M, N, K in [(513, 2048, 1536), (897, 1152, 896), (1153, 64, 1536), (65, 9728, 896),
                    (130, 1536, 8960), (66, 896, 4864)]:
        assert not blocks_pay(M, N, K)
    assert blocks_fill(130, 1536) and not blocks_fill(897, 1152)


def test_a_linear_s_route_where_tiles_are_in_part_empty():
    """What is the library's by one rule is not taken by the next one."""
    from nanorlhf_amd.ops.linear import linear_route
    for sizes, want in [
            # few rows of many columns
            ([(1, 1536, 1536), (64, 16384, 2048), (64, 151936, 2048)], "linear_rows"),
            ([(33, 32768, 1536), (17, 18944, 1536), (33, 65536, 1536), (64, 40960, 896)], None),
            ([(33, 32768, 1024), (17, 18944, 896), (65, 18944, 1536)], "linear_mid"),
            ([(65, 151936, 1536), (255, 128100, 2048), (33, 65536, 896), (96, 49152, 1024)], "linear_big"),
            ([(129, 32768, 1024), (256, 32768, 896), (129, 8960, 2048), (100, 16384, 2048)], None),
            # a last row of tiles that is half there or less, and more
            ([(257, 151936, 1536), (384, 65536, 896), (513, 24576, 1536), (640, 128100, 2048)], None),
            ([(385, 65536, 896), (641, 128100, 2048), (769, 32768, 1536)], "linear_big"),
            # many rows of few columns
            ([(46673, 4, 896), (46673, 128, 1024), (64000, 1024, 1024), (64000, 512, 896),
              (16400, 4, 2048), (30000, 128, 1536)], None),
            ([(16400, 4, 896), (30000, 128, 1024), (9000, 256, 1536)], "linear_mid"),
            ([(46673, 192, 896), (46673, 1152, 896), (64000, 3072, 1024), (64000, 640, 1536)],
             "linear_big")]:
        for M, N, K in sizes:
            assert linear_route(M, N, K) == want, (M, N, K)


def test_products_in_tiles_of_128_are_half_a_round_to_one():
    from nanorlhf_amd.ops.linear import mid_fills, mid_pays
    for M, N, K in [(1921, 1152, 896), (3584, 1152, 896), (2048, 2048, 2048)]:
        assert mid_pays(M, N, K)
    for M, N, K in [(1000, 1152, 896), (3585, 1152, 896), (2048, 2048, 2112), (2049, 2048, 1536)]:
        assert not mid_pays(M, N, K)
    assert mid_fills(1, 1, 0.0) and not mid_fills(1, 1, 0.5)
    from nanorlhf_amd.ops.lora import _mid             # of an adapter's product
    for M, N, K in [(900, 1536, 2048), (1024, 1536, 17920), (1025, 896, 896)]:
        assert _mid(M, N, K)
    for M, N, K in [(896, 1536, 17920), (1800, 1536, 8960), (3585, 1152, 896)]:
        assert not _mid(M, N, K)
    # deep ones only where the library's kernels were seen to be slow
    for M, N, K in [(1300, 1536, 10240), (2667, 1536, 16384), (999, 3584, 17920), (1800, 896, 17920)]:
        assert not _mid(M, N, K)
    assert _mid(1000, 3584, 18944) and _mid(1000, 1536, 16448)


def test_large_products_by_rounds_and_depth():
    from nanorlhf_amd.ops.linear import big_pays
    for M, N, K in [(5888, 1152, 896), (8192, 2048, 1536), (11009, 1536, 10496), (52000, 1536, 12288)]:
        assert big_pays(M, N, K)
    for M, N, K in [(4000, 1152, 896), (8192, 1792, 1536), (60000, 1536, 8960), (10700, 1536, 10496),
                    (60000, 1536, 10496), (60000, 1024, 4096)]:
        assert not big_pays(M, N, K)


def test_gated_products_of_fewer_rows():
    from nanorlhf_amd.ops.swiglu import glu_pays
    for M, I, K in [(192, 4608, 896), (212, 8960, 1536), (300, 4864, 896), (400, 8960, 1536),
                    (600, 8960, 1536)]:
        assert glu_pays(M, I, K)
    for M, I, K in [(191, 4864, 896), (212, 4096, 1024), (328, 8960, 1536), (384, 8960, 1536)]:
        assert not glu_pays(M, I, K)
    # the last 256 rows of deeper ones more than half there, and tiles enough
    for M, I, K in [(385, 8960, 1536), (511, 6144, 2048), (192, 8960, 2048), (500, 4608, 1536)]:
        assert glu_pays(M, I, K)
    for M, I, K in [(192, 6144, 1536), (256, 8832, 1536), (256, 4608, 1088)]:
        assert not glu_pays(M, I, K)


def test_gated_products_fuse_where_their_tiles_fill_the_gpu():
    from nanorlhf_amd.ops.swiglu import glu_fills
    for M, I, K in [(512, 4864, 896), (600, 8960, 1536), (16320, 8960, 1536), (512, 200, 128)]:
        assert glu_fills(M, I, K)
    for M, I, K in [(512, 1024, 1536), (1024, 2240, 1536), (600, 11008, 2048)]:
        assert not glu_fills(M, I, K)


def test_adapter_gradients_take_the_kernel_by_columns_and_rows():
    from nanorlhf_amd.ops.lora import _fast_grad
    z = torch.empty(1, dtype=torch.bfloat16)
    with torch.no_grad():
        assert _fast_grad(z.expand(50000, 17920)) and _fast_grad(z.expand(240, 37888))
        assert not _fast_grad(z.expand(4096, 37888)) and not _fast_grad(z.expand(64, 36))
        assert not _fast_grad(z.float().expand(64, 64))
    assert not _fast_grad(z.expand(64, 64))            # a recorded backward


def test_gradients_of_keys_and_values_are_divided_where_that_pays():
    if not ops.ext_available():
        pytest.skip("extensions are not built")

    def parts(heads, lens, D=128):
        return ops.ext().fa_bwd_parts(sum(lens), len(lens), *heads, D, max(lens))

    small, large = (12, 2), (28, 4)
    assert parts(small, [870] * 56) == 1 and parts(small, [3000] * 8) == 2
    assert [parts(small, [6000] * n) for n in (2, 3, 4, 5)] == [6, 3, 3, 2]
    assert parts(small, [8000] * 2 + [3000] * 6) == parts(small, [7900] + [600] * 30) == 3
    assert parts(large, [6000] * 5) == parts(large, [8000] * 4) == 1
    assert parts(large, [10000, 4000, 5000, 7000, 8300]) == 1        # 1088 workgroups undivided
    assert parts(large, [8500, 4500, 5000, 6900]) == parts(large, [7900] + [600] * 30) == 7
    assert [parts((14, 2), [6000] * n, 64) for n in (9, 12)] == [7, 1]
    assert parts((16, 16), [6000]) == 1 and parts(large, [6000] + [1] * 300000) == 1
    # what the parts take: float32 sums of both for every token and part
    for n in range(1, 200):
        for heads in (small, large, (32, 8), (40, 8)):
            lens = [8000] + [100 * n] * n
            p = parts(heads, lens)
            assert p == 1 or 2 * p * sum(lens) * heads[1] * 128 * 4 <= 7 * 1100 * 128 * 128 * 8


def test_windows_of_heads_have_places_that_fit_32_bits():
    """The kernels number heads * tiles workgroups in unsigned."""
    if not ops.ext_available():
        pytest.skip("extensions are not built")
    window = ops.ext().fa_head_window
    assert window(1280, 7, 30, False) == 72 and window(672, 12, 10, True) == 40
    assert window(60, 51, 6, True) == 60 and window(80, 16, 3, True) == 80
    for heads in (1 << 20, 16_000_000):
        most = ((1 << 32) - 1) // heads
        for causal in (False, True):
            assert window(heads, most, 100, causal) < heads
            assert window(heads, most + 1, 100, causal) == heads
