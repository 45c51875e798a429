"""Host-side logic of the package (no GPU): helper API with the reference's
names, option mapping, the C-ABI library's exports and its argument checks."""
import ctypes as C
import os
import re

import numpy as np
import pytest
import torch

from oracle import hot_oracle as orc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ----------------------------------------------------------- helper surface

def test_helpers_agree_with_oracle():
    from hot_amd import hadamard_matmul as hm
    for size in (1, 2, 4, 12, 16, 48, 49, 64, 197, 768, 3072, 11008, 12608, 25216):
        assert hm.biggest_power2_factor(size) == orc.pow2_factor(size)
        assert hm.biggest_power2_factor_max16(size) == orc.pow2_factor_max16(size)
        assert np.array_equal(hm.make_hadamard(size), orc.make_hadamard(size))
        n, rows = hm.hla_rows(size)
        n2, rows2 = orc.hla_rows(size)
        assert n == n2 and np.array_equal(rows, rows2)
        if n <= 256:
            assert np.array_equal(hm.make_WHT(size), orc.make_WHT(size))
    assert hm.make_WHT(8192).shape == (2080, 8192)
    n, rows = hm.paper_rows(16, 8)
    assert np.array_equal(rows, orc.paper_rows(16, 8)[1])
    with pytest.raises(ValueError):
        hm.hadamard(12)


def test_lowering_matmuls():
    from hot_amd import hadamard_matmul as hm
    rng = np.random.default_rng(0)
    a = rng.integers(-20, 20, (128, 48)).astype(np.float32)
    H = torch.tensor(hm.hadamard(16), dtype=torch.float32)
    assert np.array_equal(hm.lowering_matmul_front(torch.from_numpy(a), H).numpy(), orc.fwht_blocks_last(a, 16))
    assert np.array_equal(hm.lowering_matmul_back(H, torch.from_numpy(a)).numpy(), orc.fwht_blocks_first(a, 16))
    P = torch.tensor(hm.make_WHT(64), dtype=torch.float32)
    n, rows = orc.hla_rows(64)
    assert np.array_equal(hm.lowering_matmul_back(P, torch.from_numpy(a)).numpy(), orc.fwht_blocks_first(a, n, rows))
    a3 = torch.from_numpy(np.stack([a, 2 * a]))
    assert hm.lowering_matmul_back(P, a3).shape == (2, 72, 48)
    assert np.array_equal(hm.lowering_matmul_front(a3, H)[1].numpy(), orc.fwht_blocks_last(2 * a, 16))
    # whole-dimension case: plain matmul
    assert np.array_equal(hm.lowering_matmul_back(torch.tensor(hm.make_WHT(128), dtype=torch.float32),
                                                  torch.from_numpy(a)).numpy(),
                          orc.fwht_blocks_first(a, 128, orc.hla_rows(128)[1]))


def test_transform_dict_caches():
    from hot_amd.hadamard_matmul import Transform_Dict
    td = Transform_Dict()
    h = td.get_or_register("hadamard", 3072)
    assert h.shape == (16, 16) and td.get_or_register("hadamard", 3072) is h
    assert td.get_or_register("low_rank", 12608, 50).shape == (36, 64)
    with pytest.raises(NotImplementedError):
        td.get_or_register("haar", 8)


# ------------------------------------------------------------ option mapping

@pytest.fixture
def fresh_args():
    from hot_amd import args
    saved = {k: getattr(args, k) for k in dir(args) if not k.startswith("_")}
    args.hot_recipe()          # the module defaults describe a plain layer, as the reference's do
    yield args
    for k, v in saved.items():
        setattr(args, k, v)


def test_options_follow_args(fresh_args):
    from hot_amd import ops
    from hot_amd.quant_matmul import options_for
    a = fresh_args
    o = options_for(12608)
    assert (o.hla_n, o.hla_r, o.n_o) == (64, 36, 16)
    assert (o.gx_bits, o.w_bits, o.gw_bits, o.act_bits) == (4, 4, 8, 8)
    assert o.gx_round == ops.ROUND_NEAREST and o.gx_scale == ops.SCALE_TENSOR
    a.quantBWDGogi, a.quantBWDWgt, a.quantBWDGogw, a.quantBWDAct = "nq", "sawb", "stoch", "sawb"
    o = options_for(12608)
    assert (o.gx_round, o.gx_scale) == (ops.ROUND_STOCH, ops.SCALE_ROW)
    assert (o.w_round, o.w_scale) == (ops.ROUND_NEAREST, ops.SCALE_SAWB)
    assert (o.gw_round, o.gw_scale) == (ops.ROUND_STOCH, ops.SCALE_TENSOR)
    assert o.act_scale == ops.SCALE_SAWB
    # layer-wise selection: the g_W branch reads the g_x bit width (utils/quant_matmul.py:308)
    a.quantAuto = True
    a.layer_quant_dict["blk_gx"] = "norm_quantizer"
    a.layer_quant_dict["blk_gw"] = "stoch_quantizer"
    o = options_for(12608, "blk")
    assert (o.gx_scale, o.gw_scale, o.gw_bits) == (ops.SCALE_ROW, ops.SCALE_TENSOR, 4)
    a.layer_quant_dict.clear()
    a.quantAuto = False
    # token rules
    assert options_for(197).hla_n == 1
    o = options_for(8192)                           # the reference's rule, whatever the block size
    assert (o.hla_n, o.hla_r) == (8192, 2080)
    a.hla_max_block = 64
    o = options_for(8192)
    assert (o.hla_n, o.hla_r) == (64, 36)
    a.hla_max_block = 8192
    a.hla_rule = "paper"
    o = options_for(8192)
    assert (o.hla_n, o.hla_r) == (16, 8)
    a.hla_rule = "python"
    a.quantBWDGogi = "luq"                          # an entry point of its own for the g_x product
    from hot_amd.quant_matmul import gx_uses_luq
    assert gx_uses_luq() and options_for(64).gx_bits == 4
    a.quantBWDGogw = "luq"                          # and one for the g_W product
    from hot_amd.quant_matmul import gw_uses_luq
    assert gw_uses_luq() and options_for(64).gw_round == ops.ROUND_STOCH
    a.quantBWDGogw = "int"
    assert not gw_uses_luq()
    a.quantBWDGogi = "int"
    assert not gx_uses_luq()
    a.transform_scheme = "hadamard"                 # block Hadamard along the tokens, nothing dropped
    o = options_for(12608)
    assert (o.hla_n, o.hla_r, o.hla_rows) == (16, 16, tuple(range(16)))
    assert options_for(197).hla_n == 1 and options_for(200).hla_n == 8
    a.transform_scheme = "low_rank"                 # g_W side as gih_gwlr; the g_x side has a rule of its own
    from hot_amd.quant_matmul import gx_token_rule
    o = options_for(12608)
    assert (o.hla_n, o.hla_r) == (64, 36)
    assert gx_token_rule(8192)[0] == 8192 and len(gx_token_rule(8192)[1]) == 2080    # the reference's own rule
    assert gx_token_rule(25216)[0] == 128 and len(gx_token_rule(25216)[1]) == 36
    a.hla_max_block = 64
    assert gx_token_rule(8192)[0] == 64 and len(gx_token_rule(8192)[1]) == 36
    a.hla_max_block = 8192
    a.transform_scheme = "gilr_gwh"                 # g_W side as hadamard
    o = options_for(12608)
    assert (o.hla_n, o.hla_r) == (16, 16)
    assert gx_token_rule(12608)[0] == 64
    a.transform_scheme = "gilro_gwh"
    with pytest.raises(NotImplementedError):
        options_for(64)
    a.transform_scheme = "gih_gwlr"
    a.TransformInput = False
    with pytest.raises(NotImplementedError):
        options_for(64)


def test_hq_linear_surface_and_no_cpu_fallback(fresh_args):
    import torch.nn as nn
    from hot_amd.quant_matmul import FLinearQ, HQ_Linear
    lin = HQ_Linear(48, 64)
    assert isinstance(lin, nn.Linear) and lin.hadamard_out.shape == (16, 16) and lin.layer_name == " "
    assert "hadamard_out" not in lin.state_dict() and "hadamard_bs" not in lin.state_dict()
    assert {"forward", "setup_context", "backward"} <= set(vars(FLinearQ))
    with pytest.raises(RuntimeError):           # the native path refuses CPU tensors, it never falls back
        lin(torch.randn(128, 48))
    # the module defaults are the reference's: a plain full-precision layer, which runs anywhere
    fresh_args.plain_recipe()
    x = torch.randn(128, 48, requires_grad=True)
    lin(x).sum().backward()
    assert x.grad is not None and lin.weight.grad.shape == (64, 48)


def test_args_defaults_are_the_reference_defaults():
    """args.py:29-49 of the reference: widths 0, quantisers "no", transforms off, scheme gih_gwlr."""
    import importlib
    from hot_amd import args
    fresh = importlib.reload(args)
    try:
        assert (fresh.GogiQuantBit, fresh.weightQuantBit, fresh.GogwQuantBit, fresh.actQuantBit) == (0, 0, 0, 0)
        assert (fresh.quantBWDGogi, fresh.quantBWDWgt, fresh.quantBWDGogw, fresh.quantBWDAct) == ("no",) * 4
        assert not (fresh.TransformGogi or fresh.TransformWgt or fresh.TransformGogw or fresh.TransformInput)
        assert fresh.transform_scheme == "gih_gwlr" and fresh.quantAuto is False and fresh.eps == 1e-11
        fresh.canonical_recipe()
        assert (fresh.quantBWDGogi, fresh.quantBWDWgt, fresh.quantBWDGogw, fresh.quantBWDAct) == ("nq", "sawb", "nq", "sawb")
        assert (fresh.GogiQuantBit, fresh.weightQuantBit, fresh.GogwQuantBit, fresh.actQuantBit) == (4, 4, 8, 8)
        assert fresh.quantAuto and fresh.TransformGogi and fresh.TransformInput
    finally:
        fresh.plain_recipe()


def test_replace_layers_style_surgery():
    """The reference swaps layers by constructing new(in_features, out_features)
    and re-pointing weight/bias data (utils/utils.py:53-74)."""
    import torch.nn as nn
    from hot_amd.quant_matmul import HQ_Linear
    model = nn.Sequential(nn.Linear(32, 64), nn.GELU(), nn.Linear(64, 16))
    for name, mod in list(model.named_children()):
        if isinstance(mod, nn.Linear):
            new = HQ_Linear(mod.in_features, mod.out_features)
            new.weight.data = mod.weight.data
            new.bias.data = mod.bias.data
            setattr(model, name, new)
    assert isinstance(model[0], HQ_Linear) and model[2].weight.shape == (16, 64)


def test_hlq_backward_checks_like_the_reference():
    from hot_amd import HLQ_backward
    z = torch.zeros(4, 16)
    with pytest.raises(RuntimeError, match="Go must be a CUDA tensor!"):
        HLQ_backward.backward(z, z, z, 0, 0, 16, True)


def test_hlq_options_follow_the_value_of_the_block_size():
    from hot_amd import HLQ_backward
    size = torch.tensor(16)
    assert HLQ_backward.options(48, size, True).n_o == 16
    size.fill_(8)
    assert HLQ_backward.options(48, size, True).n_o == 8


def test_options_keep_the_row_list_through_a_chain_of_keys():
    """hla_rows_big is a host pointer: whichever ancestor built the array, the last of a chain of with_seed() owns it."""
    import gc
    from hot_amd import ops
    rows = tuple(range(2048))
    first = ops.HotOptions(hla_n=2048, hla_rows=rows)
    second = first.with_seed(1)
    last = second.with_seed(2).with_seed(3)
    del first, second
    gc.collect()
    noise = [(C.c_int32 * 2048)(*([7777] * 2048)) for _ in range(64)]
    c = last.to_c()
    assert c.seed == 3 and [c.hla_rows_big[i] for i in range(2048)] == list(rows) and len(noise) == 64


def test_options_under_another_key_keep_their_class():
    from hot_amd import ops

    class Options(ops.HotOptions):
        pass

    assert type(Options(seed=1).with_seed(2)) is Options


# --------------------------------------------------------------- the C ABI

def _declared():
    text = open(os.path.join(ROOT, "include", "hot_gfx950.h")).read()
    return re.findall(r"HOT_API\s+[\w\s\*]+?\b(hot_\w+)\s*\(", text)


def test_library_exports_every_declared_symbol():
    from hot_amd import _lib
    names = _declared()
    assert len(names) >= 12 and set(names) == set(_lib.EXPORTS)
    lib = C.CDLL(_lib.LIB_PATH)
    for n in names:
        assert hasattr(lib, n), n
    assert _lib.lib().hot_abi_version() == 4
    header = open(os.path.join(ROOT, "include", "hot_gfx950.h")).read()
    for name in ("HOT_MAX_HLA_N", "HOT_MAX_HLA_BIG", "HOT_HQ_WORKSPACE_BYTES", "HOT_STATIC_MAX_CHANNELS"):   # the binding repeats these constants
        assert int(re.search(r"#define\s+%s\s+(\d+)" % name, header).group(1)) == getattr(_lib, name)
    enum = re.search(r"enum hot_gemm_variant \{(.*?)\};", header, re.S).group(1)
    for name, val in re.findall(r"HOT_(GEMM_\w+)\s*=\s*(\d+)", enum):
        if name != "GEMM_VARIANTS":
            assert getattr(_lib, name) == int(val), name
    assert [_lib.lib().hot_kpad(k) for k in (1, 128, 129, 7092)] == [128, 128, 256, 7168]


def test_library_argument_checks_need_no_gpu():
    from hot_amd import _lib, ops
    lib = _lib.lib()
    one = C.c_void_p(4096)  # never dereferenced: every call below fails validation first
    assert lib.hot_hq_rowwise(one, 0, 4, 64, 12, 4, 0, 0, 0, 0, one, one, None, 0, None) == -2
    assert b"Hadamard block" in lib.hot_last_error()
    assert lib.hot_hq_rowwise(one, 0, 4, 40, 16, 4, 0, 0, 0, 0, one, one, None, 0, None) == -1
    assert lib.hot_hq_rowwise(one, 0, 4, 64, 16, 4, 0, 0, 0, 0, one, one, None, 0, None) == -3   # no workspace
    assert lib.hot_gemm_i8(one, 64, one, 64, 8, 4, 4, 100, one, 0, one, 1.0, one, 0, 4, None, None) == -1
    assert b"row pitches" in lib.hot_last_error()
    rows = (C.c_int32 * 2)(0, 0)
    assert lib.hot_hla_tokenwise(one, 0, 64, 8, 16, rows, 2, 8, 0, 0, 0, 0, one, 128, one, one, 1 << 30, None) == -1
    assert b"listed twice" in lib.hot_last_error()
    # the variant query and the named-variant entry point validate before they touch anything
    assert lib.hot_gemm_plan(12608, 768, 3072, 4, 1536, 1536, 0) == _lib.GEMM_SLOT_160X256
    assert lib.hot_gemm_plan(12608, 768, 2304, 4, 1152, 1152, 0) == _lib.GEMM_DMA_128_S3
    # INT8 products with room to spare at 128 x 128 take the shortest tile that keeps one round (ViT-B g_W products)
    assert lib.hot_gemm_plan(3072, 768, 7092, 8, 7168, 7168, 0) == _lib.GEMM_SLOT_96X128        # fc1: 192 tiles
    assert lib.hot_gemm_plan(3072, 768, 7092, 8, 7168, 7168, 1 << 30) == _lib.GEMM_SLOT_96X128  # a workspace changes nothing
    assert lib.hot_gemm_plan(2304, 768, 7092, 8, 7168, 7168, 0) == _lib.GEMM_SLOT_64X128        # qkv: 216 tiles
    assert lib.hot_gemm_plan(768, 768, 7092, 8, 7168, 7168, 1 << 30) == _lib.GEMM_SLOT_32X128   # proj: 144 tiles, no split
    assert lib.hot_gemm_plan(768, 3072, 7092, 8, 7168, 7168, 0) == _lib.GEMM_SLOT_96X128        # fc2: 192 tiles
    assert lib.hot_gemm_plan(4096, 1024, 7092, 8, 7168, 7168, 0) == _lib.GEMM_SLOT_128          # 256 tiles: nothing shorter fits
    assert lib.hot_gemm_plan(768, 768, 7092, 4, 3584, 3584, 1 << 30) == _lib.GEMM_DMA_128_SPLITK # INT4: 36 tiles, split K
    assert lib.hot_gemm_plan(8192, 4096, 11008, 4, 5504, 5504, 0) == _lib.GEMM_SLOT_256
    assert lib.hot_gemm_plan(8192, 4096, 11136, 4, 5568, 5568, 0) == _lib.GEMM_DMA_256_S4     # rows of 43.5 lines
    assert lib.hot_gemm_plan(1 << 20, 128, 8192, 8, 8192, 8192, 0) == _lib.GEMM_REG_128     # A is 8 GiB
    assert lib.hot_gemm_workspace_bytes(3072, 768, 7092, 8) == 144 * 3 * 128 * 128 * 4      # what the split-K variant would take
    assert lib.hot_gemm_i8_variant(one, 128, one, 128, 8, 4, 4, 100, one, 0, one, 1.0, one, 0, 4, None, 99, None, 0, None) == -1
    assert b"variant" in lib.hot_last_error()
    assert lib.hot_gemm_i8_variant(one, 128, one, 128, 8, 4, 4, 100, one, 0, one, 1.0, one, 0, 4, None,
                                   _lib.GEMM_DMA_128_SPLITK, None, 0, None) == -2      # nothing to split
    # the entry point without a workspace: limits checked before anything else
    assert lib.hot_hla_tokenwise_static(one, 0, 512, 64, 256, rows, 2, 8, 0, 0, 0, 0, one, 128, one, None) == -2
    assert lib.hot_hla_tokenwise_static(one, 0, 64, _lib.HOT_STATIC_MAX_CHANNELS + 8, 16, rows, 2, 8, 0, 0, 0, 0, one, 128, one, None) == -2
    assert b"channels exceed" in lib.hot_last_error()
    cfg = ops.HotOptions(hla_n=64, hla_rows=tuple(range(36))).to_c()
    need = lib.hot_backward_workspace_bytes(12608, 3072, 768, C.byref(cfg))
    # packed g_y codes + packed W codes + int8 low-rank g_y codes dominate
    assert need >= 12608 * 1536 + 768 * 1536 + 3072 * 7168
    cfg.n_o = 12            # not a power of two
    assert lib.hot_backward_workspace_bytes(12608, 3072, 768, C.byref(cfg)) == 0
    with pytest.raises(_lib.HotError):
        _lib.check(-2)


@pytest.mark.parametrize("field,value,message", [("gx_scale", 7, b"scale mode"), ("gx_scale", -1, b"scale mode"), ("gx_round", 5, b"rounding"),
                                                 ("out_dtype", 9, b"dtype")])
@pytest.mark.parametrize("hla_n", [1, 64, 256])
def test_backward_refuses_unknown_modes_before_any_launch(field, value, message, hla_n):
    """Fields outside their enums, in the fused entry points: an error from the host, nothing launched."""
    from hot_amd import _lib, ops
    lib = _lib.lib()
    one = C.c_void_p(4096)  # never dereferenced: every call below fails validation first
    cfg = ops.HotOptions(hla_n=hla_n, hla_rows=tuple(range(max(1, hla_n // 2)))).to_c()
    out = _lib.F32
    if field == "out_dtype":
        out = value
    else:
        setattr(cfg, field, value)
    big = 1 << 40
    assert lib.hot_linear_backward(one, one, 0, one, one, 256, 64, 64, C.byref(cfg), one, one, out, one, big, None, None) < 0
    assert message in lib.hot_last_error()
    assert lib.hot_linear_backward_bias(one, one, 0, one, one, 256, 64, 64, C.byref(cfg), one, one, one, out, one, big, None) < 0
    assert message in lib.hot_last_error()
    if hla_n <= 128:
        assert lib.hot_linear_backward_batched_bias(one, one, 0, one, one, 2, 128, 64, 64, C.byref(cfg), one, one, one, out, one, big, None) < 0
        assert message in lib.hot_last_error()


def test_bench_refuses_more_than_one_gpu():
    """Every box has one GPU: the benchmark says so instead of running a second rank."""
    import subprocess
    import sys
    r = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert r.returncode != 0 and "ONE GPU" in r.stderr and r.stdout.strip() == ""


def test_launch_of_the_products():
    """hot_backward_products: refused arguments, the order that the caller asks for, and both widths on either side of the lines
    between the launches (few tiles of g_x with a long K; 256 tiles of 192 x 128 of g_W; full rounds of 256 x 256 tiles)."""
    from hot_amd import ops

    def launch(L, O, I, bits=4, n=16, **kw):
        rows = orc.paper_rows(n, n // 2)[1] if n > 1 else (0,)
        return ops.backward_products(L, O, I, ops.HotOptions(n_o=16, hla_n=n, hla_rows=tuple(int(r) for r in rows), gx_bits=bits, w_bits=bits, **kw))

    assert launch(100, 64, 64) == 0 and launch(0, 64, 64) == 0 and launch(64, 72, 64) == 0      # blocks of 16 tokens and channels
    assert launch(64, 64, 20) == 0
    assert launch(64, 64, 64) == ops.PRODUCTS_PAIR_128 == launch(64, 64, 64, streams=1)
    assert launch(64, 64, 64, streams=2) == ops.PRODUCTS_APART
    for bits, longest in ((4, 3328), (8, 1664)):
        assert launch(64, longest, 64, bits) == ops.PRODUCTS_PAIR_128 and launch(64, longest + 16, 64, bits) == ops.PRODUCTS_APART
        assert launch(64, 1536, 3968, bits) == ops.PRODUCTS_PAIR_128 and launch(64, 1536, 4096, bits) == ops.PRODUCTS_PAIR_192
    assert launch(8192, 11008, 4096) == ops.PRODUCTS_PAIR_192


def test_tiling_of_the_paired_products():
    """hot_backward_pair_rows: small products in tiles of 64, those that fill the chip in larger ones, 0 where none is shared."""
    from hot_amd import ops

    def rows(L, O, I, bits=4, **kw):
        n, r = orc.hla_rows(min(L & -L, 64) or 1)
        return ops.backward_pair_rows(L, O, I, ops.HotOptions(n_o=8, hla_n=n, hla_rows=tuple(int(v) for v in r), gx_bits=bits, w_bits=bits, **kw))

    assert rows(49, 3072, 768) == rows(64, 64, 64) == rows(3003, 1000, 520) == 64
    assert rows(12608, 3072, 768) == rows(12608, 2304, 768) == rows(12608, 3072, 768, 8) == 128
    assert rows(12608, 768, 3072, 8) == rows(8192, 11008, 4096) == 192
    # up to 256 out-features no tiles of 192 rows, of any width (wider g_x, long runs of tokens), unless g_W fills the chip with them
    assert rows(15199, 128, 7848) == rows(10496, 80, 5520, 8) == rows(11776, 168, 4992) == rows(9728, 256, 9856) == 128
    assert rows(9728, 264, 9856) == rows(9728, 200, 17000) == 192
    assert rows(64, 64, 64, streams=2) == rows(64, 8192, 64) == rows(0, 64, 64) == rows(64, 64, 20) == 0


@pytest.mark.parametrize("B,T,O", [(0, 15425, 2048), (0, 4597, 9568), (0, 16411, 16), (0, 1023, 32), (0, 272, 128), (0, 12608, 3072),
                                   (1, 12608, 3072), (64, 577, 1464), (128, 197, 912), (64, 208, 768)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_runs_of_the_column_sums(B, T, O, dtype):
    """The partial sums of a bias gradient cover runs of token blocks that depend on the shape alone, so that its last bits do: 32 to 128
    codes of a channel while there are 1024 workgroups and no resident one is lost (rings of three fp32 or four 16-bit steps), cut to
    64 rows below 2048 workgroups."""
    from hot_amd import ops
    n, rows = orc.hla_rows(min(T & -T, 128))
    r, strips, size = len(rows), -(-O // 256), 4 if dtype == torch.float32 else 2
    wgs = lambda t: strips * -(-((B or 1) * T // n) // t)
    resident = lambda t: min(3, 160 * 1024 // ((3 if size == 4 else 4) * 16 * 256 * size + 256 * (t * r + 4) + 256))
    t = max(1, 16 // n)
    while t * r % 4 or t * r < 32:
        t *= 2
    while t * r < 128 and wgs(2 * t) >= 1024 and resident(2 * t) >= resident(t):
        t *= 2
    while t > max(1, 16 // n) and t * n > 64 and wgs(t) < 2048:
        t //= 2
    for scale in ("tensor", "row"):
        opt = ops.HotOptions(n_o=8, hla_n=n, hla_rows=tuple(int(v) for v in rows), gx_scale=scale, gw_scale=scale)
        assert ops.backward_gy_runs(B, T, O, 64, opt, dtype, bias=True)[0] == -(-(T // n) // t)


@pytest.mark.parametrize("B,T,O,tokens", [(0, 6879, 7424, 64), (0, 2561, 9280, 64), (0, 6698, 3712, 64), (0, 12608, 2304, 64), (64, 577, 1464, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_runs_of_a_full_launch(B, T, O, tokens, dtype):
    """Where the launch fills the chip the quantise pass takes the longest runs that cost no resident workgroup, as if every ring had all
    its buffers, in 32-bit types too: a shorter ring is no reason for a shorter run."""
    from hot_amd import ops
    n, rows = orc.hla_rows(min(T & -T, 64))
    opt = ops.HotOptions(n_o=8, hla_n=n, hla_rows=tuple(int(v) for v in rows))
    assert ops.backward_gy_runs(B, T, O, 1024, opt, dtype)[1] == -(-T // tokens)


def test_paths_of_the_channel_maxima():
    """Which arrays of per-channel maxima a statistics pass keeps, at the sizes that the tests on the GPU take for them: one for each run
    of token blocks up to 64, one for four of them up to 256 and where there is no more room, else copies that runs share (0)."""
    from hot_amd import ops

    def path(B, T, O, I, dtype=torch.float32, **kw):
        n, rows = orc.hla_rows(min(T & -T, 128))
        opt = ops.HotOptions(n_o=16, hla_n=n, hla_rows=tuple(int(v) for v in rows), gw_scale="row", **kw)
        runs, _, own, tall = ops.backward_gy_runs(B, T, O, I, opt, dtype)
        return runs, own, tall

    for dtype in (torch.float32, torch.bfloat16, torch.float16):
        for L, O, I, expected in ((1023, 32, 16, (64, 64, False)), (1025, 32, 16, (65, 17, True)), (1041, 80, 16, (66, 17, True)),
                                  (4163, 80, 16, (261, 0, False)), (8191, 16, 16, (256, 64, True)), (8193, 16, 16, (257, 0, False)),
                                  (1023, 2064, 8, (32, 32, False)), (4095, 3600, 8, (64, 16, True))):
            assert path(0, L, O, I, dtype, gx_bits=8, w_bits=8) == expected, (L, O)
        assert path(16, 577, 688, 8, dtype) == (19, 0, False)
        assert path(16, 577, 512, 8, dtype) == (19, 19, False)      # (as many of fewer channels have room)
    # one long sample: the runs of a call with a bias gradient, and the longer ones without
    for T, O, kept, longer in ((8191, 2064, 128, 64), (12608, 3072, 197, 50), (16384, 768, 256, 128)):
        n, rows = orc.hla_rows(min(T & -T, 64))
        opt = ops.HotOptions(n_o=16, hla_n=n, hla_rows=tuple(int(v) for v in rows), gx_scale="row", gw_scale="row")
        for B in (0, 1):
            assert [ops.backward_gy_runs(B, T, O, 16, opt, torch.float32, bias)[0] for bias in (True, False)] == [kept, longer]
