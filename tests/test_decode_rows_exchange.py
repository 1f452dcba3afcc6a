"""CPU: the many-row kernel's partial exchange keeps the sequence that the other decode kernels keep (store, wait,
barrier, fetch-add, barrier, load), and its plan: which calls take it, its tiles, launch and workspace."""

import pytest
import torch

from bpt_amd import decode_plan
from test_capi import align256, cpu_case
from test_exchange_isa import check_exchange, device_assembly, is_partial_load, is_partial_store, kernel_body


def test_partial_exchange_sequence(tmp_path):
    body = kernel_body(device_assembly("decode_rows_64.hip", tmp_path), "_ZN3bpt18decode_rows_kernelILi1ELi1ELb1ELb0E")
    assert any(is_partial_store(l) for l in body) and any(is_partial_load(l) for l in body)
    problems = check_exchange(body)
    assert not problems, problems[:5]


@pytest.mark.parametrize("fmt", ["fp8", "int8", "bf16"])
@pytest.mark.parametrize("nq,hq,tile", [(9, 16, 32), (16, 16, 32), (17, 16, 64), (8, 64, 64), (65, 8, 128), (255, 8, 128), (256, 64, 256), (2048, 64, 256)])
def test_plan_takes_tiles_from_17_rows(built_lib, fmt, nq, hq, tile):
    q, k, v, table, lens, ks, vs = cpu_case(fmt, b=2, nq=nq, hq=hq, max_blocks=256, nb=8192)
    grid, chunk, ws, cnt = decode_plan(q, k, v, table, lens, ks, vs, scale=0.1, max_context=4096)
    tiles = -(-nq * (hq // 8) // tile)
    assert chunk == 128 and cnt == align256(2 * 8 * tiles * 4)
    assert ws == align256(2 * grid * tile * 129 * 4)  # the no-allocation array (34 MiB) holds any call with 128-row tiles
    assert tile == 256 or ws <= 34 << 20
    assert grid == min(256 * (2 if tile == 32 else 1), 2 * 8 * tiles * 32)


def test_plan_keeps_the_vector_kernel_where_tiles_do_not_fit(built_lib):
    q, k, v, table, lens, ks, vs = cpu_case("fp8", b=2, nq=9, max_blocks=256, nb=8192)
    assert decode_plan(q.float(), k, v, table, lens, ks, vs, scale=0.1, max_context=4096)[1] == 32  # f32 q: f32 products
    q, k, v, table, lens, ks, vs = cpu_case("fp8", b=2049, nq=9, max_blocks=4)
    assert decode_plan(q, k, v, table, lens, ks, vs, scale=0.1, max_context=64)[1] == 32  # line over 4096 entries
    q, k, v, table, lens, ks, vs = cpu_case("fp8", b=2048, nq=9, max_blocks=4)
    assert decode_plan(q, k, v, table, lens, ks, vs, scale=0.1, max_context=64)[1] == 128


@pytest.mark.parametrize("fmt,b,nq,hq,hkv,context,tile", [
    ("fp8", 1, 64, 2, 2, 300, 32), ("int8", 2, 32, 16, 8, 512, 32),  # up to 256 units of 32 rows: 12, 128
    ("fp8", 1, 256, 4, 4, 1024, 32), ("fp8", 1, 256, 4, 4, 1025, 64),  # 256 and 288 of them, 144 of 64
    ("fp8", 1, 256, 4, 4, 2048, 64), ("fp8", 1, 256, 4, 4, 2049, 128),  # 256 of 64 rows and more
    ("fp8", 4, 40, 8, 8, 128, 64), ("fp8", 4, 40, 8, 8, 129, 32),  # one chunk, and two
    ("fp8", 4, 80, 8, 8, 128, 32), ("bf16", 4, 40, 8, 8, 200, 32), ("int8", 16, 17, 8, 8, 4096, 32)])
def test_plan_takes_small_tiles_where_the_chip_would_idle(built_lib, fmt, b, nq, hq, hkv, context, tile):
    q, k, v, table, lens, ks, vs = cpu_case(fmt, b=b, nq=nq, hq=hq, hkv=hkv, max_blocks=512, nb=64)
    grid, chunk, ws, cnt = decode_plan(q, k, v, table, lens, ks, vs, scale=0.1, max_context=context)
    assert chunk == 128 and ws == align256(2 * grid * tile * 129 * 4)


@pytest.mark.parametrize("q_dtype,b,nq,hq,hkv,context,vector", [
    (torch.bfloat16, 1, 24, 8, 8, 512, True),  # 32 chunks of 16 tokens in partitions of 4: eight of a sequence
    (torch.bfloat16, 1, 24, 8, 8, 500, True), (torch.bfloat16, 1, 24, 8, 8, 496, False),  # 31 chunks: not whole
    (torch.bfloat16, 1, 24, 8, 8, 256, True), (torch.bfloat16, 1, 24, 8, 8, 128, False),  # four partitions; two
    (torch.bfloat16, 1, 17, 2, 2, 160, True), (torch.bfloat16, 1, 17, 2, 2, 128, False),  # five partitions of 2; four
    (torch.bfloat16, 4, 64, 32, 8, 4096, False),  # partitions of 32 chunks
    (torch.float16, 1, 17, 4, 2, 32, True), (torch.float16, 4, 17, 4, 2, 64, False), (torch.float16, 4, 17, 4, 2, 512, True)])
def test_plan_keeps_small_bf16_calls_on_the_vector_kernel(built_lib, q_dtype, b, nq, hq, hkv, context, vector):
    q, k, v, table, lens, ks, vs = cpu_case("bf16", b=b, nq=nq, hq=hq, hkv=hkv, max_blocks=512, nb=64)
    plan = lambda q, splits=None: decode_plan(q, k, v, table, lens, ks, vs, scale=0.1, max_context=context, num_splits=splits)  # noqa: E731
    assert plan(q.to(q_dtype))[1] == (16 if vector else 128)
    assert plan(q.to(q_dtype), 2)[1] == 128  # a caller's split count keeps the tiles
