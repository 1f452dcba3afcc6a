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
