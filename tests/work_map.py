"""nano-inference_amd/csrc/work_map.h (and key_units.h) compiled for the host: the functions by which the kernels
and their launchers divide the work, callable from tests."""
from __future__ import annotations

import ctypes
import functools
import shutil
import subprocess
import tempfile
from pathlib import Path

import numpy as np

CSRC = Path(__file__).resolve().parent.parent / "nano-inference_amd" / "csrc"

SHIM = r"""
#include "work_map.h"
struct Grid {
  int32_t num_seqs, num_kv_heads, group, map_group, num_m_blocks, groups_per_xcd, order_by_len;
  int32_t pack, pack_shift, level_run, groups;
  uint32_t pack_magic;
};
extern "C" {
int64_t t_grid(Grid* p, int max_q_len, int packed) {
  set_rows(*p, max_q_len, packed);
  p->groups_per_xcd = (p->num_seqs * p->num_kv_heads + kXcds - 1) / kXcds;
  return grid_size(*p);
}
int64_t t_f32_grid(Grid* p, int64_t rows, int top_left, int cut) {
  p->groups = p->num_seqs * p->num_kv_heads;
  const int64_t n = f32_grid(p->groups, rows, p->num_m_blocks);
  p->level_run = f32_run(n, p->num_m_blocks, top_left, cut);
  return n;
}
// kind 0: prefill_map, 1: ranked, 2: pair, 3: fp32 (3-D: x, then y, then z); out[id] = seq, head,
// block or -1s
void t_map(const Grid* p, int kind, int n, const int* order, int* out) {
  for (int id = 0; id < n; ++id, out += 3) {
    int s = 0, h = 0, m = 0;
    const bool ok = kind == 0   ? (p->pack > 1 ? prefill_map<true>(*p, id, s, h, m)
                                             : prefill_map<false>(*p, id, s, h, m))
                    : kind == 1 ? prefill_map_ranked(*p, id, order, s, h, m)
                    : kind == 2 ? pair_map(*p, id, s, h, m)
                    : p->level_run
                        ? (f32_map(*p, id, 0, 0, s, h, m), true)
                        : (f32_map(*p, id % p->num_m_blocks, id / p->num_m_blocks % p->num_kv_heads,
                                   id / p->num_m_blocks / p->num_kv_heads, s, h, m),
                           true);
    out[0] = ok ? s : -1;
    out[1] = ok ? h : -1;
    out[2] = ok ? m : -1;
  }
}
int t_div(int x, int d) {
  uint32_t m;
  int32_t s;
  block_divisor(d, m, s);
  return key_block(x, m, s);
}
int t_pack_uncut(const Grid* p, int max_q_len) { return pack_uncut(*p, max_q_len); }
int64_t t_blocks(int group, int max_q_len, int packed) {
  return packed ? packed_blocks(group, max_q_len) : head_blocks(group, max_q_len);
}
int64_t t_span(int64_t q_tok, int64_t q_head, int pack, int d) {
  return q_span_bytes(q_tok, q_head, pack, d);
}
int t_ranges(int tiles, int splits, int f32) {
  return f32 ? f32_ranges(tiles, splits) : key_ranges(tiles, splits);
}
int64_t t_range_tile(int tiles, int s, int n) { return range_tile(tiles, s, n); }
int t_split_count(int64_t nwg, int64_t tiles, int top_left) {
  return split_count(nwg, tiles, top_left);
}
int t_f32_split_count(int64_t nwg, int64_t keys, int64_t rows) {
  return f32_split_count(nwg, keys, rows);
}
int t_few(int64_t total, int64_t alone) { return few_units(total, alone); }
int t_merge_waves(int64_t pairs, int64_t ranges, int64_t sequences) {
  return merge_waves(pairs, ranges, sequences);
}
int64_t t_few_per(int64_t total, int64_t alone, int64_t ranges, int64_t sequences) {
  return few_units_a_range(total, alone, ranges, sequences);
}
}
"""


class Grid(ctypes.Structure):
    _fields_ = [(n, ctypes.c_int32) for n in (
        "num_seqs", "num_kv_heads", "group", "map_group", "num_m_blocks", "groups_per_xcd",
        "order_by_len", "pack", "pack_shift", "level_run", "groups")] + [("pack_magic", ctypes.c_uint32)]


@functools.lru_cache(maxsize=None)
def lib():
    cxx = shutil.which("g++") or shutil.which("c++") or "/opt/rocm/llvm/bin/clang++"
    out = Path(tempfile.mkdtemp(prefix="work_map_"))
    (out / "shim.cpp").write_text(SHIM)
    subprocess.run([cxx, "-std=c++17", "-O1", "-shared", "-fPIC",
                    f"-I{CSRC}", str(out / "shim.cpp"), "-o", str(out / "shim.so")], check=True)
    so = ctypes.CDLL(str(out / "shim.so"))
    shutil.rmtree(out)
    for name in ("t_grid", "t_f32_grid", "t_blocks", "t_span", "t_range_tile", "t_few_per"):
        getattr(so, name).restype = ctypes.c_int64
    i64 = ctypes.c_int64
    so.t_f32_grid.argtypes = [ctypes.c_void_p, i64, ctypes.c_int, ctypes.c_int]
    so.t_span.argtypes = [i64, i64, ctypes.c_int, ctypes.c_int]
    so.t_split_count.argtypes = [i64, i64, ctypes.c_int]
    so.t_f32_split_count.argtypes = [i64, i64, i64]
    so.t_merge_waves.argtypes = [i64, i64, i64]
    so.t_few.argtypes = [i64, i64]
    so.t_few_per.argtypes = [i64, i64, i64, i64]
    return so


def grid(seqs, hkv, group, max_q_len, packed, ranked=False):
    """The bf16 grid of a call and its number of workgroups."""
    g = Grid(num_seqs=seqs, num_kv_heads=hkv, group=group, order_by_len=int(ranked))
    return g, lib().t_grid(ctypes.byref(g), max_q_len, int(packed))


def packs_uncut(seqs, hkv, group, max_q_len):
    g = Grid(num_seqs=seqs, num_kv_heads=hkv, group=group)
    return bool(lib().t_pack_uncut(ctypes.byref(g), max_q_len))


def mapped(g, kind, n, order=None):
    """(sequence, head, block) of the first n workgroups that have work, in grid order."""
    out = np.empty((n, 3), dtype=np.int32)
    order = np.ascontiguousarray(order if order is not None else np.arange(g.num_seqs), np.int32)
    lib().t_map(ctypes.byref(g), ("dense", "ranked", "pair", "f32").index(kind), n,
                order.ctypes.data_as(ctypes.c_void_p), out.ctypes.data_as(ctypes.c_void_p))
    return [tuple(x) for x in out[out[:, 0] >= 0].tolist()]
