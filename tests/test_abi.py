"""The C ABI: the built library loads and exports every function include/baretile_amd.h declares. CPU only: nothing
here calls into a GPU."""
import ctypes, os, re
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "baretile_amd.h")


def declared():
  text = open(HEADER).read()
  text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
  return sorted(set(re.findall(r"\b(bt_[a-z0-9_]+)\s*\(", text)))


def test_header_declares_the_abi():
  names = declared()
  assert {"bt_open", "bt_close", "bt_alloc", "bt_matmul", "bt_attention", "bt_bfp_pack", "bt_bfp_unpack"} <= set(names)


def test_library_exports_every_declared_symbol():
  from baretile_amd import _lib
  lib = ctypes.CDLL(_lib.PATH)
  missing = [n for n in declared() if not hasattr(lib, n)]
  assert not missing, missing
  # the ctypes table covers the same functions
  assert set(declared()) == set(_lib.SIGNATURES) | {"bt_last_error"}


def test_load_and_version():
  from baretile_amd import _lib
  lib = _lib.load()
  assert lib.bt_version() == 1


def test_errors_map_to_exceptions():
  from baretile_amd import _lib
  lib = _lib.load()
  # a null runtime is a bad argument, whatever the machine has
  with pytest.raises(ValueError, match="no runtime"): _lib.call("wait", None, 1.0)
  with pytest.raises(ValueError, match="no runtime"): _lib.call("alloc", None, 16, ctypes.byref(ctypes.c_uint64()))


def test_struct_sizes_match_the_header(tmp_path):
  # the ctypes mirrors against what a C compiler makes of include/baretile_amd.h: sizes and every field's offset
  import shutil, subprocess
  from baretile_amd import _lib
  cc = shutil.which("gcc") or shutil.which("cc")
  if cc is None: pytest.skip("no C compiler")
  structs = {"bt_operand": _lib.Operand, "bt_inst": _lib.Inst, "bt_program": _lib.Program,
             "bt_attention_args": _lib.AttentionArgs, "bt_row_args": _lib.RowArgs, "bt_rope_args": _lib.RopeArgs}
  cname = {("bt_program", "inputs"): "in"}  # Python can't name a field `in`
  lines = ['#include <stdio.h>', '#include <stddef.h>', '#include "baretile_amd.h"', "int main(void) {"]
  for name, cls in structs.items():
    lines.append(f'  printf("{name} %zu\\n", sizeof({name}));')
    for field, *_ in cls._fields_:
      lines.append(f'  printf("{name}.{field} %zu\\n", offsetof({name}, {cname.get((name, field), field)}));')
  lines.append("  return 0; }")
  src = tmp_path / "sizes.c"
  src.write_text("\n".join(lines) + "\n")
  exe = tmp_path / "sizes"
  subprocess.run([cc, "-I", os.path.join(ROOT, "include"), str(src), "-o", str(exe)], check=True)
  got = dict(l.split() for l in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines())
  for name, cls in structs.items():
    assert int(got[name]) == ctypes.sizeof(cls), name
    for field, *_ in cls._fields_:
      assert int(got[f"{name}.{field}"]) == getattr(cls, field).offset, (name, field)


def test_a_program_built_again_keeps_its_own_inputs_and_limits():
  from baretile_amd import _lib
  from baretile_amd.program import Program
  def build(ptr, const=2.0, dtype="bf16"):
    p = Program(dtype)
    x, y = (p.load(p.input(_lib.operand(ptr + i, "bf16", 1, 1, 1))) for i in range(2))
    return p.build(p.op("add", p.op("mul", x, p.const(const)), y))
  a, b, c, d = build(16), build(32), build(16, 3.0), build(16, dtype="fp32")
  assert [a.inputs[i].ptr for i in range(2)] == [16, 17] and [b.inputs[i].ptr for i in range(2)] == [32, 33]
  code = lambda p: (p.n_inst, p.n_inputs, p.dtype, p.result, [(i.op, i.dst, i.a, i.b, i.c, i.imm) for i in p.inst])
  assert code(a) == code(b) != code(c) and code(d)[2] != code(a)[2]
  for _ in range(2):  # a refusal is a refusal again
    p = Program("bf16")
    v = p.load(p.input(_lib.operand(16, "bf16")))
    vs = [p.op("add", v, p.const(float(i))) for i in range(17)]
    out = vs[0]
    for u in vs[1:]: out = p.op("mul", u, out)
    with pytest.raises(ValueError, match="more than|at most"): p.build(out)


@pytest.mark.parametrize("hd", [64, 128])
def test_attention_scratch_of_rows_with_regions(hd):
  # rows with regions of their own, said to be apart: parts chosen by the caller keep the packed tiles' partial sums (a tile 16 pairs,
  # 32 + 16 hd floats a part), the library's own plan fits the 8 MiB of bt_attention_noalloc at every size
  from baretile_amd import _lib
  def scratch(kvh, rep, rows, keys, parts, fmt):
    args = _lib.AttentionArgs(4096, 4096, 4096, 4096, 4096, rows * hd, hd, keys * hd, hd, keys * hd, hd, rows * hd, hd, rows,
                              kvh * rep, rep, rows, keys, hd, 0, parts, 1, 0, 0, 4096, rows, fmt, 0, 4096, 4096)
    need = ctypes.c_uint64()
    _lib.call("attention_scratch", ctypes.byref(args), ctypes.byref(need))
    return need.value
  assert scratch(8, 2, 32, 32 * 512, 8, _lib.BF16) == 8 * 4 * 8 * (32 + 16 * hd) * 4
  for kvh in (1, 2, 3, 8, 10, 40, 170, 341, 512, 4000):
    for rep in (1, 4, 17):
      for rows in (2, 8, 31, 32):
        for keys in (100, 512, 1000, 4096):
          for fmt in (_lib.BF16, _lib.BFP8): assert scratch(kvh, rep, rows, keys * rows, 0, fmt) <= 8 << 20


@pytest.mark.parametrize("hd", [64, 128])
def test_attention_plans_by_region_where_rows_are_apart(hd):
  # rows whose regions may be shared take the plan of a call without regions where that splits the keys (64 pairs a key
  # head) or the tiles by row would be more than 384; the others, and rows said to be apart, the plan by row, within
  # bt_attention_noalloc's 8 MiB at every size
  from baretile_amd import _lib
  def scratch(kvh, rep, rows, keys, fmt, firsts, apart):
    args = _lib.AttentionArgs(4096, 4096, 4096, 4096, 4096, rows * hd, hd, keys * hd, hd, keys * hd, hd, rows * hd, hd, rows,
                              kvh * rep, rep, rows, keys, hd, 0, 0, apart, 0, 0, firsts, rows, fmt, 0, 4096, 4096)
    need = ctypes.c_uint64()
    _lib.call("attention_scratch", ctypes.byref(args), ctypes.byref(need))
    return need.value
  for kvh in (1, 2, 3, 8, 10, 40, 170, 341, 512, 4000):
    for rep in (1, 4, 17):
      for rows in (1, 2, 8, 31, 32, 33):
        for keys in (100, 512, 1000, 4096):
          for fmt in (_lib.BF16, _lib.BFP8):
            plain, apart = scratch(kvh, rep, rows, keys * rows, fmt, 0, 0), scratch(kvh, rep, rows, keys * rows, fmt, 4096, 1)
            by_row = rep * rows > 64 and rows <= 32 and kvh * rows * -(-rep // 16) <= 384
            assert scratch(kvh, rep, rows, keys * rows, fmt, 4096, 0) == (apart if by_row else plain)
            assert plain == scratch(kvh, rep, rows, keys * rows, fmt, 0, 1) and apart <= 8 << 20
  # 8 slots of 512 rows, 3 heads a key head: 9 parts of one block of keys for each of 24 tiles
  assert scratch(3, 3, 8, 8 * 512, _lib.BF16, 4096, 1) == 24 * 9 * (32 + 16 * hd) * 4
