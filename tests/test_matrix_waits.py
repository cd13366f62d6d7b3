"""Matrix instructions that are written by hand (mul of mfma_tile.h) are seen by no compiler, which
puts no wait states round them: the built kernels are looked through for those that they need."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROCM = Path("/opt/rocm/llvm/bin")
OPS = Path(__file__).resolve().parents[1] / "xotorch_amd" / "ops"
AFTER = 18  # wait states until a sum may be read or written by others, of the longest instruction
BEFORE = 2  # from a vector instruction's result to a product that reads it


def _registers(text):
  """The vector registers that operands name: ('v' or 'a', number)"""
  found = set()
  for kind, one, lo, hi in re.findall(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])", text):
    found.update((kind, n) for n in range(int(one or lo), int(one or hi) + 1))
  return found


def _kernels(name, tmp):
  """(kernel, [(opcode, operands, where a branch goes)]) of a built extension"""
  fat, obj = tmp / "fat", tmp / "obj"
  subprocess.run(["objcopy", "--dump-section", f".hip_fatbin={fat}", str(OPS / f"{name}.so"), str(tmp / "rest")], check=True)
  subprocess.run([str(ROCM / "clang-offload-bundler"), "--unbundle", "--type=o", f"--input={fat}",
                  "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", f"--output={obj}"], check=True)
  text = subprocess.run([str(ROCM / "llvm-objdump"), "-d", "--no-show-raw-insn", str(obj)], check=True, capture_output=True, text=True).stdout
  for part in re.split(r"^[0-9a-f]+ <(?=_Z)", text, flags=re.M)[1:]:
    kernel, body = part.split(">:", 1)
    lines = re.findall(r"^\s+(\w+)([^\n]*?)\s*// ([0-9A-F]+):([^\n]*)", body, re.M)
    at = {int(where, 16): i for i, (_, _, where, _) in enumerate(lines)}
    code = []
    for i, (op, rest, where, tail) in enumerate(lines):
      to = None
      if op.startswith(("s_cbranch", "s_branch")):
        step = int(rest.split()[0])
        to = at.get(int(where, 16) + 4 + 4 * (step - 65536 if step >= 32768 else step))
      code.append((op, rest, to))
    yield kernel, code


def _faults(code):
  """Uses of a sum less than AFTER wait states behind the product that makes it, and products that
  read what a vector instruction wrote less than BEFORE ago"""
  def states(op, rest):
    return int(rest.split()[0], 0) + 1 if op == "s_nop" else 1

  def loop_of(i):
    """The innermost loop round instruction i, as first and last instruction"""
    spans = [(to, j) for j, (op, _, to) in enumerate(code) if to is not None and to <= i <= j]
    return min(spans, key=lambda span: span[1] - span[0], default=None)

  def guard(i):
    """Whether this is mul_last's branch: where steps are left it is not taken, and the loop goes on behind
    the product that follows; else the same product and a wait lie behind the kernel's end"""
    to = code[i][2]
    return (code[i][0] == "s_cbranch_scc0" and to is not None and to + 3 < len(code) and code[to][:2] == code[i + 1][:2]
            and code[to + 1][0] == code[to + 2][0] == "s_nop" and states(*code[to + 1][:2]) + states(*code[to + 2][:2]) >= AFTER
            and code[to + 3][0] == "s_branch" and code[to + 3][2] == i + 2)

  def follow(start, budget, stop):
    """What may run within `budget` wait states behind instruction `start`"""
    todo, seen = [(start + 1, budget, loop_of(start) if guard(start - 1) else None)], {}
    while todo:
      i, left, inside = todo.pop()
      if left <= 0 or not 0 <= i < len(code) or seen.get((i, inside), 0) >= left or (inside and not inside[0] <= i <= inside[1]):
        continue
      seen[i, inside] = left
      op, rest, to = code[i]
      if op == "s_endpgm" or stop(i, op, rest):
        continue
      left -= states(op, rest)
      if to is not None:
        todo.append((to, left, inside))
      if op != "s_branch":
        todo.append((i + 1, left, loop_of(i) if guard(i) else inside))

  found = []
  for i, (op, rest, _) in enumerate(code):
    if op.startswith("v_mfma"):
      sums = _registers(rest.split(",")[0])

      def reads_sum(j, op2, rest2, sums=sums, i=i):
        if op2.startswith("v_mfma"):  # a sum's own next is in order; others' operands are not
          if sums & _registers(",".join(re.split(r",(?![^\[]*\])", rest2)[1:3])):
            found.append((i, j))
        elif op2.startswith(("v_", "ds_", "buffer_", "global_", "scratch_", "flat_")) and sums & _registers(rest2):
          found.append((i, j))
        return False
      follow(i, AFTER, reads_sum)
    elif op.startswith("v_") and not op.startswith(("v_cmp", "v_readfirstlane", "v_readlane")):
      made = _registers(rest.split(",")[0])

      def multiplies(j, op2, rest2, made=made, i=i):
        if op2.startswith("v_mfma") and made & _registers(",".join(re.split(r",(?![^\[]*\])", rest2)[1:])):
          found.append((i, j))
        return False
      follow(i, BEFORE, multiplies)
  return found


@pytest.mark.parametrize("name", ["_hip_tile", "_hip_gemm", "_hip_experts"])
def test_matrix_instructions_by_hand_are_waited_for(name, tmp_path):
  if not (OPS / f"{name}.so").exists() or not shutil.which("objcopy") or not (ROCM / "llvm-objdump").exists():
    pytest.skip("no built extension, or no tools to look through it")
  bad, some = {}, 0
  for kernel, code in _kernels(name, tmp_path):
    if "wide_kernel" in kernel or "gemm_kernel" in kernel or "expert_tile_kernel" in kernel:
      some += 1
      found = _faults(code)
      if found:
        i, j = found[0]
        bad[kernel] = len(found), j - i, " ".join(code[i][:2]), " ".join(code[j][:2])
  assert some and not bad, bad


@pytest.mark.parametrize("name,kernels", [("_hip_lora", "sums_kernel"), ("_hip_gemm", "gemm_kernel")])
def test_what_is_read_across_is_multiplied(name, kernels, tmp_path):
  """Transposing reads from LDS are hidden from the compiler like the products, which may then be of other
  registers: all that they bring are operands."""
  if not (OPS / f"{name}.so").exists() or not shutil.which("objcopy") or not (ROCM / "llvm-objdump").exists():
    pytest.skip("no built extension, or no tools to look through it")
  some = 0
  for kernel, code in _kernels(name, tmp_path):
    read = set().union(*(_registers(rest.split(",")[0]) for op, rest, _ in code if op.startswith("ds_read_b64_tr")))
    multiplied = set().union(*(_registers(",".join(re.split(r",(?![^\[]*\])", rest)[1:3])) for op, rest, _ in code if op.startswith("v_mfma")))
    some += kernels in kernel and bool(read)
    assert kernels not in kernel or read <= multiplied, (kernel, sorted(read - multiplied))
  assert some
