"""What the compiler is told, and what it makes of it, where results cannot show a mistake: inline assembly that writes a register
must say so, and loads that are meant to stay on their way must not be waited for."""

import ctypes
import glob
import os
import re
import shutil
import subprocess

import pytest
import torch

from ampere_kv_engine_amd.csrc import build

OBJDUMP = next((p for p in (shutil.which("llvm-objdump"), "/opt/rocm/llvm/bin/llvm-objdump") if p and os.path.exists(p)), None)


def test_inline_assembly_that_writes_m0_says_so():
    blocks = []
    for path in sorted(glob.glob(os.path.join(build.HERE, "*.hip")) + glob.glob(os.path.join(build.HERE, "*.h"))):
        with open(path) as handle:
            blocks += [(os.path.basename(path), block) for block in re.findall(r"\basm volatile\((.*?)\);", handle.read(), re.S)]
    writers = [(name, block) for name, block in blocks if re.search(r"s_mov_b32 m0", block)]
    assert writers, "no block writes m0 any more: this test can go"
    for name, block in writers:
        assert block.count(":") == 3 and '"m0"' in block.split(":")[3], f"{name}: {block}"


def _device_codes(library, folder):
    """A built library's code for the device, a file per source."""
    if library is None or OBJDUMP is None:
        pytest.skip("the library is not built, or there is nothing to list it with")
    copied = shutil.copy(library, folder)
    subprocess.run([OBJDUMP, "--offloading", copied], cwd=folder, check=True, capture_output=True)
    return glob.glob(os.path.join(folder, "*gfx950"))


def _device_code(dim, folder):
    code, = _device_codes(build.attention_library_path(dim), folder)
    return code


def _kernel_facts(codes):
    """Per kernel what the compiler says of it: mangled name -> dict of numbers."""
    readelf = os.path.join(os.path.dirname(OBJDUMP), "llvm-readelf")
    facts = {}
    for code in codes:
        notes = subprocess.run([readelf, "--notes", code], check=True, capture_output=True, text=True).stdout
        for kernel in re.split(r"\n  - ", notes)[1:]:
            name = re.search(r"^ *\.name: +(_Z\S+)$", kernel, re.M)
            if name:
                facts[name[1]] = {key: int(value) for key, value in re.findall(r"^ *\.(\w+): +(\d+)$", kernel, re.M)}
    return facts


def _kernel(code, name):
    """(address, instruction, target) of the first kernel whose mangled name holds `name`."""
    listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code], check=True, capture_output=True, text=True).stdout
    kernel = re.split(r"\n\n", listing[listing.index(name):])[0]
    lines = [re.match(r"\s+(\S.*?)\s*// ([0-9A-F]+):(?:.*<.*\+0x([0-9a-f]+)>)?", line) for line in kernel.splitlines()]
    return [(int(m[2], 16), m[1], int(m[3], 16) if m[3] else None) for m in lines if m]


def _prompt_kernel(dim, pages_per_step, folder):
    return _kernel(_device_code(dim, folder), f"attention_prompt_kernelILi{pages_per_step}E")


@pytest.mark.parametrize("dim", build.DEFAULT_HEAD_DIMS)
def test_single_tokens_ask_ahead_only_where_registers_hold_it(dim, tmp_path):
    """Kernels of single tokens that ask for a step's keys and values while the step before is computed hold two steps' values: none
    of them keeps registers in memory (the compiler's own count), and the launch that holds prompt portions too, which the portions'
    registers bound to two waves a SIMD at heads of 192, keeps no more than without (188 to 212 bytes a lane; asking ahead 480)."""
    kernels = [(name, facts["private_segment_fixed_size"]) for name, facts in _kernel_facts([_device_code(dim, str(tmp_path))]).items()]
    ahead = [(name, scratch) for name, scratch in kernels if re.search(r"attention_(items|mfma)_kernelI\S*Lb1EEEv", name)
             and ("items" in name or re.search(r"kernelILi1E(Lb[01]E){4}Lb1EEEv", name))]
    pair = [(name, scratch) for name, scratch in kernels if "attention_pair_kernel" in name]
    assert len(ahead) >= 2 and (len(pair) == 6 or dim % 64 != 0)
    assert [(name, scratch) for name, scratch in ahead if scratch != 0] == []
    assert [(name, scratch) for name, scratch in pair if scratch > (216 if dim == 192 else 0)] == []


@pytest.mark.parametrize("dim", [64, 128, 192, 256])
def test_waves_without_keys_ask_for_none(dim, tmp_path):
    """The kernel whose four waves share an item, asking ahead: before its first load of keys (the first that is marked read-once)
    stands a branch over all of the matrix instructions to where the wave's empty result is left in LDS."""
    code = _kernel(_device_code(dim, str(tmp_path)), "attention_items_kernelILb1ELb1ELNS_5ItemsE1ELb1EEEv")
    start = code[0][0]
    first_load = next(i for i, (_, text, _) in enumerate(code) if text.startswith("global_load") and text.endswith(" nt"))
    last_product = max(i for i, (_, text, _) in enumerate(code) if "v_mfma" in text)
    landings = [next((i for i, (at, _, _) in enumerate(code) if at == start + target), None)
                for _, text, target in code[:first_load] if text.startswith(("s_cbranch", "s_branch")) and target is not None]
    results = [i for i in landings if i is not None and i > last_product
               and any(text.startswith("ds_write") for _, text, _ in code[i:]) and not code[i][1].startswith("s_endpgm")]
    assert results


@pytest.mark.parametrize("pages_per_step", [1, 2])
@pytest.mark.parametrize("dim", [64, 128])
def test_calm_turns_of_the_prompt_attention_wait_for_counted_loads_alone(dim, pages_per_step, tmp_path):
    """The loop of four calm turns (a turn multiplies D / 16 times for the scores and D / 8 times for the sums and asks for D / 64
    pieces of keys and as many of values) waits for memory four times, and each time leaves the loads of two turns on their way."""
    code = _prompt_kernel(dim, pages_per_step, str(tmp_path))
    start = code[0][0]
    loops = []
    for index, (at, text, target) in enumerate(code):
        if text.startswith(("s_cbranch", "s_branch")) and target is not None and start + target <= at:
            body = [t for a, t, _ in code[:index + 1] if a >= start + target]
            if (sum("v_mfma" in t for t in body), sum("global_load_lds" in t for t in body)) == (4 * (dim // 16 + dim // 8), 4 * 2 * dim // 64):
                loops.append(body)
    assert len(loops) == 1
    waits = [re.search(r"vmcnt\((\d+)\)", t) for t in loops[0] if t.startswith("s_waitcnt")]
    assert [int(w[1]) for w in waits if w] == [4 * dim // 64] * 4


@pytest.mark.parametrize("kernel,waves", [("ILi1ELb0ELb0ELb0ELb1EE", 20), ("ILi2ELb0ELb0ELb0ELb1EE", 16), ("ILi2ELb1ELb0ELb0ELb1EE", 12)])
def test_decode_products_that_scale_their_sums_leave_a_unit_its_waves(kernel, waves, tmp_path):
    """One row tile a wave, two, and gated: what the product asks for early must not cost a unit a wave (512 registers a lane and
    SIMD, handed out in eights)."""
    facts = _kernel_facts(_device_codes(build.library_path(), str(tmp_path)))
    registers, = [f["vgpr_count"] for name, f in facts.items() if "linear_decode_kernel" + kernel in name]
    assert 4 * (512 // (-(-registers // 8) * 8)) >= waves, registers


@pytest.mark.skipif(torch.cuda.is_available(), reason="the operands are no memory: nothing may be launched")
def test_gated_single_tokens_of_any_number_are_taken():
    """4,096 tokens of a million heads are more (token, head) rows than 31 bits count: they are taken in several launches, not refused."""
    library = ctypes.CDLL(build.ensure_parts())
    entry, operand, nothing = library.akv_gated_attention_singles, ctypes.c_void_p(4096), ctypes.c_void_p(0)
    entry.restype = ctypes.c_int
    long, real = ctypes.c_long, ctypes.c_float
    status = lambda q_heads, segments: entry(
        operand, operand, operand, nothing, long(0), 0, operand, operand, operand, nothing, 1, operand, operand, segments, 4096, 4096,
        q_heads, 1, 64, 64, 16, long(1), real(1.0), real(0.0), 0, 0, 0, long(q_heads * 64), real(1.0), nothing, 1, 0, nothing, nothing)
    assert status(1 << 20, 1) == -2                 # (its tiles of 16 heads do not fit the grid)
    assert status(1 << 19, 1 << 20) == -2           # (nor tokens x segments)
    assert status(1 << 19, 2) not in (0, -1, -2)    # (taken: what fails is the launch, for want of a device)


@pytest.mark.parametrize("kernel", ["linear_mid_kernel", "linear_decode_kernel", "sample_parts_kernel"])
def test_sums_for_other_blocks_have_arrived_before_the_tick(kernel, tmp_path):
    """Blocks that hand sums to each other store them with device scope and tick a counter.  Whoever stores waits until its stores
    have been acknowledged: the wave that ticks before its tick, every other wave before the barrier that lets the first one tick."""
    checked = 0
    for code in _device_codes(build.library_path(), str(tmp_path)):
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", code], check=True, capture_output=True, text=True).stdout
        for body in re.split(r"\n\n", listing):
            if not re.match(rf"\s*[0-9a-f]+ <_Z\S*{kernel}", body):
                continue
            instructions = [re.sub(r"\s*//.*", "", line).strip() for line in body.splitlines()[1:]]
            waiting = False                  # device-scope stores that nothing has waited for
            for text in instructions:
                if text.startswith("global_store") and "sc1" in text.split():
                    waiting, checked = True, checked + 1
                elif re.match(r"s_waitcnt .*vmcnt\(0\)", text):
                    waiting = False
                assert not (waiting and text.startswith(("s_barrier", "global_atomic_add"))), body.splitlines()[0]
    assert checked


def test_divider_is_exact(tmp_path):
    """`Divider` (common.h) against the language's division: every small divisor, those beside powers of two and large ones, at the
    multiples where a quotient changes and at the ends of its range."""
    source = tmp_path / "divider.hip"
    source.write_text("""
#include "common.h"
#include <cstdio>
int main() {
  long wrong = 0;
  auto check = [&](long by) {
    const akv::Divider d = akv::Divider::of(static_cast<int>(by));
    const long last = 0x7fffffffL / by;
    for (long q : {0L, 1L, 2L, 3L, last / 3, last / 2, last - 1, last})
      for (long x = q * by - 1; x <= q * by + 1; ++x)
        if (x >= 0 && x <= 0x7fffffffL) {
          const int got = d.quotient(static_cast<int>(x));
          wrong += got != x / by || d.rest(static_cast<int>(x), got) != x % by;
        }
    wrong += d.quotient(0x7fffffff) != 0x7fffffffL / by;
  };
  for (long by = 1; by <= 5000; ++by) check(by);
  for (int bit = 2; bit < 31; ++bit)
    for (long by = (1L << bit) - 1; by <= (1L << bit) + 1; ++by) check(by);
  for (long by = 0x7fffffffL; by > 5000; by -= 1 + by / 977) check(by);
  std::printf("%ld\\n", wrong);
  return 0;
}
""")
    program = tmp_path / "divider"
    subprocess.run([build._hipcc(), "-O1", "-std=c++17", f"--offload-arch={build.ARCH}", f"-I{build.HERE}", str(source), "-o", str(program)],
                   check=True, capture_output=True)
    assert subprocess.run([str(program)], check=True, capture_output=True, text=True).stdout.strip() == "0"
