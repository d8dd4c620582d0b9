"""Addresses of the copies of __tc::largeHalfProduct, computed on the CPU by the device code itself: its LargeHalfOperand is
taken out of a generated source, with the loads, the LDS stores and the copy instruction replaced by checks of their operands.
Every access lies inside the operand, and so does the scalar offset of a copy whose lanes are all past the end of the reduction
(a lane's own offset is what sends it out of the buffer's bounds)."""
import os
import re
import subprocess

import pytest

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly

CLANG = "/opt/rocm/llvm/bin/clang++"

HARNESS = r"""
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#define __device__
#define __forceinline__ inline
typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef char ldschar;
struct Resource { int64_t bytes; };
template <typename T> T tmin(T a, T b) { return a < b ? a : b; }
static const uint64_t kBase = uint64_t(1) << 44;
static int64_t operandBytes, loads, copies, stores;
static bool ldsTaken[4096];
static Resource resource(void*, int, int64_t bytes, int) { return Resource{bytes}; }
#define REQUIRE(c) do { if (!(c)) { printf("%s\n", #c); exit(1); } } while (0)
static halfx8 loaded(const char* from) {
  const int64_t at = (int64_t)((uint64_t)from - kBase);
  ++loads;
  REQUIRE(at >= 0 && at + 16 <= operandBytes);
  return halfx8{1, 1, 1, 1, 1, 1, 1, 1};
}
static void stored(ldschar* to, halfx8) {
  ++stores;
  REQUIRE((uint64_t)to < 2 * 32768);
}
// raw buffer: a lane whose offset is not below the size less the scalar offset reads zeros
static void copied(int from, const Resource& rs, int scalar, bool dead) {
  ++copies;
  REQUIRE(rs.bytes == operandBytes);
  REQUIRE(scalar >= 0 && scalar < rs.bytes);
  const uint32_t lane = (uint32_t)from;
  if (dead) REQUIRE(lane >= rs.bytes - scalar);
  else REQUIRE(lane + 16 <= rs.bytes - scalar);
}
@OPERAND@
template <bool KInner, int R, int K> void check() {
  typedef LargeHalfOperand<KInner, R, K> Operand;
  operandBytes = (int64_t)R * K * 2;
  for (int first : {0, (R - 1) / 256 * 256}) {
    for (int wave = 0; wave < 8; ++wave) {
      for (int lane = 0; lane < 64; ++lane) {
        Operand o;
        o.init((const _Float16*)kBase, (ldschar*)0, first, lane, wave);
        for (int t = 0; t < Operand::kTiles; ++t) {
          for (int i = 0; i < 4; ++i) {
            o.copy(i, t, t & 1, lane);
            o.store(i, t, t & 1, lane, o.request(i, t, lane));
          }
        }
      }
    }
  }
}
int main() {
@CHECKS@
  REQUIRE(loads == copies && loads == stores && loads > 0);
  puts("in bounds");
}
"""


def operand():
    text, _ = tc.map_only("def f(float16(M, K) A, float16(N, K) B) -> (O) { O(m, n) +=! float(A(m, r_k)) * float(B(n, r_k)) }", "f",
                          [ShapeOnly((4096, 4096), "float16")] * 2,
                          "naive;tile=256,256,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    body = text[text.index("template <bool KInner, int R, int K> struct LargeHalfOperand"):text.index("// All wavefronts have read")]
    reads = body.index("  // the values of step `s`")          # (reads of LDS: not looked at here)
    body = body[:reads] + "};\n"

    def once(pattern, replacement):
        nonlocal body
        body, n = re.subn(pattern, replacement, body, flags=re.S)
        assert n == 1, (pattern, n)

    once(r"__builtin_amdgcn_make_buffer_rsrc\(", "resource(")
    once(r"__amdgpu_buffer_rsrc_t", "Resource")
    once(r'asm volatile\("s_mov_b32 m0[^;]*?"v"\(from\),\s*"s"\(rs\),\s*"s"\((.*?)\)\s*: "[^;]*;', r"copied(from, rs, \1, isDead(i, t, lane));")
    once(r"\*\(const halfx8u\*\)(\(.*?\));", r"loaded\1;")
    once(r"\*\(__attribute__\(\(address_space\(3\)\)\) halfx8\*\)\((.*?)\) = v;", r"stored(\1, v);")
    return body


# (rows of the operand, points of the reduction) by order: innermost, the points are a multiple of eight, else the rows are
INNERMOST = [(r, k) for r in (8, 255, 256, 264, 4096) for k in (256, 264, 320, 328, 376)] + [(1048575, 1016)]
OUTERMOST = [(r, k) for r in (8, 248, 256, 264, 4096) for k in (256, 257, 258, 259, 260, 261, 264, 319, 320, 321, 324, 325)] + [
    (4177912, 257), (4129768, 260)]                         # just below 2 GiB


@pytest.mark.skipif(not os.path.exists(CLANG), reason="no clang")
def test_copies_stay_inside_their_operand(tmp_path):
    checks = "".join(f"  check<true, {r}, {k}>();\n" for r, k in INNERMOST) + "".join(f"  check<false, {r}, {k}>();\n" for r, k in OUTERMOST)
    source = tmp_path / "addresses.cc"
    source.write_text(HARNESS.replace("@OPERAND@", operand()).replace("@CHECKS@", checks))
    binary = str(tmp_path / "addresses")
    subprocess.run([CLANG, "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize=null,alignment,pointer-overflow", "-fno-sanitize-recover=all", "-Wno-unknown-attributes",
                    str(source), "-o", binary], check=True)
    run = subprocess.run([binary], capture_output=True, text=True)
    assert run.returncode == 0 and run.stdout == "in bounds\n", run.stdout + run.stderr


def test_copies_wait_for_the_register_they_read():
    """m0, the place in LDS, is written by the instruction in front: one wait state has to lie between them (the compiler puts
    s_nop there where it makes the copy itself), and the assembly says that it writes m0."""
    text, _ = tc.map_only("def f(float16(M, K) A, float16(N, K) B) -> (O) { O(m, n) +=! float(A(m, r_k)) * float(B(n, r_k)) }", "f",
                          [ShapeOnly((4096, 4096), "float16")] * 2,
                          "naive;tile=256,256,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    blocks = [b for b in re.findall(r"asm volatile\((.*?)\);\n", text, flags=re.S) if "m0" in b]
    assert blocks and all(re.search(r"s_mov_b32 m0, %0\\n\\ts_nop \d\\n\\tbuffer_load", b) and b.rstrip().endswith('"m0"') for b in blocks)
