"""The size rules of llamanyon.rs_amd/csrc/dispatch.hpp, compiled for the host
with g++ and called through ctypes: the same source that the GPU library
dispatches by, without a GPU."""
import ctypes
import os
import subprocess

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
Q4_0, Q8_0, Q4_K, Q6_K = 2, 8, 12, 14
CUS = 256  # MI355X
SMALL, SPLIT, ROUNDS = 0, 1, 2  # GemmPlan::Kind

SHIM = """
#include "dispatch.hpp"
extern "C" {
int plan(unsigned dt, int m, int rows, int cols, int cus, long *out) {
  const swamp::GemmPlan p = swamp::plan_gemm_bf16(dt, m, rows, cols, cus);
  out[0] = p.parts; out[1] = p.pieces; out[2] = p.kps; out[3] = long(p.part_bytes);
  return int(p.kind);
}
int dequantize_once(unsigned dt, int m, int rows, int cols, int cus) {
  return swamp::gemm_dequantize_once(dt, m, rows, cols, cus);
}
int in_registers(unsigned dt, int n, int rows, int cols, int cus) {
  return swamp::small_batch_in_registers(dt, n, rows, cols, cus);
}
int k_groups(int n, int rows, int cols, int cus) {
  return swamp::small_batch_k_groups(n, rows, cols, cus);
}
int product_staged(unsigned dt, int rows, int cols, int add, int cus) {
  return swamp::swiglu_product_staged(dt, rows, cols, add != 0, cus);
}
}
"""


class Rules:
    def __init__(self, folder):
        src, lib = os.path.join(folder, "rules.cpp"), os.path.join(folder, "rules.so")
        with open(src, "w") as f:
            f.write(SHIM)
        subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC",
                        "-I" + os.path.join(REPO, "include"),
                        "-I" + os.path.join(REPO, "llamanyon.rs_amd", "csrc"), src, "-o", lib],
                       check=True)
        self.lib = ctypes.CDLL(lib)

    def plan(self, dt, m, rows, cols, cus=CUS):
        """(kind, parts, pieces, K steps per piece, bytes of partial sums)"""
        out = (ctypes.c_long * 4)()
        return (self.lib.plan(dt, m, rows, cols, cus, out), *out)

    def dequantize_once(self, dt, m, rows, cols, cus=CUS):
        return bool(self.lib.dequantize_once(dt, m, rows, cols, cus))

    def in_registers(self, dt, n, rows, cols, cus=CUS):
        return bool(self.lib.in_registers(dt, n, rows, cols, cus))

    def product_staged(self, dt, rows, cols, add=False, cus=CUS):
        return bool(self.lib.product_staged(dt, rows, cols, int(add), cus))

    def k_groups(self, n, rows, cols, cus=CUS):
        return bool(self.lib.k_groups(n, rows, cols, cus))
