"""The 16-byte pieces of rows that start at any byte (sofie_amd/csrc/row_chunk.h), worked out on the host by the header that the
kernels are compiled from: the bytes asked for, zeros behind the row, and no access outside the aligned dwords of the row. The
library holds no 64-bit shift whose amount lies in the last vector register of a wavefront's allocation."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include <cstring>
#include <initializer_list>
#include <sys/mman.h>
#include <unistd.h>
#define __device__
#define __forceinline__ inline
namespace sofie { typedef int v4i __attribute__((vector_size(16))); }
static unsigned __builtin_amdgcn_alignbyte(unsigned hi, unsigned lo, unsigned sh)
{
   return (unsigned)(((((unsigned long long)hi) << 32) | lo) >> (8 * (sh & 3)));
}
#include "row_chunk.h"
using namespace sofie;

template <bool SHIFTS> int check(unsigned char *page, size_t size, int K, int at, int end)
{
   // one page between two that may not be touched: the row ends `end` bytes in front of the page's end (its last dword is the
   // page's last one) or starts `at` bytes behind its start
   int bad = 0;
   for (unsigned char *row : {page + at, page + size - end - K}) {
      if (!SHIFTS && (reinterpret_cast<uintptr_t>(row) % 4 || K % 4)) continue;
      for (size_t i = 0; i < size; ++i) page[i] = 0xee;
      for (int i = 0; i < K; ++i) row[i] = (unsigned char)(1 + i * 37 % 250);
      for (int k = 0; k < K + 200; k += 16) {
         RowChunk c;
         load_row_chunk<SHIFTS>(c, row, k, K);
         const v4i v = trim_row_chunk(row_chunk<SHIFTS>(c, row, k, K), k, K);
         unsigned char got[16];
         memcpy(got, &v, 16);
         for (int i = 0; i < 16; ++i) bad += got[i] != (k + i < K ? row[k + i] : 0);
      }
   }
   return bad;
}

int main()
{
   const size_t size = (size_t)sysconf(_SC_PAGESIZE);
   unsigned char *three = (unsigned char *)mmap(nullptr, 3 * size, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS, -1, 0), *page = three + size;
   mprotect(three, size, PROT_NONE);
   mprotect(three + 2 * size, size, PROT_NONE);
   int bad = 0;
   for (int K = 16; K < 150; ++K)
      for (int o = 0; o < 4; ++o) {
         const int b = check<true>(page, size, K, o, o) + check<false>(page, size, K, o, o);
         if (b && !bad) printf("K %d offset %d: %d bytes wrong\n", K, o, b);
         bad += b;
      }
   return bad != 0;
}
"""


def test_row_chunks_on_the_host(tmp_path):
    src, exe = tmp_path / "chunk.cpp", tmp_path / "chunk"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wno-unknown-pragmas", "-I" + os.path.join(ROOT, "sofie_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], stdout=subprocess.PIPE, text=True, timeout=60)
    assert res.returncode == 0, res.stdout[-2000:]


def test_no_64_bit_shift_by_the_last_register(tmp_path):
    """Such a shift takes its amount from another register on this device. The kernels' register counts and instructions as
    the compiler listed them for the library that is loaded."""
    objdump, readelf = "/opt/rocm/llvm/bin/llvm-objdump", "/opt/rocm/llvm/bin/llvm-readelf"
    library = os.path.join(ROOT, "sofie_amd", "libsofie_hip.so")
    if not (os.path.exists(objdump) and os.path.exists(readelf)):
        pytest.skip("no llvm-objdump")
    copy = tmp_path / "library.so"
    copy.write_bytes(open(library, "rb").read())
    subprocess.run([objdump, "--offloading", str(copy)], check=True, stdout=subprocess.DEVNULL, cwd=tmp_path)
    objects = sorted(p for p in tmp_path.iterdir() if "gfx950" in p.name)
    assert objects
    shift = re.compile(r"v_(?:lshlrev_b64|lshrrev_b64|ashrrev_i64)(?:_e64)? v\[[0-9:]+\], v(\d+),")
    found, kernels = [], 0
    for obj in objects:
        notes = subprocess.run([readelf, "--notes", str(obj)], check=True, stdout=subprocess.PIPE, text=True).stdout
        count = {}
        for block in notes.split("- .agpr_count:")[1:]:
            name, vgprs = re.search(r"\.name:\s+(\S+)", block), re.search(r"\.vgpr_count:\s+(\d+)", block)
            assert name and vgprs
            count[name.group(1)] = int(vgprs.group(1))
        kernels += len(count)
        code = subprocess.Popen([objdump, "-d", "--no-show-raw-insn", str(obj)], stdout=subprocess.PIPE, text=True)
        kernel = None
        for line in code.stdout:
            if line.endswith(">:\n"):
                kernel = line[line.index("<") + 1:-3]
            elif "64" in line:
                m = shift.search(line)
                # (registers are allocated in eights)
                if m and kernel in count and int(m.group(1)) + 1 >= (count[kernel] + 7) // 8 * 8:
                    found.append((kernel, count[kernel], line.strip()))
        assert code.wait() == 0
    assert kernels > 300
    assert not found, found[:5]
