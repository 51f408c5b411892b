"""The 32-bit byte offsets of Jacobian rows, host code with the overflow check on: right up to the last row
below 2^32 bytes, for every row length of the tile kernels, and not used beyond."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "common.h"
#include <cstdio>
using namespace tdi;
int main()
{
    for (int K = 1; K <= 112; ++K) {
        const int ldI = dI_stride(K);
        const long long area = (1ll << 32) / (4 * ldI);      // the first area whose rows reach 2^32 bytes, or the last below
        for (long long a = area - 2; a <= area + 2; ++a) {
            const bool far = rows_far((int)a, K);
            if (far != (a * ldI * 4 >= (1ll << 32))) return printf("rule: K %d area %lld\n", K, a), 1;
            if (far) continue;
            for (long long pos : {0ll, a / 3, a / 2, a / 2 + 1, a - 1})
                if (dI_offset((int)pos, ldI) != (unsigned long long)pos * ldI * 4) return printf("K %d row %lld\n", K, pos), 1;
        }
    }
    return 0;
}
"""


def test_offsets_up_to_the_limit(tmp_path):
    src, exe = tmp_path / "rows.hip", tmp_path / "rows"
    src.write_text(SOURCE)
    subprocess.check_call([os.environ.get("HIPCC", "/opt/rocm/bin/hipcc"), "--offload-host-only", "-std=c++17", "-O1",
                           "-Xarch_host", "-fsanitize=undefined", "-Xarch_host", "-fno-sanitize-recover=all",
                           "-I" + os.path.join(ROOT, "3di_amd", "csrc"), str(src), "-o", str(exe)])
    subprocess.check_call([str(exe)])
