"""The workspace-size queries are arithmetic: they make no call into the HIP
runtime (a process may ask before it forks, or without a GPU) and give the
same size whatever the current device's CU count is."""
import subprocess
import sys

import pytest

import strata_hip as H

# Stands in for the runtime's device queries (loaded ahead of it, so the
# library's references find these): counts the calls, reports `cus` CUs.
STAND_IN = """
static int calls, cus = 256;
int hipGetDevice(int *d) { ++calls; *d = 0; return 0; }
int hipDeviceGetAttribute(int *v, int attr, int dev) { ++calls; (void)attr; (void)dev; *v = cus; return 0; }
int stand_in_calls(void) { return calls; }
void stand_in_cus(int n) { cus = n; }
"""

PROBE = """
import ctypes as C, sys
top = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
top.stand_in_cus(int(sys.argv[3]))
lib = C.CDLL(sys.argv[2])
v = C.c_uint64()
u64, out = C.c_uint64, C.byref(v)
sizes = []
for rows, cols, m, mode in ((4096, 12288, 333, 1), (12288, 4096, 100, 0), (96, 2304, 9, 1), (700, 1792, 257, 0)):
    assert lib.sh_matmul_workspace_bytes(12, u64(rows), u64(cols), m, mode, out) == 0
    sizes.append(v.value)
for n_tok, n_embd, n_ff in ((17, 4096, 12288), (77, 4096, 12288), (33, 1024, 512), (1, 2048, 768)):
    assert lib.sh_ffn_workspace_bytes(n_tok, u64(n_embd), u64(n_ff), out) == 0
    sizes.append(v.value)
for n_tok in (1, 16, 96):
    assert lib.sh_moe_workspace_bytes(n_tok, 8, u64(128), u64(2048), u64(768), 12, 14, out) == 0
    sizes.append(v.value)
    q = (C.c_uint32 * 8)(0, 12, 12, 14, 12, 12, 14, 0)
    assert lib.sh_moe_layer_workspace_bytes(n_tok, 8, u64(128), u64(2048), u64(768), u64(768), q, out) == 0
    sizes.append(v.value)
assert lib.sh_gemv_workspace_bytes(12, u64(4096), u64(4096), 8, out) == 0
sizes.append(v.value)
print(top.stand_in_calls(), *sizes)
"""


@pytest.mark.timeout(120)
def test_size_queries_leave_the_device_alone(tmp_path):
    src, so = tmp_path / "stand_in.c", tmp_path / "stand_in.so"
    src.write_text(STAND_IN)
    subprocess.run(["cc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    got = []
    for cus in (256, 32):
        r = subprocess.run([sys.executable, "-c", PROBE, str(so), H.load_library()._name, str(cus)],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        calls, *sizes = r.stdout.split()
        assert calls == "0"
        got.append(sizes)
    assert got[0] == got[1]
