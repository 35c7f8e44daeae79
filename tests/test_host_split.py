"""CPU check of the k-means driver's empty-cluster split where there is no
device memory for its workspace: the driver's source, compiled with stand-ins
for the device layer, must hand the split to the host, not fail."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r'''
#include "yael_kmeans.c"

static int picks;
void *yh_buf(int slot, size_t bytes) { (void)slot; (void)bytes; return NULL; }
size_t yk_split_ws_bytes(int ne, int d) { return (size_t)ne * d * 4; }
int yk_split_pick(const int *counts, int k, int ne, const double *rd, const int *empties,
                  void *ws) {
  (void)counts; (void)k; (void)ne; (void)rd; (void)empties; (void)ws;
  picks++;
  return YK_OK;
}

int main(void) {
  int counts[4] = {3, 0, 5, 0}, done = 7;
  int rc = yh_split_device(8, 4, NULL, NULL, counts, 2, 1u, &done);
  printf("rc %d done %d picks %d\n", rc, done, picks);
  return 0;
}
'''


def test_split_without_device_memory_is_the_hosts(tmp_path):
    src, exe = tmp_path / "split.c", tmp_path / "split"
    src.write_text(PROGRAM)
    host = os.path.join(ROOT, "yael_amd", "csrc", "host")
    subprocess.check_call(["gcc", "-std=gnu99", "-O1", "-w", "-I", host, "-o", str(exe), str(src),
                           "-lm", "-lpthread", "-Wl,--unresolved-symbols=ignore-all"])
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert out.stdout == "rc 0 done 0 picks 0\n", (out.returncode, out.stdout, out.stderr)
