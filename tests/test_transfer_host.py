"""The staged copies' host side against stand-ins for the HIP calls (fake_hip.h),
without a GPU: what a failing call leaves behind."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def run(tmp_path, body):
    main = tmp_path / "main.cpp"
    main.write_text('#include "fake_hip.h"\n#include "transfer.h"\n#include <vector>\n'
                    "#define CHECK(x) do { if (!(x)) { printf(\"%s\\n\", #x); return 1; } } while (0)\n"
                    "int main() {\n" + body + "  return 0;\n}\n")
    exe, rocm = str(tmp_path / "main"), os.environ.get("ROCM_PATH", "/opt/rocm")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-pthread",
                    f"-I{rocm}/include", "-I", os.path.join(ROOT, "tests"),
                    "-I", os.path.join(ROOT, "pypde_amd", "csrc"), "-o", exe, str(main),
                    os.path.join(ROOT, "pypde_amd", "csrc", "transfer.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout


def test_copies_arrive(tmp_path):
    run(tmp_path, """
  for (size_t n : {size_t(8), size_t(1) << 20, (size_t(1) << 20) + 8, (size_t(21) << 20) + 24}) {
    std::vector<char> a(n), dev(n), b(n);
    for (size_t i = 0; i < n; i++) a[i] = (char)(i * 31 + i / 4096);
    CHECK(pypde::copy_to_device(dev.data(), a.data(), n, 0, nullptr) == hipSuccess);
    CHECK(dev == a && fake::pending.empty());
    CHECK(pypde::copy_to_host(b.data(), dev.data(), n, 0, nullptr) == hipSuccess);
    CHECK(b == a && fake::pending.empty());
  }
  pypde::release_idle_transfer();
  CHECK(fake::live_buffers == 0);
""")


def test_no_copy_is_in_flight_after_a_failed_event(tmp_path):
    """A buffer goes back to the pool, where the next copy overwrites it, only
    when nothing reads or writes it any more."""
    run(tmp_path, """
  const size_t n = (size_t(3) << 20) + 8;
  std::vector<char> a(n, 1), dev(n);
  for (int fail = 0; fail < 4; fail++) {
    fake::records_left = fail;
    CHECK(pypde::copy_to_device(dev.data(), a.data(), n, 0, nullptr) != hipSuccess);
    CHECK(fake::pending.empty());
    fake::records_left = fail;
    CHECK(pypde::copy_to_host(a.data(), dev.data(), n, 0, nullptr) != hipSuccess);
    CHECK(fake::pending.empty());
  }
""")


def test_memory_of_the_runtime_is_left_to_it(tmp_path):
    """Pinned, managed and device memory go to the runtime in one copy; the
    host touches none of it and allocates no buffer."""
    run(tmp_path, """
  const size_t n = (size_t(2) << 20) + 8;
  std::vector<char> a(n, 7), dev(n), b(n);
  for (hipMemoryType t : {hipMemoryTypeHost, hipMemoryTypeDevice, hipMemoryTypeManaged}) {
    std::fill(dev.begin(), dev.end(), 0);
    std::fill(b.begin(), b.end(), 0);
    fake::known[a.data()] = t;
    fake::known[b.data()] = t;
    const size_t before = fake::done;
    CHECK(pypde::copy_to_device(dev.data(), a.data(), n, 0, nullptr) == hipSuccess);
    CHECK(pypde::copy_to_host(b.data(), dev.data(), n, 0, nullptr) == hipSuccess);
    CHECK(fake::host_allocations == 0 && fake::done == before + 2);
    CHECK(b == a && fake::pending.empty());
  }
""")
