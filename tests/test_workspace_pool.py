"""The single ops' scratch pool (csrc/workspace.h) on the host, against a HIP
runtime of a few functions: its bound holds while calls return blocks together,
and an allocation that fails gets what the pool keeps."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "deltaserve-vllm_amd", "csrc")

HIP = r"""
#pragma once
#include <cstddef>
#include <cstdlib>
#include <functional>
#include <map>
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
typedef void* hipStream_t;
constexpr unsigned hipHostMallocPortable = 1;
inline std::function<void()> on_free;                    // before a block is freed
inline size_t device_bytes = ~size_t(0), device_used = 0;
inline std::map<void*, size_t> sizes;
inline hipError_t hipMalloc(void** p, size_t n) {
  if (device_used + n > device_bytes) return hipErrorOutOfMemory;
  *p = malloc(1);
  sizes[*p] = n;
  device_used += n;
  return hipSuccess;
}
inline hipError_t hipFree(void* p) {
  if (on_free) on_free();
  device_used -= sizes[p];
  sizes.erase(p);
  free(p);
  return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
inline hipError_t hipHostFree(void* p) { return hipFree(p); }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
"""

MAIN = r"""
#include "workspace.h"
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <thread>
using namespace dsb;
#define CHECK(c) do { if (!(c)) { printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)
constexpr size_t MB = 1u << 20;

int main() {
  {  // one call frees what makes room for its block while another returns its own
    BlockPool pool(false, 100 * MB);
    BlockPool::Block old[3], a = pool.get(60 * MB), b = pool.get(60 * MB);
    for (auto& o : old) o = pool.get(32 * MB);
    for (auto& o : old) pool.put(o);
    CHECK(pool.held() == 96 * MB);
    std::mutex mu;
    std::condition_variable cv;
    bool freeing = false, returned = false;
    on_free = [&] {
      std::unique_lock<std::mutex> lk(mu);
      if (freeing) return;
      freeing = true;
      cv.notify_all();
      cv.wait_for(lk, std::chrono::seconds(10), [&] { return returned; });
    };
    std::thread t([&] { pool.put(a); });
    {
      std::unique_lock<std::mutex> lk(mu);
      CHECK(cv.wait_for(lk, std::chrono::seconds(10), [&] { return freeing; }));
    }
    pool.put(b);
    {
      std::lock_guard<std::mutex> lk(mu);
      returned = true;
      cv.notify_all();
    }
    t.join();
    on_free = nullptr;
    CHECK(pool.held() <= 100 * MB);
    CHECK(pool.held() == 60 * MB);
    pool.trim(0);
    CHECK(pool.held() == 0 && device_used == 0);
  }
  {  // memory that the pool keeps idle goes to an allocation that fails without it
    device_bytes = 400 * MB;
    { Scratch s(nullptr); CHECK(s.dev<char>(200 * MB)); }
    CHECK(device_pool(0).held() >= 200 * MB);
    void* p = nullptr;
    CHECK(device_malloc(&p, 300 * MB) == hipSuccess && p);
    CHECK(device_pool(0).held() == 0);
    void* q = nullptr;
    CHECK(device_malloc(&q, 200 * MB) == hipErrorOutOfMemory);
    hipFree(p);
  }
  puts("ok");
  return 0;
}
"""


def test_pool_bound_and_out_of_memory(tmp_path):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP)
    (tmp_path / "main.cpp").write_text(MAIN)
    exe = tmp_path / "pool"
    subprocess.run(["g++", "-std=c++17", "-pthread", f"-I{tmp_path}", f"-I{CSRC}",
                    str(tmp_path / "main.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
