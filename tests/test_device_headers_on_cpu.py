"""Parts of the device headers compiled for the CPU: what no result shows
(which of two ways a solve takes, an error in the middle of a transfer) is
looked at there.  A header of a few lines stands in for HIP's."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gazpart_amd",
                    "csrc")

HIP_STUB = r"""
#pragma once
#include <algorithm>
#include <cmath>
#include <cstring>
using std::max; using std::min;
#define __device__
#define __host__
#define __forceinline__ inline
#define __noinline__ __attribute__((noinline))
inline int __double2hiint(double x) {
  unsigned long long u;
  std::memcpy(&u, &x, 8);
  return (int)(u >> 32);
}
"""


def run(tmp_path, stub, src, *flags):
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(stub)
    (tmp_path / "t.cpp").write_text(src)
    exe = str(tmp_path / "t")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", f"-I{tmp_path}", f"-I{CSRC}", *flags,
                    str(tmp_path / "t.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, (r.returncode, r.stdout, r.stderr)
    return r.stdout


CONTACT = r"""
#include <cstdio>
#include <random>
#include "gp_contact.h"
using namespace gp;
int main() {
  std::mt19937_64 g(5);
  std::normal_distribution<double> nd;
  std::uniform_real_distribution<double> un(0, 1);
  // spheres; spheroids with the x axis, and with any common axis; spheroids;
  // tri-axial bodies; a sphere and a spheroid
  for (int kind = 0; kind < 6; ++kind) {
    const int n = 4000;
    int left = 0, differ = 0;
    for (int k = 0; k < n; ++k) {
      const double a = 0.02;
      double b = kind == 0 || kind == 5 ? a : a / (1 + 2 * un(g)), c = b;
      if (kind == 4) c = a / (1 + 2 * un(g));
      const double b2 = kind == 5 ? a / 2 : b, c2 = kind == 5 ? a / 2 : c;
      double q1[4] = {1, 0, 0, 0}, q2[4] = {1, 0, 0, 0}, d[3], bi[3], bj[3], r = 0;
      auto turn = [&](double* q) {
        double s = 0;
        for (int i = 0; i < 4; ++i) { q[i] = nd(g); s += q[i] * q[i]; }
        for (int i = 0; i < 4; ++i) q[i] /= std::sqrt(s);
      };
      if (kind != 1) { turn(q1); turn(q2); }
      if (kind == 2) std::copy(q1, q1 + 4, q2);
      for (double& x : d) { x = nd(g); r += x * x; }
      r = (0.5 + 0.6 * un(g)) * 2 * a / std::sqrt(r);
      ContactPair cp;
      for (int i = 0; i < 3; ++i) {
        cp.b1[i] = 1 + un(g);
        cp.b2[i] = cp.b1[i] + r * d[i];
      }
      cp.E1 = ell_matrix(q1, a, b, c);
      cp.E2 = ell_matrix(q2, a, b2, c2);
      double e[3], s = 0;   // the start on the line of centres
      for (int i = 0; i < 3; ++i) { e[i] = cp.b1[i] - cp.b2[i]; s += e[i] * e[i]; }
      LmState t{};
      t.x[1] = std::asin(e[2] / std::sqrt(s));
      t.x[0] = std::acos(std::min(1.0, std::max(-1.0, e[0] / std::sqrt(s) / std::cos(t.x[1]))));
      t.iter = 1;
      LmState f = t;
      lm_rest(&cp, &f, 300);
      if (!lm_run<true>(cp, t, 300)) {
        ++left;
        lm_rest(&cp, &t, 300);
      }
      differ += t.nfev != f.nfev || t.info != f.info || t.x[0] != f.x[0] || t.x[1] != f.x[1];
    }
    std::printf("%d %d\n", left, differ);
  }
}
"""


def test_contact_solves_stay_in_the_plain_loop(tmp_path):
    """Bodies of any symmetry solve in the loop without scaled sums (an exact
    zero or its residue in a component leaves the norm as it is), with the
    iterates of the run that has them.  A solve may leave where every
    component is tiny: at most 1 in 1000."""
    out = run(tmp_path, HIP_STUB, CONTACT, "-ffp-contract=off")
    for left, differ in (map(int, line.split()) for line in out.splitlines()):
        assert left <= 4 and differ == 0, out


XFER_STUB = r"""
#pragma once
#include <atomic>
#include <cstdlib>
#include <cstring>
typedef int hipError_t;
typedef void* hipEvent_t;
typedef void* hipStream_t;
enum { hipSuccess = 0, hipErrorUnknown = 999 };
enum { hipEventDisableTiming, hipMemcpyDeviceToHost, hipMemcpyHostToDevice };
inline std::atomic<int> calls{0}, copies{0}, last_copy{0}, waited{0}, fail_at{-1}, allocs{0};
inline std::atomic<size_t> largest{0};
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, int) { *e = e; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n) {
  ++allocs;
  if (n > largest) largest = n;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n) { return hipHostMalloc(p, n); }
inline hipError_t hipFree(void* p) { return hipHostFree(p); }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, int, hipStream_t) {
  if (copies++ == fail_at) return hipErrorUnknown;
  std::memcpy(d, s, n);
  last_copy = ++calls;
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t) { waited = ++calls; return hipSuccess; }
"""

XFER = r"""
#include <cstdio>
#include <new>
#include <vector>
#include "gp_xfer.h"
static std::atomic<int> news_left{-1};   // -1: any number
void* operator new(size_t n) {
  if (news_left >= 0 && news_left-- == 0) throw std::bad_alloc();
  return std::malloc(n);
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }
int main() {
  const size_t n = (size_t)37 << 20;
  std::vector<char> a(n), b(n);
  for (size_t i = 0; i < n; ++i) a[i] = (char)(i * 7 + (i >> 12));
  gpx::Xfer x;
  // memory for no, one, two threads
  for (int k = 0; k < 3; ++k) {
    for (int way = 0; way < 2; ++way) {
      std::fill(b.begin(), b.end(), 0);
      news_left = k;
      const hipError_t e = way ? x.h2d(b.data(), a.data(), n, nullptr) : x.d2h(b.data(), a.data(), n, nullptr);
      news_left = -1;
      if (e != hipSuccess || a != b) return 1;
    }
  }
  // an error ends a transfer when the copies before it are complete
  for (int at = 0; at < 9; at += 2) {
    copies = 0;
    fail_at = at;
    auto f = [&](int w, long long) { return hipMemcpyAsync(x.pin[w], a.data(), 1000, 0, nullptr); };
    if (gpx::Xfer::run(4, 9, nullptr, f) != hipErrorUnknown) return 2;
    if (waited < last_copy) return 3;
  }
  x.release();
  // a list that grows by a few entries a call, to the largest chunk and past it
  gpx::Xfer y;
  fail_at = -1;
  allocs = 0;
  largest = 0;
  for (size_t m = 100; m < n; m += m < 200000 ? 4100 : 99991)
    if (y.d2h(b.data(), a.data(), m, nullptr) != hipSuccess) return 4;
  y.release();
  // 4 KB to 4 MB in doublings, once a worker
  if (allocs > 11 * gpx::XFER_WORKERS || largest > gpx::XFER_CHUNK) return 5;
}
"""


def test_transfer_without_threads_and_after_an_error(tmp_path):
    """A worker that cannot be started leaves its chunks to the others, and no
    exception crosses the C entry; a transfer that fails returns when nothing
    it has queued uses its buffers any more; buffers grow by doubling, to a chunk at
    most."""
    run(tmp_path, XFER_STUB, XFER)


ORDER = r"""
#include <cstdio>
#include <vector>
#include "gp_order.h"
using namespace gp;
int main() {
  const int nzs[] = {1, 2, 3, 7, 20, 54, 244, 320};
  for (int nz : nzs)
    for (int nb = 1; nb < 40 * nz + 700; nb += nb < 300 ? 1 : 97) {
      const int nbox = nz * nz * nz, np = 256 * nb - 17;
      const LayerMap lm = layer_map(nb, np, nbox, nz);
      const bool want = nb >= 32 * nz && np < 6 * nbox;
      if ((lm.layers == nz) != want || (lm.layers != 0) != want) return 1;
      LayerMap m;   // the order itself, also where the rule does not take it
      m.nb = nb;
      m.layers = nz;
      m.per = (nb + 8 * nz - 1) / (8 * nz);
      if (want && (lm.nb != m.nb || lm.per != m.per)) return 2;
      std::vector<int> seen(nb + 1, 0);
      for (int b = 0; b < layer_grid(m); ++b) {
        const int i = layer_item(m, b);
        if (i < 0 || i > nb) return 3;
        seen[i]++;
      }
      for (int i = 0; i < nb; ++i)
        if (seen[i] != 1) return 4;
    }
  // the largest products
  LayerMap m;
  m.nb = 8388607; m.layers = 1290; m.per = (m.nb + 8 * 1290 - 1) / (8 * 1290);
  std::printf("%d\n", layer_item(m, layer_grid(m) - 8 * m.per + 7));
}
"""


def test_layer_order_of_the_library(tmp_path):
    """The advance's workgroup order as the library has it takes every
    workgroup exactly once, and is on only where cells hold fewer than six
    particles on average."""
    out = run(tmp_path, HIP_STUB, ORDER)
    nb, n = 8388607, 8 * 1290
    assert int(out) == (n - 1) * nb // n
