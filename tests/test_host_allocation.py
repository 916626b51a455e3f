"""The host codec where memory runs out: with each of its allocations failing in turn, every entry
point returns a status (a thread that is not joined on the way out would end the process)."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "georefine_amd" / "csrc"

_PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include "host_codec.cpp"

static std::atomic<long> until_failure{-1};  // allocations that still succeed; negative: all
void *operator new(size_t n) {
  if (until_failure.load() >= 0 && until_failure.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

template <class Call>
int each_allocation(const char *name, Call call) {
  for (long k = 0; k < 1000; ++k) {
    until_failure = k;
    const int status = call();
    const bool failed = until_failure.exchange(-1) < 0;
    if (failed != (status != 0)) return std::printf("%s: allocation %ld %s, status %d\n", name, k, failed ? "failed" : "was not reached", status), 1;
    if (!failed) return std::printf("%s: %ld\n", name, k), 0;
    std::fflush(stdout);
  }
  return 1;
}

int main() {
  const uint32_t rows = 4096, cols = 1024, nr = 4, nc = 4;  // four million words: counted on four threads
  const size_t n = (size_t)rows * cols;
  std::vector<uint16_t> words(n), out(n);
  uint32_t x = 1;
  for (auto &w : words) x = x * 1664525u + 1013904223u, w = (uint16_t)((x >> 30) << 7 | (x >> 20 & 31));
  std::vector<uint8_t> rc(rows), cc(cols), buffer(2 * n + 8);
  for (uint32_t i = 0; i < rows; ++i) rc[i] = (uint8_t)(i % nr);
  for (uint32_t i = 0; i < cols; ++i) cc[i] = (uint8_t)(i % nc);
  std::vector<uint32_t> freq(nr * nc * 1024), states(n / 64), offsets(n / 64);
  std::vector<uint64_t> row_sum(rows), col_sum(cols);
  size_t begin = 0;
  int bad = each_allocation("sums", [&] { return grf_bctx_sums(words.data(), rows, cols, row_sum.data(), col_sum.data()); });
  bad |= each_allocation("frequencies", [&] {
    return bcx_frequencies(words.data(), n, rows, cols, rc.data(), cc.data(), nr, nc, 0, freq.data()); });
  bad |= each_allocation("encode", [&] {
    return grf_bctx_encode(words.data(), rows, cols, rc.data(), cc.data(), nr, nc, 0, freq.data(), buffer.data(), buffer.size(), &begin); });
  const uint8_t *stream = buffer.data() + begin;
  const size_t bytes = buffer.size() - begin;
  uint8_t *packed = nullptr;
  size_t packed_bytes = 0;
  bad |= bcx_pack6(words.data(), n, &packed, &packed_bytes);
  uint64_t progress = 0;
  bad |= each_allocation("words", [&] {
    progress = 0;
    const int status = grf_bctx_words(stream, bytes, rows, cols, rc.data(), cc.data(), nr, nc, freq.data(), 64, states.data(),
                                      offsets.data(), packed, packed_bytes, nullptr, out.data(), &progress);
    return (progress == (status ? ~0ull : n)) ? status : 99; });
  bad |= out != words;
  bad |= each_allocation("decode", [&] {
    return bcx_decode(stream, bytes, n, rows, cols, rc.data(), cc.data(), nr, nc, 0, nullptr, freq.data(), out.data()); });
  bad |= each_allocation("checkpoint", [&] {
    return bcx_checkpoint(stream, bytes, n, rows, cols, rc.data(), cc.data(), nr, nc, 0, nullptr, freq.data(), 64, states.data(),
                          offsets.data(), out.data()); });
  bcx_free(packed);
  return bad;
}
"""


def test_every_failed_allocation_is_a_status(tmp_path):
    source, program = tmp_path / "allocation.cpp", tmp_path / "allocation"
    source.write_text(_PROGRAM)
    built = subprocess.run(["g++", "-O1", "-std=c++17", "-pthread", "-I", str(CSRC), str(source), "-o", str(program)],
                           capture_output=True, text=True)
    if built.returncode and "not found" in built.stderr:
        pytest.skip("no host compiler")
    assert built.returncode == 0, built.stderr[-2000:]
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=100)
    assert done.returncode == 0, (done.returncode, done.stdout, done.stderr[-500:])
