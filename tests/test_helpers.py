"""Helper threads (csrc/helpers.hpp): where the system gives fewer than asked for,
those there are run and the call goes on. On the CPU, with a thread type that
is refused after the first few."""
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
SOURCE = """
#include "helpers.hpp"
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <thread>
static int allowed;
struct Limited {
  std::thread thread;
  template <class Body> explicit Limited(const Body &body) {
    if (allowed-- <= 0) throw std::system_error(std::make_error_code(std::errc::resource_unavailable_try_again));
    thread = std::thread(body);
  }
  Limited(Limited &&) = default;
};
int main(int, char **arguments) {
  allowed = std::atoi(arguments[1]);
  std::atomic<int> ran{0};
  std::vector<Limited> threads;
  vsplat::start_helpers(threads, 3, [&] { ++ran; });
  for (auto &t : threads) t.thread.join();
  std::printf("%zu %d", threads.size(), ran.load());
}
"""


@pytest.mark.parametrize("allowed", [0, 1, 3, 9])
def test_fewer_helpers_than_asked_for(allowed, tmp_path):
    source, program = tmp_path / "helpers.cpp", tmp_path / "helpers"
    source.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-I", ROOT / "vibe-splat_amd" / "csrc", source, "-o", program],
                   check=True)
    out = subprocess.run([program, str(allowed)], check=True, capture_output=True, text=True).stdout
    assert out == f"{min(allowed, 3)} {min(allowed, 3)}"
