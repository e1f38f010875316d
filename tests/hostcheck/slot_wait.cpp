// CPU check of csrc/slot_wait.hpp: prints one line per case, exits 1 at the
// first that is wrong.  Build: g++ -std=c++17 -O2 slot_wait.cpp -lpthread
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>

#include "../../fast-rbd-gradients_amd/csrc/slot_wait.hpp"

namespace {

constexpr int kLost = 719, kFailed = 700;
int failures = 0;

void expect(const char* what, int got, int want) {
  std::printf("%s: %d\n", what, got);
  if (got != want) { std::printf("  expected %d\n", want); ++failures; }
}

}  // namespace

int main() {
  auto pause = [] { std::this_thread::yield(); };
  auto never = [] { return false; };
  long asked = 0;

  expect("there at once", rbdi::wait_for_word([] { return true; }, pause,
                                              [&](int*) { ++asked; return true; }, kLost), 0);
  expect("  times the stream was asked", int(asked), 0);

  // a word that another thread sets while the stream is busy
  std::atomic<bool> word{false};
  std::thread setter([&] {
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    word = true;
  });
  expect("set later", rbdi::wait_for_word([&] { return word.load(); }, pause, [&](int*) { ++asked; return true; }, kLost), 0);
  setter.join();

  // a stream that ends with an error, at once and after it was busy for a while
  expect("stream failed", rbdi::wait_for_word(never, pause, [](int* e) { *e = kFailed; return false; }, kLost), kFailed);
  asked = 0;
  expect("stream failed later",
         rbdi::wait_for_word(never, pause, [&](int* e) { *e = kFailed; return ++asked < 20; }, kLost), kFailed);
  expect("  times the stream was asked", int(asked), 20);

  // a stream that has drained: the word arrived in the meantime, or never will
  bool drained = false;
  expect("arrived before the stream drained",
         rbdi::wait_for_word([&] { return drained; }, pause, [&](int*) { drained = true; return false; }, kLost), 0);
  expect("drained without the word", rbdi::wait_for_word(never, pause, [](int*) { return false; }, kLost), kLost);
  return failures ? 1 : 0;
}
