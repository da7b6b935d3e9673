// What a thread is about to do, for the case that it does not come back from
// it: where a process ends in a fault or an abort, a line of each thread's own
// goes to stderr before whatever handled that before handles it.
//
// For work that runs rarely and that code of others may end (a race of library
// algorithms): handlers stand while a note does, and are taken back with the
// last one, unless somebody has put others in their place since.

#pragma once

#include <signal.h>
#include <sys/syscall.h>
#include <unistd.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <mutex>

namespace vllm_amd {

class FaultNote {
 public:
  FaultNote() {
    std::lock_guard<std::mutex> g(mutex());
    if (holders()++ == 0) {
      struct sigaction act {};
      act.sa_sigaction = &handle;
      act.sa_flags = SA_SIGINFO | SA_ONSTACK;
      sigemptyset(&act.sa_mask);
      for (int i = 0; i < SIGNALS; ++i) sigaction(SIGNAL[i], &act, &before(i));
    }
    const long me = syscall(SYS_gettid);
    for (Slot& s : slots()) {
      long free = 0;
      if (s.thread.compare_exchange_strong(free, me)) {
        slot_ = &s;
        break;
      }
    }
  }
  FaultNote(const FaultNote&) = delete;
  FaultNote& operator=(const FaultNote&) = delete;
  ~FaultNote() {
    std::lock_guard<std::mutex> g(mutex());
    if (slot_ != nullptr) {
      slot_->length.store(0);
      slot_->thread.store(0);
    }
    if (--holders() > 0) return;
    for (int i = 0; i < SIGNALS; ++i) {
      struct sigaction now {};
      sigaction(SIGNAL[i], nullptr, &now);
      if ((now.sa_flags & SA_SIGINFO) && now.sa_sigaction == &handle)
        sigaction(SIGNAL[i], &before(i), nullptr);
    }
  }

  // Replaces this thread's line. (More than eight threads at a time: none.)
  __attribute__((format(printf, 2, 3))) void say(const char* format, ...) {
    if (slot_ == nullptr) return;
    slot_->length.store(0);
    va_list args;
    va_start(args, format);
    const int n = vsnprintf(slot_->line, sizeof slot_->line - 1, format, args);
    va_end(args);
    if (n <= 0) return;
    const int room = (int)sizeof slot_->line - 2;
    const int end = n < room ? n : room;
    slot_->line[end] = '\n';
    slot_->length.store(end + 1);
  }

 private:
  struct Slot {
    std::atomic<long> thread{0};
    std::atomic<int> length{0};
    char line[240];
  };
  static constexpr int SIGNALS = 4;
  static constexpr int SIGNAL[SIGNALS] = {SIGSEGV, SIGBUS, SIGFPE, SIGABRT};

  static std::mutex& mutex() { static std::mutex m; return m; }
  static int& holders() { static int n = 0; return n; }
  static Slot (&slots())[8] { static Slot s[8]; return s; }
  static struct sigaction& before(int i) {
    static struct sigaction b[SIGNALS];
    return b[i];
  }

  // Calls nothing that a signal handler may not call.
  static void handle(int sig, siginfo_t* info, void*) {
    const long me = syscall(SYS_gettid);
    for (Slot& s : slots())
      if (s.thread.load() == me && s.length.load() > 0) {
        static const char head[] = "[vllm_amd] ended in: ";
        (void)!write(2, head, sizeof head - 1);
        (void)!write(2, s.line, s.length.load());
      }
    for (int i = 0; i < SIGNALS; ++i)
      if (SIGNAL[i] == sig) sigaction(sig, &before(i), nullptr);
    // A faulting access comes again by itself; a signal that was sent does not.
    if (info == nullptr || info->si_code <= 0) raise(sig);
  }

  Slot* slot_ = nullptr;
};

}  // namespace vllm_amd
