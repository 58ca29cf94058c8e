// Steps on their way to a thread that launches them in order.  Nothing is lost by an exception on either side: what the launches throw comes out of
// push or finish, the thread has ended when the queue is gone, and steps end on the caller's thread only (their buffers and graphs are its own to free).
#pragma once
#include <condition_variable>
#include <deque>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>

namespace ug_llama {

template <typename Step>
class StepQueue {
 public:
  static constexpr size_t kAhead = 3;

  explicit StepQueue(std::function<void(Step&)> run) : run_(std::move(run)), thread_([this] { loop(); }) {}
  ~StepQueue() {
    std::deque<Step> dropped;  // (after finish there are none: these belong to a caller that gives up, or were behind one that threw)
    {
      std::lock_guard<std::mutex> g(mu_);
      dropped.swap(waiting_);
    }
    close();
  }
  // Waits while kAhead steps are waiting.  Steps that have been launched end here.
  void push(Step&& st) {
    std::deque<Step> launched;
    {
      std::unique_lock<std::mutex> g(mu_);
      room_.wait(g, [this] { return waiting_.size() < kAhead || error_; });
      if (error_) std::rethrow_exception(error_);
      waiting_.push_back(std::move(st));
      launched.swap(launched_);
    }
    some_.notify_one();
  }
  // Returns when every step has been launched.
  void finish() {
    close();
    if (error_) std::rethrow_exception(error_);
  }

 private:
  void close() {
    if (!thread_.joinable()) return;
    {
      std::lock_guard<std::mutex> g(mu_);
      closed_ = true;
    }
    some_.notify_one();
    thread_.join();
  }
  void loop() {
    for (;;) {
      std::unique_lock<std::mutex> g(mu_);
      some_.wait(g, [this] { return closed_ || !waiting_.empty(); });
      if (waiting_.empty()) return;
      Step st = std::move(waiting_.front());
      waiting_.pop_front();
      g.unlock();
      std::exception_ptr error;
      try {
        run_(st);
      } catch (...) {
        error = std::current_exception();
      }
      g.lock();
      launched_.push_back(std::move(st));
      error_ = error;
      g.unlock();
      room_.notify_one();
      if (error) return;
    }
  }
  std::function<void(Step&)> run_;
  std::mutex mu_;
  std::condition_variable room_, some_;
  std::deque<Step> waiting_, launched_;
  std::exception_ptr error_;
  bool closed_ = false;
  std::thread thread_;
};

}  // namespace ug_llama
