// Checks of csrc/qpip_mailbox.hpp on the host: where a call's block goes. Prints the first
// statement that does not hold and returns 1.
#include <cstdio>
#include <set>
#include <stdexcept>
#include <thread>
#include <vector>

#include "qpip_mailbox.hpp"

namespace {

std::set<void*> live;  // blocks allocated and not freed
int made = 0;

void* make()
{
  void* p = ::operator new(64);
  live.insert(p);
  ++made;
  return p;
}

void drop(void* p)
{
  live.erase(p);
  ::operator delete(p);
}

int device = 0;

void* call(qpip::MailboxList& list, int on, bool fails_before, bool fails_after)
{
  void* p = nullptr;
  device  = on;
  try {
    qpip::Mailbox box(list, [] { return device; }, make);
    p = box.get();
    if (fails_before) throw std::runtime_error("not launched");
    box.launched();
    if (fails_after) throw std::runtime_error("in flight");
    box.landed();
  } catch (std::runtime_error const&) {
  }
  return p;
}

int check(bool ok, char const* what)
{
  if (!ok) std::printf("does not hold: %s\n", what);
  return ok ? 0 : 1;
}

}  // namespace

int main()
{
  qpip::MailboxList list;
  auto const idle = [] { return true; };
  int bad         = 0;
  void* const a   = call(list, 0, false, false);
  bad += check(call(list, 0, false, false) == a && made == 1, "a block given back is lent again");
  bad += check(call(list, 0, true, false) == a && call(list, 0, false, false) == a && made == 1,
               "a call that fails before its launch gives its block back");
  bad += check(call(list, 0, false, true) == a, "the block of a call that fails in flight");
  void* const b = call(list, 0, false, false);
  bad += check(b != a && made == 2, "... is not lent again");
  for (int i = 0; i < 100; ++i) call(list, 1, false, true);
  bad += check(made == 101, "calls that fail in flight each need a block (one was free)");
  list.trim(0, [] { return false; }, drop);
  bad += check(live.size() == 101 && live.count(a) == 1,
               "a device that is not idle keeps its blocks, and no block was free");
  list.trim(0, idle, drop);
  bad += check(live.size() == 100 && live.count(a) == 0, "trim frees its own device's blocks");
  list.trim(1, idle, drop);
  bad += check(live.empty(), "and the other device's when that is trimmed");
  call(list, 0, false, false);
  list.trim(0, [] { return false; }, drop);
  bad += check(live.empty(), "a free block is freed without waiting");
  return bad ? 1 : 0;
}
