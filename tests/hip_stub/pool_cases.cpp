// Cases of the workspace pool (tom_amd/csrc/pool.hip) against hip_runtime.h of
// this folder. pool_cases NAME: exit status 0 where the case holds.
#include <stdio.h>
#include <string.h>

#include "../../tom_amd/csrc/pool.hip"

using namespace tomhip;

#define HOLDS(c)                                    \
  do {                                              \
    if (!(c)) {                                     \
      printf("line %d: not so: %s\n", __LINE__, #c); \
      return 1;                                     \
    }                                               \
  } while (0)

// A block that cannot be renewed leaves a null pointer behind, which is put
// without harm; the block itself went back once.
static int renew() {
  FakeStream s;
  work_device_up(0);
  float* p = nullptr;
  work_renew(&p, 4096, &s);
  HOLDS(p);
  float* q = p;
  work_renew(&p, 8192, &s);
  HOLDS(p && p != q);
  fake().limit = 1 << 20;
  bool threw = false;
  try {
    work_renew(&p, 2 << 20, &s);
  } catch (const Error&) {
    threw = true;
  }
  HOLDS(threw && p == nullptr);
  work_put(p, &s);
  work_device_down(0);
  HOLDS(fake().live.empty() && fake().freed_twice.empty());
  return 0;
}

// A block whose stream has work queued is waited for also where the next call
// names the same handle: a handle is not a stream (a destroyed stream's may
// come back as another one's).
static int same_handle() {
  FakeStream s;
  work_device_up(0);
  void* p = work_get(4096, &s);
  ++s.queued;
  work_put(p, &s);
  s.done = 0;
  HOLDS(work_get(4096, &s) == p);
  HOLDS(fake().waits == 1);
  // once the stream has run dry nothing is waited for
  s.done = s.queued;
  work_put(p, &s);
  HOLDS(work_get(4096, &s) == p);
  HOLDS(fake().waits == 1);
  work_put(p, &s);
  work_device_down(0);
  HOLDS(fake().live.empty());
  return 0;
}

// hipStreamPerThread is another stream in every thread, so neither a query nor
// an event of the thread that gives a block back says when the work of another
// one has left it: such a block goes to the driver, which waits for the device.
static int per_thread() {
  work_device_up(0);
  void* p = work_get(4096, hipStreamPerThread);
  work_put(p, hipStreamPerThread);  // dry in this thread
  HOLDS(fake().frees == 1);
  FakeStream s;
  p = work_get(8192, &s);
  ++s.queued;
  work_put(p, &s);
  HOLDS(work_get(8192, hipStreamPerThread) == p && fake().waits == 1);
  work_put(p, hipStreamPerThread);
  HOLDS(fake().frees == 2);
  work_device_down(0);
  HOLDS(fake().live.empty() && fake().freed_twice.empty());
  return 0;
}

// A plan's blocks are kept for the next call only where the device could be
// waited for.
static int all_of_a_plan() {
  FakeStream s;
  work_device_up(0);
  void* p = work_get(4096, &s);
  void* q = work_get(8192, &s);
  ++s.queued;
  work_put_all({p, nullptr, q});
  HOLDS(fake().frees == 0 && work_get(4096, &s) == p && work_get(8192, &s) == q && fake().waits == 0);
  fake().sync_fails = true;
  work_put_all({p, nullptr, q});
  HOLDS(fake().frees == 2 && fake().live.empty());
  work_device_down(0);
  return 0;
}

// Memory that is no workspace (a network's, a table's) is found where the
// workspaces that wait for a next call hold it.
static int other_memory() {
  FakeStream s;
  work_device_up(0);
  fake().limit = 8 << 20;
  void* p = work_get(6 << 20, &s);
  work_put(p, &s);
  HOLDS(fake().used == 6 << 20);
  void* q = device_malloc(4 << 20);
  HOLDS(q && fake().used == 4 << 20);
  bool threw = false;
  try {
    device_malloc(8 << 20);
  } catch (const Error&) {
    threw = true;
  }
  HOLDS(threw);
  (void)hipFree(q);
  work_device_down(0);
  HOLDS(fake().live.empty() && fake().freed_twice.empty());
  return 0;
}

// What waits can be asked for; what is in use stays.
static int trim() {
  FakeStream s;
  work_device_up(0);
  void* p = work_get(4096, &s);
  work_put(work_get(8192, &s), &s);
  HOLDS(fake().live.size() == 2);
  work_trim(0);
  HOLDS(fake().live.size() == 1 && fake().live.count(p));
  work_put(p, &s);
  HOLDS(work_get(4096, &s) == p);
  return 0;
}

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*f)();
  } cases[] = {{"renew", renew}, {"same_handle", same_handle}, {"per_thread", per_thread},
                 {"all_of_a_plan", all_of_a_plan}, {"other_memory", other_memory},
                 {"trim", trim}};
  for (auto& c : cases)
    if (argc == 2 && !strcmp(argv[1], c.name)) return c.f();
  printf("no such case\n");
  return 2;
}
