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

int main(int argc, char** argv) {
  const struct {
    const char* name;
    int (*f)();
  } cases[] = {{"renew", renew}};
  for (auto& c : cases)
    if (argc == 2 && !strcmp(argv[1], c.name)) return c.f();
  printf("no such case\n");
  return 2;
}
