// Checks zkx::SpareMemory (the transforms' scratch) against an allocator that
// refuses.  Prints "ok" or the first wrong step.
#include <stdio.h>
#include <stdlib.h>

#include <map>

#include "spare.h"

static size_t limit, used, asked, freed;
static std::map<void *, size_t> live;

static void *take(size_t n)
{
    asked++;
    if (used + n > limit) return nullptr;
    void *p = malloc(1);
    live[p] = n;
    used += n;
    return p;
}

static void give(void *p)
{
    freed++;
    used -= live.at(p);
    live.erase(p);
    free(p);
}

#define EXPECT(c)                                 \
    do {                                          \
        if (!(c)) {                               \
            printf("line %d: %s\n", __LINE__, #c); \
            return 1;                             \
        }                                         \
    } while (0)

int main()
{
    {
        zkx::SpareMemory s(take, give);
        limit = 100;
        EXPECT(s.hold(4, 10) == 4 && used == 40 && s.get());
        EXPECT(s.hold(3, 10) == 3 && asked == 1);            // fits what is there
        EXPECT(s.hold(6, 10) == 6 && used == 60 && asked == 2);  // grown, the old part given back
        void *const was = s.get();
        EXPECT(s.hold(9, 10) == 6 && s.get() == was);        // refused: keeps what it has
        EXPECT(asked == 3 && used == 60);
        for (uint32_t k = 0; k < s.kRefusedCalls; k++) EXPECT(s.hold(9 + k % 2, 10) == 6);
        EXPECT(asked == 3);                                  // and does not ask each time
        limit = 200;
        EXPECT(s.hold(9, 10) == 9 && asked == 4 && used == 90);  // until it does again
        EXPECT(s.drop() && used == 0 && !s.get() && !s.drop());
        limit = 5;
        EXPECT(s.hold(1, 10) == 0 && asked == 5 && s.hold(2, 10) == 0 && asked == 5);
        EXPECT(s.hold(1, 4) == 1 && asked == 6);             // less than was refused is asked for
        EXPECT(!live.empty());
    }
    EXPECT(live.empty() && used == 0);
    puts("ok");
    return 0;
}
