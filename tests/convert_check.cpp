/* Host check of convert_out (p2m_convert.h): a map in pieces through a
 * device buffer that may not be had at every size, the pieces in order, each
 * once, within the buffer, and through the host where no buffer is to be had;
 * an error ends it. */
#include "p2m_convert.h"
#include <cstdio>
#include <vector>

struct Ops {
    int64_t n, room;               /* buffers of up to `room` values can be had */
    int64_t cap = 0, next = 0, pieces = 0, host = 0, fail_at = -1;
    bool ok = true;
    bool buffer(int64_t k)
    {
        if (k <= cap) return true;
        cap = 0;
        if (k > room) return false;
        cap = k;
        return true;
    }
    int piece(int64_t i, int64_t k)
    {
        ok &= i == next && k > 0 && i + k <= n;
        next = i + k;
        return pieces++ == fail_at ? -3 : 0;
    }
    int on_device(int64_t i, int64_t k) { ok &= k <= cap; return piece(i, k); }
    int on_host(int64_t i, int64_t k) { host += k; return piece(i, k); }
};

int main()
{
    long bad = 0, runs = 0;
    for (int64_t n : {0, 1, 15, 16, 17, 63, 64, 65, 1000, 4096, 4097})
        for (int64_t room = 0; room <= 300; ++room)
            for (int kept = 0; kept < 2; ++kept) {
                Ops o{n, room};
                if (kept && room >= 40) o.cap = 40;
                const int rc = convert_out(o, n, 256, 16);
                ++runs;
                const int64_t want = n < 256 ? n : 256;
                bool fine = rc == 0 && o.ok && o.next == n;
                /* the host only where not even the least buffer is to be had, or a shorter map's whole */
                fine &= o.host == 0 || (o.host == n && (room < 16 || (n < 16 && room < n)));
                /* whole pieces where there is room for them */
                if (n > 0 && room >= want) fine &= o.pieces == (n + want - 1) / want;
                if (!fine && ++bad < 10) printf("n %ld room %ld kept %d: rc %d next %ld host %ld pieces %ld\n", (long)n, (long)room, kept, rc, (long)o.next, (long)o.host, (long)o.pieces);
            }
    for (int64_t at : {0, 1, 3}) {
        Ops o{1000, 300};
        o.fail_at = at;
        ++runs;
        if (convert_out(o, 1000, 256, 16) != -3 || o.pieces != at + 1) ++bad;
    }
    printf("checked %ld copies, %ld mismatches\n", runs, bad);
    return bad != 0;
}
