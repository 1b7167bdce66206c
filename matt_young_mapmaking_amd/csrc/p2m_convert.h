/* A map copied out in the other precision: through a device buffer of at
 * most `most` values, of as many as can be had down to `least`, else converted
 * by the host, as many at a time.  Host code; Ops gives the steps:
 *   bool buffer(k)            a device buffer of k values at least, or false
 *   int on_device(i, k)       values [i, i + k) through that buffer
 *   int on_host(i, k)         through host memory
 * which return 0 or an error. */
#ifndef P2M_CONVERT_H
#define P2M_CONVERT_H

#include <stdint.h>

template <typename Ops>
static inline int convert_out(Ops &o, int64_t n, int64_t most, int64_t least)
{
    int64_t piece = n < most ? n : most;
    bool device = piece > 0 && o.buffer(piece);
    while (!device && piece > least) {
        piece = piece / 2 > least ? piece / 2 : least;
        device = o.buffer(piece);
    }
    for (int64_t i = 0; i < n; i += piece) {
        const int64_t k = n - i < piece ? n - i : piece;
        const int rc = device ? o.on_device(i, k) : o.on_host(i, k);
        if (rc) return rc;
    }
    return 0;
}

#endif
