// One progress step's uploads ahead, on the host: frames waiting in a row, with copies that end at once
// (pageable memory) or stay queued (pinned). Prints the frames a step takes in each case.
#include <cstdio>
#include <vector>

#include "apsm_serve_ahead.h"

static int framesTaken( int waiting, size_t bytes, size_t held, size_t most, bool pageable )
{
    AheadStep step( most );
    int n = 0;
    while ( n < waiting && step.take( held, bytes, [ & ] { return !pageable && n >= 2; } ) )
    {
        held += bytes;
        n++;
    }
    return n;
}

int main()
{
    const size_t mb = size_t( 1 ) << 20;
    printf( "%d %d %d %d %d\n", framesTaken( 100, mb, 0, 64 * mb, true ), framesTaken( 100, mb, 0, 64 * mb, false ),
            framesTaken( 1, mb, 0, 64 * mb, true ), framesTaken( 100, 40 * mb, 0, 64 * mb, true ), framesTaken( 100, mb, 64 * mb, 64 * mb, true ) );
    return 0;
}
