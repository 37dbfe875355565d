// Reads of the window sequencer against the floats its block buffers are reserved with, on the host:
// for every windowSize, block length reserved and run, and window fill, the last float that a step's
// package copies (whole 256-float pieces of the image with the self entries, and of the eviction
// shares) and the left rows' loads touch. Prints the largest overrun of each buffer per windowSize
// that has one, and the number of layouts looked at.
#include <algorithm>
#include <cstdint>
#include <cstdio>

#include "apsm_detect_launch.h"
#include "apsm_win_layout.h"

using namespace apsm;

// Last float + 1 that the steps of a block of n steps read from the Gram buffer; a package past the last
// step is the last step's again.
static int64_t gramEnd( int n, int newRel0, int Wc, int tp )
{
    int64_t end = Wc * winImg( tp ); // the images at the block start
    for ( int m : { 0, n / 2, n - 1 } )
    {
        const int64_t row = winRow( m, newRel0, Wc, tp );
        const int64_t o4 = ( winOlder( m, newRel0, Wc ) + 3 ) & ~3;
        end = std::max( end, row + winPkGram( tp ) );
        // planes at 0, o4 and 2 o4, 4 floats from j <= max(o4 - 4, 0)
        end = std::max( end, row + winImg( tp ) + 4 + 2 * o4 + std::max<int64_t>( o4 - 4, 0 ) + 4 );
    }
    return end;
}

static int64_t evEnd( int64_t U, int n, int w2, int tp )
{
    return ( U * n - 1 ) * winEvStride( w2 ) + winPkEv( tp );
}

int main()
{
    int64_t looked = 0, bad = 0;
    for ( int Wc = 1; Wc <= 160; Wc++ )
    {
        const int tp = winTp( Wc ), w2 = 2 * Wc;
        int64_t overGram = 0, overEv = 0;
        for ( int steps = 1; Wc + steps <= kActMax; steps++ )
        {
            if ( steps > 1 && winGactFloats( Wc, steps ) > gramRow<int64_t>( kActMax ) )
                break;
            const int64_t gram = winGactFloats( Wc, steps );
            for ( int n : { 1, 2, steps / 2, steps - 1, steps } )
            {
                if ( n < 1 || n > steps )
                    continue;
                for ( int newRel0 : { 0, 1, Wc / 2, Wc - 1 } )
                    if ( newRel0 < Wc )
                        overGram = std::max( overGram, gramEnd( n, newRel0, Wc, tp ) - gram );
                for ( int64_t U : { 1, 2, 3, 10, 1024 } )
                    overEv = std::max( overEv, evEnd( U, n, w2, tp ) - winEvFloats( U, steps, w2 ) );
                looked++;
            }
        }
        if ( overGram > 0 || overEv > 0 )
        {
            bad++;
            printf( "windowSize %d: %lld floats past the Gram, %lld past the eviction shares\n", Wc, (long long)overGram, (long long)overEv );
        }
    }
    printf( "%lld layouts, %lld windows with reads out of range\n", (long long)looked, (long long)bad );
    return bad ? 1 : 0;
}
