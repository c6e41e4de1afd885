// ckd_b07_scan.h -- where the in-place blur's scan (k_blur07.hip) runs its
// chunks without the edges' tests.  No includes: a plain host compiler takes it.
#pragma once

namespace ckd {

// lanes of a channel: the most steps of a chunk
constexpr int kB07ScanLanes = 16;

// The last step at which a chunk of the middle run may start, on a line of len
// pixels and nSteps steps: its lanes' pixels stay before the line's last one, and
// a line that stops before its last pixel (nSteps = len - 1) leaves its last step,
// which saves the state, to a chunk with the tests.
constexpr int b07_scan_last(int len, int nSteps)
{
    return (nSteps < len ? nSteps : len) - kB07ScanLanes - 1;
}

} // namespace ckd
