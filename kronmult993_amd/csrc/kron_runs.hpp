// kron_runs.hpp -- a batch cut into runs of consecutive entries, one per workgroup (host and device).
//
// Run lengths come from the caller as well (entries_per_workgroup, any positive int) and grids are rounded up to whole
// XCD stripes, so index * length goes up to 7 * 2^31 past the batch: it is formed in 64 bits, and a run past the batch
// is empty instead of wrapping to a negative entry.
#pragma once

namespace kronruns
{

// first entry of run `index`, nb for a run past the batch
constexpr int begin(long index, long length, int nb)
{
    return index * length < nb ? static_cast<int>(index * length) : nb;
}
// first entry after the run that begins at `first`
constexpr int end(int first, long length, int nb)
{
    return nb - first > length ? first + static_cast<int>(length) : nb;
}
// runs in a batch
constexpr long count(int nb, long length)
{
    return (nb + length - 1) / length;
}

} // namespace kronruns
