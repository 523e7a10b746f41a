// Host side shared by the persistent solver kernels.
#pragma once

#include <cstddef>
#include <mutex>

// The slots of their grid-wide sums (grid_sync.hpp): this many words, each set
// to the empty value before a solve.
size_t persist_slot_words();
unsigned long long persist_slot_empty();
// Held from the launch of a persistent kernel until it has ended: one per
// device at a time (two that shared the CUs could each hold some the other
// waits for).
std::mutex& persist_mutex(int device);
// Polls before a workgroup of a persistent kernel gives up waiting for another
// (CLSPARSE_AMD_PERSIST_SPIN=<n>; default 131072, about 0.1 s). The solve then goes on in
// separate launches from the x it had before that launch, with the rows of
// workgroups that came to the launch's end as these have left them.
int persist_spin_limit();
// CLSPARSE_AMD_PERSIST_REFUSE=1 (for tests): every persistent launch is taken as
// refused by the device.
bool persist_refused();
// CLSPARSE_AMD_CG_PERSIST=0 keeps the launch-per-step iterations.
bool persist_enabled();
