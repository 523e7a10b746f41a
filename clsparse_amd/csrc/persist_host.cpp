// Host side shared by the persistent solver kernels.
#include "persist_host.hpp"

#include <cstdlib>

#include "grid_sync.hpp"

size_t persist_slot_words() { return kSlotWords; }
unsigned long long persist_slot_empty() { return kSlotEmpty; }

std::mutex& persist_mutex(int device)
{
    static std::mutex m[64];
    return m[static_cast<unsigned>(device) % 64];
}

int persist_spin_limit()
{
    const char* e = std::getenv("CLSPARSE_AMD_PERSIST_SPIN");
    const int n = e ? std::atoi(e) : 0;
    return n > 0 ? n : kSpinLimit;
}

bool persist_refused()
{
    const char* e = std::getenv("CLSPARSE_AMD_PERSIST_REFUSE");
    return e && e[0] == '1';
}

bool persist_enabled()
{
    const char* e = std::getenv("CLSPARSE_AMD_CG_PERSIST");
    return !(e && e[0] == '0');
}
