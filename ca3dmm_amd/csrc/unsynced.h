// Nested entry calls without a synchronisation of their own.
#pragma once

namespace ca3 {

// Until its end, the entries that this thread calls return as soon as their
// work is queued, whatever hip_proxy_set_sync says.  The mode itself stays as
// the caller set it, for the other threads too.
struct Unsynced {
    Unsynced();
    ~Unsynced() { end(); }
    void end();
    Unsynced(const Unsynced &) = delete;
    Unsynced &operator=(const Unsynced &) = delete;
    bool on = true;
};

}  // namespace ca3
