/*
 * The memory that calls on a device keep between them: one buffer, grown and not shrunk.
 * Plain C++, so that its refusals can be tested without a device.
 */
#ifndef MGX_CALL_BUFFER_H
#define MGX_CALL_BUFFER_H

#include <cstddef>

namespace mgx {

enum class Held { None, Needed, All };

/*
 * Makes p hold needed bytes and, where there is memory for them, extra bytes more that the
 * caller can do without; says which.  alloc returns null when there is no memory.  A larger
 * buffer is taken beside the old one first, so that where only the extra bytes are refused a
 * buffer that holds the needed ones stays: freeing it would wait for the device, and it would
 * have to be allocated again, in every call.
 */
template <typename Alloc, typename Free>
Held hold(unsigned char *&p, std::size_t &bytes, std::size_t needed, std::size_t extra, Alloc alloc, Free release)
{
    const std::size_t all = needed + extra;
    if (p && bytes >= all) return Held::All;
    unsigned char *q = alloc(all);
    if (!q && p) {
        if (extra > 0 && bytes >= needed) return Held::Needed;
        release(p);
        p = nullptr;
        bytes = 0;
        q = alloc(all);
    }
    Held held = Held::All;
    std::size_t size = all;
    if (!q && extra > 0) {
        q = alloc(needed);
        held = Held::Needed;
        size = needed;
    }
    if (!q) return Held::None;
    if (p) release(p);
    p = q;
    bytes = size;
    return held;
}

} // namespace mgx

#endif
