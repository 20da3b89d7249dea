// Scalars the device sends to a host that polls for them (dot products, residual norms).
//
// Plain C++: the entries live in pinned memory that the runtime allocates, the kernels write
// them with tell_host (vector_kernels.hpp).
#pragma once

namespace ppf
{
  /// One scalar: the value, then (tag << 1) | flag once the value is visible.
  struct HostScalar
  {
    double       value;
    unsigned int word;
  };

  /// Tags of the scalars and the entries they go to.  At most four scalars are under way at a
  /// time (the residual of a CG step, the two maxima of a plan compared in the step enqueued
  /// ahead, and that step's residual), so an entry is read before it is issued again.
  class HostScalarRing
  {
  public:
    static constexpr int size = 4;

    explicit HostScalarRing(unsigned int last_tag = 0)
      : tag(last_tag)
    {}

    /// Empties the entries before the first use: pinned memory comes with any contents, such
    /// as the entries of an earlier context, whose tags began at 1 too and would be taken for the
    /// scalars of this one.  (Later an entry holds a tag of this ring, an older one than is
    /// awaited there.)
    static void
    clear(HostScalar *entries)
    {
      for (int k = 0; k < size; ++k)
        *reinterpret_cast<volatile unsigned int *>(&entries[k].word) = 0u;
    }

    /// Tag of the next scalar, 1 .. 2^31 - 1.
    unsigned int
    issue()
    {
      tag = tag % 0x7fffffffu + 1u;
      return tag;
    }

    static HostScalar *
    entry(HostScalar *entries, unsigned int t)
    {
      return entries + t % size;
    }

    /// The entry's word, read from memory (it is written behind the compiler's back).
    static unsigned int
    word(const HostScalar *e)
    {
      return *reinterpret_cast<const volatile unsigned int *>(&e->word);
    }

    static bool
    ready(unsigned int w, unsigned int t)
    {
      return (w >> 1) == t;
    }

  private:
    unsigned int tag;
  };
} // namespace ppf
