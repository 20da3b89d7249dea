// Prints what the ring of scalars sent to the host makes of memory with stale entries.
#include "host_scalars.hpp"

#include <iostream>

int
main()
{
  using ppf::HostScalar;
  using ppf::HostScalarRing;
  // memory an earlier context has left: scalars 1 .. 4 of its own
  HostScalar entries[HostScalarRing::size];
  for (unsigned int t = 1; t <= 4; ++t)
    *HostScalarRing::entry(entries, t) = {100.0 + t, t << 1};

  HostScalarRing ring;
  HostScalarRing::clear(entries);
  int            stale = 0, missed = 0;
  unsigned int   first = 0;
  for (int k = 0; k < 9; ++k)
    {
      const unsigned int t = ring.issue();
      if (k == 0)
        first = t;
      HostScalar *e = HostScalarRing::entry(entries, t);
      stale += HostScalarRing::ready(HostScalarRing::word(e), t);
      *e = {double(k), (t << 1) | 1u}; // the device answers
      missed += !HostScalarRing::ready(HostScalarRing::word(e), t);
    }
  std::cout << "first: " << first << "\nstale: " << stale << "\nmissed: " << missed << "\n";

  // an emptied entry is no tag's, also where the tags start again
  HostScalarRing late(0x7ffffffeu);
  const unsigned a = late.issue(), b = late.issue();
  std::cout << "last: " << a << "\nwrapped: " << b << "\nempty: "
            << HostScalarRing::ready(HostScalarRing::word(HostScalarRing::entry(entries, b)), b)
            << "\n";
}
