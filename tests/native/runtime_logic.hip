// Prints host evaluations of functions that the kernels and their launches share.
#include "vector_kernels.hpp"

#include <iostream>

int
main()
{
  // CG's end flag as the launches with scalars 5, 6 and 7 find it when 6 ends the iteration
  std::cout << "turn_open: " << ppf::cg_ended_before(0, 5) << ppf::cg_ended_before(0, 6) << "\n"
            << "turn_racing: " << ppf::cg_ended_before(6, 6) << "\n"
            << "turn_after: " << ppf::cg_ended_before(6, 7) << "\n"
            << "turn_last_tag: " << ppf::cg_ended_before(0x7fffffff, 1)
            << ppf::cg_ended_before(0x7fffffff, 0x7fffffffu) << "\n";
}
