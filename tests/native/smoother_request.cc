// Prints which operator launches would take a parked smoother step.
#include "smoother_request.hpp"

#include <iostream>
#include <stdexcept>

int
main()
{
  using namespace ppf;
  SmootherRequest<double> slot, step;
  double                  x[1], y[1], z[1];
  step.block = 2;
  step.dst   = y;
  step.src   = x;
  step.kind  = Smoother::Chebyshev;

  std::cout << "before: " << slot.waits_for(2, y, x) << "\n";
  {
    SmootherScope<double> scope(slot, step);
    std::cout << "other_block: " << slot.waits_for(1, y, x) << "\n"
              << "other_dst: " << slot.waits_for(2, z, x) << "\n"
              << "other_src: " << slot.waits_for(2, y, z) << "\n"
              << "own: " << slot.waits_for(2, y, x) << slot.taken << "\n";
    slot.take(7);
    std::cout << "taken: " << slot.waits_for(2, y, x) << slot.taken << slot.blocks << "\n";
  }
  {
    // an application that compares two paths on A x
    SmootherScope<double> scope(slot, step);
    slot.withdraw();
    std::cout << "withdrawn: " << slot.waits_for(2, y, x) << slot.taken << "\n";
  }
  // an application that throws, one that no launch took, and a second one after each
  try
    {
      SmootherScope<double> scope(slot, step);
      throw std::runtime_error("allocation");
    }
  catch (const std::runtime_error &)
    {}
  std::cout << "after_throw: " << slot.waits_for(2, y, x) << slot.taken << "\n";
  {
    SmootherScope<double> scope(slot, step);
  }
  std::cout << "not_taken: " << slot.waits_for(2, y, x) << slot.taken << "\n";
}
