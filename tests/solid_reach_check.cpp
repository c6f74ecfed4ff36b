// solid_reach and solid_errors (torchhull_amd/csrc/solid_reach.h) of the lines `total H W` on standard input, for
// masks with fractions: prints `reach row column` per line.
#include <cstdio>

#include "../torchhull_amd/csrc/solid_reach.h"

int main()
{
    float total;
    int H, W;
    while (std::scanf("%f %d %d", &total, &H, &W) == 3)
    {
        const thull::SolidErrors e = thull::solid_errors(total, H, W);
        std::printf("%.9g %.9g %.9g\n", thull::solid_reach(false, true, total, H, W), e.row, e.column);
    }
    return 0;
}
