// Flat sky background with an optional linear gradient, measured from the
// centre (1, 1) of the first pixel.  The gradient defaults to zero.
type = FOREGROUND;

params
{
    { "bg" },
    { "dx", PARAMETER, UNBOUNDED, -0.0f },
    { "dy", PARAMETER, UNBOUNDED, -0.0f }
};

data
{
    float level; // background level
    float2 grad; // gradient (d/dx, d/dy)
};

static float foreground(local data* this, float2 x)
{
    float f = this->level;
    // (no gradient, the default: the same value without seven of a ray's
    // instructions, of 66 behind a tabulated lens with two Sersic sources)
    if(this->grad.x != 0 || this->grad.y != 0)
    {
        lensed_branch();
        f += fma(this->grad.x, x.x - 1, this->grad.y*(x.y - 1));
    }
    return f;
}

static void set(local data* this, float bg, float dx, float dy)
{
    this->level = bg;
    this->grad = (float2)(dx, dy);
}
