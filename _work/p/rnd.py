import random
rng=random.Random(11)
